"""Rows gathered inside the hops' launches: batches on the caller's stream whose misses come over the host link, with rows on
both sides of each length from which a gather of its own takes over, few and most nodes cached, no cache, one to three hops,
no seeds, one seed and repeated ones, groups, and the caller's own buffers."""
import ctypes

import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu

N_NODES = 6_000


@pytest.fixture(scope="module")
def graph():
    rng = np.random.default_rng(21)
    return rng, *random_graph(rng, N_NODES, 10, hubs=4, hub_deg=2000)


# elements of a row (4 bytes each), share of the nodes in the cache (0: none)
@pytest.mark.parametrize("dim,cached", [(4, 0.3), (100, 0.3), (640, 0.3), (641, 0.3), (384, 0.8), (385, 0.8), (1024, 0.8), (1025, 0.8),
                                        (128, 0.95), (129, 0.95), (33, 0.0), (1024, 0.0), (1025, 0.0)])
@pytest.mark.parametrize("fanout", [[20], [25, 10], [5, 4, 3]])
def test_rows_match_the_table(lmi, oracle, graph, dim, cached, fanout):
    rng, indptr, indices = graph
    feats = make_features(lmi, rng, N_NODES, dim)
    batch = 257
    srv = lmi.Server(batch, fanout, dim, pipes=2, seed=3)
    stream, buffers = lmi.stream_create(), []
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.tune("small_edges", 0)
        rows = int(cached * N_NODES)
        slot = np.full(N_NODES, -1, np.int32)
        if rows:
            srv.build_static_cache(rows, lmi.TABLE_HASH)
            slot = oracle.static_cache_build(indptr, rows)
        before = srv.routes()
        sizes = [batch, 0, 1, 64, 256, batch]
        for it, n in enumerate(sizes):
            seeds = rng.integers(0, N_NODES, n).astype(np.int32)   # repeated ones among them
            srv.run_once(seeds, rng_seed=it + 1, pipe=it & 1, stream=stream)
            g = srv.fetch(pipe=it & 1, stream=stream)
            assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds, fanout, it + 1))
            np.testing.assert_array_equal(g.cache_index, slot[g.ids])
            assert g.features.tobytes() == feats.array[g.ids].tobytes()
        if rows or dim <= 1024:   # taken in order from the first: all of it on the caller's stream
            assert srv.routes()["one_pass_gathers"] - before["one_pass_gathers"] == len(sizes)
        # the same into buffers of the caller's, headers included
        seeds = rng.integers(0, N_NODES, batch).astype(np.int32)
        v = srv.view(0)
        out = lmi.BatchView()
        ctypes.memmove(ctypes.byref(out), ctypes.byref(v), ctypes.sizeof(out))
        d = srv_alloc(lmi, buffers, batch * 4)
        lmi.check(lmi.lib().lmi_copy_to_device(d, seeds.ctypes.data_as(ctypes.c_void_p), batch * 4))
        out.node_counter, out.edge_counter = srv_alloc(lmi, buffers, 64), srv_alloc(lmi, buffers, 64)
        for n in (batch, 0):
            srv.run_once_static(d, n, out, rng_seed=9, stream=stream)
            lmi.check(lmi.lib().lmi_stream_sync(stream))
            o = oracle.sample_batch(indptr, indices, seeds[:n], fanout, 9)
            nc, ec = np.empty(16, np.int32), np.empty(16, np.int32)
            for host, dev in ((nc, out.node_counter), (ec, out.edge_counter)):
                lmi.check(lmi.lib().lmi_copy_to_host(host.ctypes.data_as(ctypes.c_void_p), dev, 64))
            assert list(nc) == list(o.node_counter) and list(ec) == list(o.edge_counter)
            got = np.empty((len(o.ids), dim), np.float32)
            src = np.empty(len(o.agg_src_off), np.int32)
            if len(o.ids):
                lmi.check(lmi.lib().lmi_copy_to_host(got.ctypes.data_as(ctypes.c_void_p), out.features, got.nbytes))
            if len(src):
                lmi.check(lmi.lib().lmi_copy_to_host(src.ctypes.data_as(ctypes.c_void_p), out.agg_src_off, src.nbytes))
            assert got.tobytes() == feats.array[o.ids].tobytes()
            np.testing.assert_array_equal(src, o.agg_src_off)
        after = srv.routes()
        # the graph's lowest 5 % have no neighbours: hardly a row of theirs is met
        early = dim * 4 <= 512 or (dim * 4 <= 4096 and cached < 0.95)
        assert after["early_rows"] - before["early_rows"] == (len(sizes) + 2 if early else 0)
        tiles = after["tile_rows"] - before["tile_rows"]
        assert tiles <= (len(sizes) + 2 if early else 0)
        assert dim * 4 > 400 or tiles > 0                  # not where one seed's rows are all there is to move
        assert cached == 0.0 or dim < 1024 or tiles == 0   # too many bytes a thread
        srv.status()
    finally:
        for p in buffers:
            lmi.check(lmi.lib().lmi_device_free(p))
        srv.close()
        feats.free()


@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("cached", [0.0, 0.3])
@pytest.mark.parametrize("knob,value", [(None, None), ("gather_nontemporal", 0), ("gather_unroll", 4), ("gather_tile_rows", 5), ("gather_blocks", 40)])
def test_knobs_keep_a_launch_of_their_own(lmi, oracle, graph, knob, value, cached, small):
    """A knob of the gather acts on a gather: the rows are in no other launch then."""
    rng, indptr, indices = graph
    dim, fanout, batch = 33, [10, 5], 24
    feats = make_features(lmi, rng, N_NODES, dim)
    srv = lmi.Server(batch, fanout, dim, pipes=1, seed=3)
    stream = lmi.stream_create()
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        if not small:
            srv.tune("small_edges", 0)
        if cached:
            srv.build_static_cache(int(cached * N_NODES), lmi.TABLE_RANK)
        if knob:
            srv.tune(knob, value)
        for it in range(2):
            seeds = rng.integers(0, N_NODES, batch).astype(np.int32)
            srv.run_once(seeds, rng_seed=it + 1, stream=stream)
            g = srv.fetch(stream=stream)
            assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds, fanout, it + 1))
            assert g.features.tobytes() == feats.array[g.ids].tobytes()
        routes = srv.routes()
        taken = knob is None or (knob == "gather_unroll" and cached > 0)   # with a cache that knob has never acted on this gather
        assert routes["small_batches"] == (2 if small else 0)
        assert routes["one_pass_gathers"] == 2
        assert routes["small_rows" if small else "early_rows"] == (2 if taken else 0)
        srv.status()
    finally:
        srv.close()
        feats.free()


# threads of a tile, nodes per lane group, tiles per CU that a launch may have of it
SHAPES = [(256, 1, 1), (512, 1, 1), (1024, 1, 1), (512, 2, 2), (512, 4, 2), (1024, 4, None)]


@pytest.fixture(scope="module")
def wide_graph():
    rng = np.random.default_rng(22)
    return rng, *random_graph(rng, 150_000, 12, hubs=100, hub_deg=300)


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("fanout", [3, 20])   # lane groups of 4 and 32
@pytest.mark.parametrize("cached,group", [(0.3, 1), (0.0, 1), (0.0, 3)])   # three batches: without a cache always in line
def test_rows_by_every_tile(lmi, oracle, wide_graph, shape, fanout, cached, group):
    """The last hop's tiles gather what they add and fill in their edges' local ids, at the largest batch that still takes the
    tile and with one node more than the tile before may have."""
    rng, indptr, indices = wide_graph
    n_nodes, dim, lanes, cus = len(indptr) - 1, 4, 4 if fanout == 3 else 32, 256
    feats = make_features(lmi, rng, n_nodes, dim)
    most = [cus * per_cu // group * (threads // lanes * nodes) for threads, nodes, per_cu in SHAPES[:-1]]
    sizes = [most[shape - 1] + 1 if shape else most[0] // 2, most[shape] if shape < len(most) else most[-1] + 1000]
    if sizes[-1] * (1 + fanout) * group > 4_000_000:
        sizes = sizes[:1]
    srv = lmi.Server(sizes[-1], [fanout], dim, pipes=group, seed=3)
    stream = lmi.stream_create()
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.tune("small_edges", 0)
        slot = np.full(n_nodes, -1, np.int32)
        if cached:
            srv.build_static_cache(int(cached * n_nodes), lmi.TABLE_RANK)
            slot = oracle.static_cache_build(indptr, int(cached * n_nodes))
        for it, n in enumerate(sizes):
            seeds = [rng.integers(0, n_nodes, n).astype(np.int32) for _ in range(group)]
            if group == 1:
                srv.run_once(seeds[0], rng_seed=it + 1, stream=stream)
            else:
                srv.run_group(list(range(group)), [0] * group, seeds=seeds, rng_seeds=[it + 1 + k for k in range(group)], stream=stream)
            for k in range(group):
                g = srv.fetch(pipe=k, stream=stream)
                assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds[k], [fanout], it + 1 + k))
                np.testing.assert_array_equal(g.cache_index, slot[g.ids])
                assert g.features.tobytes() == feats.array[g.ids].tobytes()
            routes = srv.routes()
            threads, nodes, _ = SHAPES[shape]
            assert (routes["hop_threads"][0], routes["hop_nodes"][0]) == (threads, threads // lanes * nodes)
            assert routes["early_rows"] == routes["tile_rows"] == (it + 1) * group
        srv.status()
    finally:
        srv.close()
        feats.free()


def srv_alloc(lmi, buffers, n):
    p = ctypes.c_void_p()
    lmi.check(lmi.lib().lmi_device_alloc(n, ctypes.byref(p)))
    buffers.append(p.value)
    return p.value
