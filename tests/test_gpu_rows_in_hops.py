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
        before = srv.routes()["one_pass_gathers"]
        sizes = [batch, 0, 1, 64, 256, batch]
        for it, n in enumerate(sizes):
            seeds = rng.integers(0, N_NODES, n).astype(np.int32)   # repeated ones among them
            srv.run_once(seeds, rng_seed=it + 1, pipe=it & 1, stream=stream)
            g = srv.fetch(pipe=it & 1, stream=stream)
            assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds, fanout, it + 1))
            np.testing.assert_array_equal(g.cache_index, slot[g.ids])
            assert g.features.tobytes() == feats.array[g.ids].tobytes()
        if rows or dim <= 1024:   # taken in order from the first: all of it on the caller's stream
            assert srv.routes()["one_pass_gathers"] - before == len(sizes)
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
        srv.status()
    finally:
        for p in buffers:
            lmi.check(lmi.lib().lmi_device_free(p))
        srv.close()
        feats.free()


def srv_alloc(lmi, buffers, n):
    p = ctypes.c_void_p()
    lmi.check(lmi.lib().lmi_device_alloc(n, ctypes.byref(p)))
    buffers.append(p.value)
    return p.value
