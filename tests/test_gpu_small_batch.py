"""Batches sampled by one workgroup: the same outputs as the oracle and as the general path (small_edges = 0), at seed
counts around a wavefront, more known nodes than the workgroup keeps rows of, tables bounded by the graph or by the batch."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu

SHAPES = [  # nodes, mean degree, batch, fanouts
    (30_000, 9, 65, [10, 5]),
    (30_000, 9, 17, [5, 4, 3]),
    (30_000, 30, 300, [4, 3]),     # 1 500 known nodes at the second hop
    (30_000, 40, 90, [64]),        # lane groups of a wavefront
    (900, 12, 64, [25, 10]),       # every node of the graph in the table
    (5, 3, 3, [1, 1, 1]),
]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("cache", ["static", "int8", "none"])
def test_small_batches_match_the_oracle_and_the_general_path(lmi, oracle, shape, cache):
    n_nodes, deg, batch, fanout = shape
    rng = np.random.default_rng(n_nodes + batch)
    indptr, indices = random_graph(rng, n_nodes, deg, hubs=min(3, n_nodes), hub_deg=900)
    feats = make_features(lmi, rng, n_nodes, 48)
    srv = lmi.Server(batch, fanout, 48, pipes=3, seed=3)
    stream = lmi.stream_create()
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        if cache == "static":
            srv.build_static_cache(max(1, n_nodes // 4), n_nodes % 3)
        elif cache == "int8":
            srv.build_int8_cache(max(1, n_nodes // 4), 2)
        slot = oracle.static_cache_build(indptr, max(1, n_nodes // 4))
        for it, n in enumerate([batch, 0, 1, min(64, batch), batch // 2]):
            seeds = rng.integers(0, n_nodes, n).astype(np.int32)   # repeated ones among them
            got = []
            for edges in (1 << 20, 0):
                srv.tune("small_edges", edges)
                before = srv.routes()["small_batches"]
                srv.run_once(seeds, rng_seed=it + 1, pipe=2, stream=stream)
                got.append(srv.fetch(pipe=2, stream=stream))
                srv.run_group([0, 1], [0, 0], seeds=[seeds, seeds[:n // 2]], rng_seeds=[it + 1, it + 2], stream=stream)
                got += [srv.fetch(pipe=0, stream=stream), srv.fetch(pipe=1, stream=stream)]
                assert srv.routes()["small_batches"] - before == (3 if edges else 0)
            for k, (a, b) in enumerate(zip(got[:3], got[3:])):
                mine, key = (seeds[:n // 2], it + 2) if k == 2 else (seeds, it + 1)
                assert_batch_equal(a, oracle.sample_batch(indptr, indices, mine, fanout, key))
                assert_batch_equal(a, b)
                np.testing.assert_array_equal(a.labels, b.labels)
                if cache != "none":
                    np.testing.assert_array_equal(a.cache_index, slot[a.ids])
                assert a.features.tobytes() == b.features.tobytes()
                if cache != "int8":
                    assert a.features.tobytes() == feats.array[a.ids].tobytes()
    finally:
        srv.close()
        feats.free()


def test_conditions_presampling_and_a_table_that_was_never_wiped(lmi, oracle):
    rng = np.random.default_rng(1)
    n_nodes, batch, fanout = 20_000, 32, [10, 5]
    indptr, indices = random_graph(rng, n_nodes, 12)
    feats = make_features(lmi, rng, n_nodes, 16)
    srv = lmi.Server(batch, fanout, 16, pipes=2, seed=9)
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        train = rng.choice(n_nodes, 4 * batch, replace=False).astype(np.int32)
        srv.load_idset(lmi.MODE_TRAIN, train)
        srv.presample(4)
        hot = srv.hotness(n_nodes)
        want = np.zeros(n_nodes, np.uint32)
        for b in range(4):
            o = oracle.sample_batch(indptr, indices, train[b * batch:(b + 1) * batch], fanout, 9 + b)
            np.add.at(want, o.ids, 1)
        np.testing.assert_array_equal(hot, want)
        assert srv.routes()["small_batches"] == 4
        seeds = train[:batch].copy()
        # pipe 1: a small batch first, then the general kernels on the table that it did not touch
        srv.run_once(seeds, rng_seed=5, pipe=1)
        srv.op_batch_generate(seeds, rng_seed=5, pipe=1)
        for hop in range(2):
            srv.op_random_sample(hop, pipe=1)
        assert_batch_equal(srv.fetch(pipe=1, features=False), oracle.sample_batch(indptr, indices, seeds, fanout, 5))
        seeds[7] = n_nodes
        srv.run_once(seeds, rng_seed=5)
        with pytest.raises(lmi.LegionError):
            srv.fetch()
        seeds[7] = 0
        srv.run_once(seeds, rng_seed=5)
        with pytest.raises(lmi.LegionError):
            srv.status(clear=True)
        assert_batch_equal(srv.fetch(features=False), oracle.sample_batch(indptr, indices, seeds, fanout, 5))
    finally:
        srv.close()
        feats.free()


def test_segments_looked_up_in_another_cache_than_they_were_sampled_beside(lmi, oracle):
    """A batch sampled by one workgroup leaves no dedup table in memory; a lookup in a dynamic cache built afterwards, which
    offers a repeated seed once, does not need it."""
    rng = np.random.default_rng(4)
    n_nodes, batch, dim, fanout, sets, ways = 20_000, 65, 16, [10, 5], 40, 8
    indptr, indices = random_graph(rng, n_nodes, 9)
    feats = make_features(lmi, rng, n_nodes, dim)
    srv = lmi.Server(batch, fanout, dim, pipes=2, seed=9)
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.build_lru_cache(sets, ways)
        for it in range(3):   # the clock of the cache moves on
            srv.run_once(rng.integers(0, n_nodes, batch).astype(np.int32), rng_seed=it + 1)
        srv.build_static_cache(n_nodes // 4)
        seeds = rng.integers(0, n_nodes, batch).astype(np.int32)
        seeds[[5, 40, 64]] = seeds[3]
        srv.run_once(seeds, rng_seed=7, pipe=1)
        o = oracle.sample_batch(indptr, indices, seeds, fanout, 7)
        assert_batch_equal(srv.fetch(pipe=1), o)
        assert srv.routes()["small_batches"] == 1   # not with the dynamic cache
        srv.build_lru_cache(sets, ways)
        cache = oracle.Lru(sets, ways, dim * 4)
        hit = cache.access(o.ids, feats.array.view(np.uint8).reshape(n_nodes, dim * 4))[0]
        for segment in range(3):
            srv.op_cache_lookup(segment, pipe=1)
        srv.op_io_complete(pipe=1)
        g = srv.fetch(pipe=1)
        np.testing.assert_array_equal(g.cache_index, hit)
        assert g.features.tobytes() == feats.array[o.ids].tobytes()
        keys = srv.cache_dump(sets * ways)
        assert (keys >= 0).any()
        np.testing.assert_array_equal(keys.ravel(), cache.state()[0].ravel())
    finally:
        srv.close()
        feats.free()
