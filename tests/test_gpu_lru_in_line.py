"""The LRU cache where its lookup rides in the flag scans (batches taken in order on one stream), beside its lookup as a
launch of its own (batches in flight, another stream, profiled): every mixture leaves the oracle's cache."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ways", [3, 8])
@pytest.mark.parametrize("fanout", [[12, 6], [5, 4, 3]])
def test_lookups_in_flag_scans_and_alone_mixed(lmi, oracle, ways, fanout):
    rng = np.random.default_rng(ways)
    n_nodes, batch, dim, sets = 20_000, 400, 100, 150
    indptr, indices = random_graph(rng, n_nodes, 12, hubs=3, hub_deg=900)
    feats = make_features(lmi, rng, n_nodes, dim)
    host_rows = feats.array.view(np.uint8).reshape(n_nodes, dim * 4)
    srv = lmi.Server(batch, fanout, dim, pipes=2, seed=3)
    streams = [lmi.stream_create(), lmi.stream_create()]
    cache = oracle.Lru(sets, ways, dim * 4)
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.build_lru_cache(sets, ways)
        for it in range(12):
            seeds = rng.integers(0, n_nodes, batch if it % 3 else 65).astype(np.int32)   # repeated ones among them
            seeds[1] = seeds[0]
            stream, pipe = streams[it // 5 % 2], it % 2
            if it == 7:
                srv.profile_enable(1)
            if it == 9:
                srv.profile_enable(0)
            srv.run_once(seeds, rng_seed=it + 1, pipe=pipe, stream=stream)
            o = oracle.sample_batch(indptr, indices, seeds, fanout, it + 1)
            hit = cache.access(o.ids, host_rows)[0]
            if it in (3, 4):
                continue   # not taken before the next batch is issued
            g = srv.fetch(pipe=pipe, stream=stream)
            assert_batch_equal(g, o)
            np.testing.assert_array_equal(g.cache_index, hit)
            assert g.features.tobytes() == feats.array[o.ids].tobytes()
        keys, use = srv.cache_dump(sets * ways, with_aux=True)
        want = cache.state()
        np.testing.assert_array_equal(keys.ravel(), want[0].ravel())
        np.testing.assert_array_equal(use.ravel(), want[1].ravel())
        routes = srv.routes()   # some ways each
        assert 0 < routes["lru_scan_lookups"] < 12 and 0 < routes["lru_place_copies"] < 12
    finally:
        srv.close()
        feats.free()


def test_streams_that_come_and_go_between_batches(lmi, oracle):
    """Streams destroyed behind their batch, unsynchronised: a new one may get the same handle."""
    rng = np.random.default_rng(5)
    n_nodes, batch, dim, sets, ways, fanout = 20_000, 500, 100, 300, 8, [12, 6]
    indptr, indices = random_graph(rng, n_nodes, 12, hubs=3, hub_deg=900)
    feats = make_features(lmi, rng, n_nodes, dim)
    host_rows = feats.array.view(np.uint8).reshape(n_nodes, dim * 4)
    srv = lmi.Server(batch, fanout, dim, pipes=4, seed=3)
    cache = oracle.Lru(sets, ways, dim * 4)
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.build_lru_cache(sets, ways)
        for it in range(24):
            seeds = rng.choice(n_nodes, batch, replace=False).astype(np.int32)
            stream = lmi.stream_create()
            srv.run_once(seeds, rng_seed=it + 1, pipe=it % 4, stream=stream)
            srv.batch_wait(it % 4, stream)
            o = oracle.sample_batch(indptr, indices, seeds, fanout, it + 1)
            hit = cache.access(o.ids, host_rows)[0]
            if it % 4 == 3:
                g = srv.fetch(pipe=it % 4, stream=stream)
                assert_batch_equal(g, o)
                np.testing.assert_array_equal(g.cache_index, hit)
                assert g.features.tobytes() == feats.array[o.ids].tobytes()
            lmi.check(lmi.lib().lmi_stream_destroy(stream))
        lmi.check(lmi.lib().lmi_device_sync())
        keys, use = srv.cache_dump(sets * ways, with_aux=True)
        want = cache.state()
        np.testing.assert_array_equal(keys.ravel(), want[0].ravel())
        np.testing.assert_array_equal(use.ravel(), want[1].ravel())
    finally:
        srv.close()
        feats.free()


@pytest.mark.parametrize("dim,dtype,sets,ways", [
    (2, np.float32, 150, 8),        # 8 bytes: less than a unit, placed and copied apart
    (4, np.float32, 150, 3),        # one unit
    (5, np.float32, 150, 8),        # 20 bytes: units that overlap, at 4-byte alignment
    (66, np.float16, 150, 8),       # 132
    (1433, np.float32, 40, 8),      # 5 732
    (33, np.float32, 6, 64),        # 132, and a tile of 32 misses that grants up to 64 ways each
])
def test_rows_of_every_size_reach_the_cache(lmi, oracle, dim, dtype, sets, ways):
    """Rows copied into the cache are read back as hits by later batches of the same nodes."""
    rng = np.random.default_rng(dim + ways)
    n_nodes, batch, fanout = 5_000, 200, [6, 4]
    indptr, indices = random_graph(rng, n_nodes, 12)
    feats = make_features(lmi, rng, n_nodes, dim, dtype)
    host_rows = feats.array.view(np.uint8).reshape(n_nodes, -1)
    srv = lmi.Server(batch, fanout, dim, feat_dtype=lmi.F16 if dtype == np.float16 else lmi.F32, pipes=2, seed=3)
    stream = lmi.stream_create()
    cache = oracle.Lru(sets, ways, host_rows.shape[1])
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.build_lru_cache(sets, ways)
        hits = 0
        for it in range(6):
            seeds = rng.integers(0, 400, batch).astype(np.int32)   # the same few hundred nodes, repeated ones among them
            srv.run_once(seeds, rng_seed=it // 2 + 1, pipe=it % 2, stream=stream)
            o = oracle.sample_batch(indptr, indices, seeds, fanout, it // 2 + 1)
            slots = cache.access(o.ids, host_rows)[0]
            hits += int((slots >= 0).sum())
            g = srv.fetch(pipe=it % 2, stream=stream)
            assert_batch_equal(g, o)
            np.testing.assert_array_equal(g.cache_index, slots)
            assert g.features.tobytes() == feats.array[o.ids].tobytes()
        assert hits > 100
        keys, use = srv.cache_dump(sets * ways, with_aux=True)
        want = cache.state()
        np.testing.assert_array_equal(keys.ravel(), want[0].ravel())
        np.testing.assert_array_equal(use.ravel(), want[1].ravel())
        routes = srv.routes()
        assert routes["lru_scan_lookups"] == 6 and routes["lru_place_copies"] == (6 if host_rows.shape[1] >= 16 else 0)
    finally:
        srv.close()
        feats.free()
