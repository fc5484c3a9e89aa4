"""The end of a batch on the caller's stream: another stream that takes the batch waits for that batch and for none queued
behind it, and does not need the stream that carried it any more.  The pipe's next batch waits for the stream that took the
batch where that is so without a side stream."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu

NOT_READY = 600   # hipErrorNotReady


def make_server(lmi, cache, batch, n_nodes, dim, rng):
    indptr, indices = random_graph(rng, n_nodes, 25, hubs=3, hub_deg=900)
    feats = make_features(lmi, rng, n_nodes, dim)
    srv = lmi.Server(batch, [12, 8], dim, pipes=3, seed=3)
    srv.load_graph(indptr, indices)
    srv.attach_features(feats)
    if cache == "static":
        srv.build_static_cache(n_nodes, lmi.TABLE_RANK)
    elif cache == "int8":
        srv.build_int8_cache(n_nodes, lmi.TABLE_HASH)
    elif cache == "lru":
        srv.build_lru_cache(n_nodes // 8, 8)
    elif cache == "groups":
        srv.build_static_cache(n_nodes // 2, lmi.TABLE_RANK)
    if cache == "in line":
        srv.tune("split_miss", 0)
    return srv, indptr, indices, feats


@pytest.mark.parametrize("group", [False, True])
@pytest.mark.parametrize("cache", ["static", "int8", "none"])
def test_taking_a_batch_does_not_wait_for_the_next_ones(lmi, oracle, cache, group):
    rng = np.random.default_rng(1)
    n_nodes, batch = 60_000, 2000
    srv, indptr, indices, feats = make_server(lmi, cache, batch, n_nodes, 64, rng)
    runner, taker = lmi.stream_create(), lmi.stream_create()
    try:
        seeds = rng.choice(n_nodes, batch, replace=False).astype(np.int32)
        srv.run_once(seeds, rng_seed=9, pipe=2, stream=runner)
        srv.batch_wait(2, taker)
        lmi.check(lmi.lib().lmi_device_sync())
        if group:
            srv.run_group([0, 2], [0, 0], seeds=[seeds, seeds], rng_seeds=[1, 2], stream=runner)
        else:
            srv.run_once(seeds, rng_seed=1, pipe=0, stream=runner)
        for it in range(300):   # some 100 us each on the device
            srv.run_once(seeds, rng_seed=100 + it, pipe=1, stream=runner)
        srv.batch_wait(0, taker)
        lmi.check(lmi.lib().lmi_stream_sync(taker))
        assert lmi.lib().hipStreamQuery(runner) == NOT_READY, "the taker has waited for the whole queue"
        lmi.check(lmi.lib().lmi_stream_sync(runner))
        assert_batch_equal(srv.fetch(pipe=0, stream=taker), oracle.sample_batch(indptr, indices, seeds, [12, 8], 1))
    finally:
        srv.close()
        feats.free()


@pytest.mark.parametrize("cache", ["static", "int8", "lru", "none", "in line", "groups"])
def test_a_pipe_whose_stream_is_gone(lmi, oracle, cache):
    """groups: their misses are gathered on the side stream, released ahead of the HBM gather."""
    rng = np.random.default_rng(2)
    n_nodes, batch, dim = 20_000, 300, 16
    srv, indptr, indices, feats = make_server(lmi, cache, batch, n_nodes, dim, rng)
    if cache == "lru":
        host_rows, lru = feats.array.view(np.uint8).reshape(n_nodes, dim * 4), oracle.Lru(n_nodes // 8, 8, dim * 4)
    try:
        for it in range(12):
            stream, others = lmi.stream_create(), [lmi.stream_create() for _ in range(it % 3)]
            seeds = rng.choice(n_nodes, batch, replace=False).astype(np.int32)
            if cache == "groups":
                srv.run_group([it % 2, 2], [0, 0], seeds=[seeds, seeds], rng_seeds=[it + 1, 99], stream=stream)
            else:
                srv.run_once(seeds, rng_seed=it + 1, pipe=it % 2, stream=stream)
            srv.batch_wait(it % 2, stream)
            o = oracle.sample_batch(indptr, indices, seeds, [12, 8], it + 1)
            hit = lru.access(o.ids, host_rows)[0] if cache == "lru" else None
            lmi.check(lmi.lib().lmi_stream_sync(stream))
            lmi.check(lmi.lib().lmi_stream_destroy(stream))
            stream = lmi.stream_create()
            if it % 4 != 3:   # now and then the pipe's next batch is the first to ask
                g = srv.fetch(pipe=it % 2, stream=stream)
                assert_batch_equal(g, o)
                if cache == "lru":
                    np.testing.assert_array_equal(g.cache_index, hit)
                if cache != "int8":
                    assert g.features.tobytes() == feats.array[g.ids].tobytes()
            lmi.check(lmi.lib().lmi_stream_sync(stream))
            for old in others + ([stream] if cache in ("static", "int8") else []):   # the others are followed
                lmi.check(lmi.lib().lmi_stream_destroy(old))
    finally:
        srv.close()
        feats.free()


@pytest.mark.parametrize("cache", ["none", "in line", "lru", "groups"])
def test_the_next_batch_of_a_pipe_waits_for_the_stream_that_took_the_last_one(lmi, oracle, cache):
    rng = np.random.default_rng(3)
    n_nodes, batch, dim = 20_000, 300, 16
    srv, indptr, indices, feats = make_server(lmi, cache, batch, n_nodes, dim, rng)
    runner, taker = lmi.stream_create(), lmi.stream_create()
    big, kept = lmi.C.c_void_p(), lmi.C.c_void_p()
    half = 1 << 28
    try:
        lmi.check(lmi.lib().lmi_device_alloc(2 * half, lmi.C.byref(big)))
        size = int(srv.view(0).max_nodes) * dim * 4
        lmi.check(lmi.lib().lmi_device_alloc(size, lmi.C.byref(kept)))

        def serve(seeds, key):
            if cache == "groups":
                srv.run_group([0, 2], [0, 0], seeds=[seeds, seeds], rng_seeds=[key, 99], stream=runner)
            else:
                srv.run_once(seeds, rng_seed=key, pipe=0, stream=runner)

        for it in range(4):
            a, b = (rng.choice(n_nodes, batch, replace=False).astype(np.int32) for _ in range(2))
            serve(a, 2 * it + 1)
            srv.batch_wait(0, taker)
            for _ in range(40):   # some 0.1 ms each, then the read of the outputs
                lmi.check(lmi.lib().lmi_copy_device(big.value + half, big, half, taker))
            lmi.check(lmi.lib().lmi_copy_device(kept, srv.view(0).features, size, taker))
            serve(b, 2 * it + 2)
            lmi.check(lmi.lib().lmi_device_sync())
            o = oracle.sample_batch(indptr, indices, a, [12, 8], 2 * it + 1)
            rows = lmi.to_host(kept, len(o.ids) * dim, np.float32)
            assert rows.tobytes() == feats.array[o.ids].tobytes(), "the next batch has overwritten rows that were being read"
    finally:
        srv.close()
        feats.free()
        for ptr in (big, kept):
            if ptr:
                lmi.check(lmi.lib().lmi_device_free(ptr))
