"""The end of a batch that ran on the caller's stream alone: another stream that takes the batch waits for that batch and for
none queued behind it, and does not need the stream that carried it any more."""
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
            for old in others + [stream]:
                lmi.check(lmi.lib().lmi_stream_destroy(old))
    finally:
        srv.close()
        feats.free()
