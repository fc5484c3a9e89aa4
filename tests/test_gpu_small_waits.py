"""Gather workgroups beside a small batch whose wait for the ids does not end: they leave, and the sampling one gathers every
row.  Forced from the host (no patience at all), and launches of several streams at once, whose workgroups wait side by side."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu

N_NODES, FANOUT = 3_000, [10, 5]


@pytest.fixture(scope="module")
def graph():
    rng = np.random.default_rng(41)
    return rng, *random_graph(rng, N_NODES, 9, hubs=3, hub_deg=800)


def check(srv, oracle, graph, feats, slot, pipe, seeds, key, stream):
    _, indptr, indices = graph
    g = srv.fetch(pipe=pipe, stream=stream)
    assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds, FANOUT, key))
    np.testing.assert_array_equal(g.cache_index, slot[g.ids])
    assert g.features.tobytes() == feats.array[g.ids].tobytes()


@pytest.mark.parametrize("dim", [4, 37, 1433, 4100])
@pytest.mark.parametrize("cached", [0, N_NODES // 3, N_NODES])
def test_rows_that_gather_workgroups_leave(lmi, oracle, graph, dim, cached):
    rng, indptr, indices = graph
    feats = make_features(lmi, rng, N_NODES, dim)
    srv = lmi.Server(24, FANOUT, dim, pipes=2, seed=3)
    stream = lmi.stream_create()
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        slot = np.full(N_NODES, -1, np.int32)
        if cached:
            srv.build_static_cache(cached, lmi.TABLE_RANK)
            slot = oracle.static_cache_build(indptr, cached)
        srv.tune("small_patience", 0)
        before = srv.routes()["small_rows"]
        sizes = [24, 0, 1, 7, 24]
        for it, n in enumerate(sizes):
            seeds = rng.integers(0, N_NODES, n).astype(np.int32)
            srv.run_once(seeds, rng_seed=it + 1, pipe=it & 1, stream=stream)
            check(srv, oracle, graph, feats, slot, it & 1, seeds, it + 1, stream)
        assert srv.routes()["small_rows"] - before == (len(sizes) if cached or dim <= 1024 else 0)
        srv.status()
    finally:
        srv.close()
        feats.free()


def test_several_streams(lmi, oracle, graph):
    """Three servers' groups and one server's single batches, each on a stream of its own, none waited for in between."""
    rng, indptr, indices = graph
    dim, rounds = 37, 6
    feats = make_features(lmi, rng, N_NODES, dim)
    slot = oracle.static_cache_build(indptr, N_NODES)
    servers = []
    try:
        for k in range(4):
            srv = lmi.Server(24, FANOUT, dim, pipes=4, seed=3)
            servers.append((srv, lmi.stream_create()))
            srv.load_graph(indptr, indices)
            srv.attach_features(feats)
            srv.build_static_cache(N_NODES, lmi.TABLE_RANK)
        for it in range(rounds):
            seeds = [[rng.integers(0, N_NODES, 24).astype(np.int32) for _ in range(4)] for _ in servers]
            for k, (srv, stream) in enumerate(servers):
                if k < 3:
                    srv.run_group([0, 1, 2, 3], [0] * 4, seeds=seeds[k], rng_seeds=[10 * it + p + 1 for p in range(4)], stream=stream)
                else:
                    for p in range(4):
                        srv.run_once(seeds[k][p], rng_seed=10 * it + p + 1, pipe=p, stream=stream)
            for k, (srv, stream) in enumerate(servers):
                for p in range(4):
                    check(srv, oracle, graph, feats, slot, p, seeds[k][p], 10 * it + p + 1, stream)
        for srv, _ in servers:
            assert srv.routes()["small_rows"] == 4 * rounds
            srv.status()
    finally:
        for srv, _ in servers:
            srv.close()
        feats.free()
