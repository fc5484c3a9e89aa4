"""Batches sampled by one workgroup whose rows other workgroups of the launch look up and gather: rows from 16 bytes to more
than a tile, row counts around a tile, no seeds, repeated ones, groups, one to three hops, each kind of cache that has it."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu

N_NODES = 3_000


@pytest.fixture(scope="module")
def graph():
    rng = np.random.default_rng(31)
    return rng, *random_graph(rng, N_NODES, 9, hubs=3, hub_deg=800)


@pytest.mark.parametrize("dim", [4, 37, 1433, 4100])
@pytest.mark.parametrize("cache,table", [("static", "hash"), ("static", "rank"), ("full", "direct"), ("none", None)])
@pytest.mark.parametrize("fanout", [[20], [10, 5], [5, 4, 3]])
def test_rows_and_slots(lmi, oracle, graph, dim, cache, table, fanout):
    rng, indptr, indices = graph
    feats = make_features(lmi, rng, N_NODES, dim)
    batch, n_pipes = 24, 8
    srv = lmi.Server(batch, fanout, dim, pipes=n_pipes, seed=3)
    stream = lmi.stream_create()
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        slot = np.full(N_NODES, -1, np.int32)
        if cache != "none":
            rows = N_NODES if cache == "full" else N_NODES // 3
            srv.build_static_cache(rows, {"hash": lmi.TABLE_HASH, "rank": lmi.TABLE_RANK, "direct": lmi.TABLE_DIRECT}[table])
            slot = oracle.static_cache_build(indptr, rows)
        one_pass = cache != "none" or dim <= 1024   # longer rows without a cache are listed

        def check(pipe, seeds, key):
            g = srv.fetch(pipe=pipe, stream=stream)
            assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds, fanout, key))
            np.testing.assert_array_equal(g.cache_index, slot[g.ids])
            assert g.features.tobytes() == feats.array[g.ids].tobytes()

        before = srv.routes()
        sizes = [batch, 0, 1, 7, batch]
        for it, n in enumerate(sizes):   # each taken before the next is issued
            seeds = rng.integers(0, N_NODES, n).astype(np.int32)
            if n > 3:
                seeds[n - 1] = seeds[0]
            srv.run_once(seeds, rng_seed=it + 1, pipe=it & 1, stream=stream)
            check(it & 1, seeds, it + 1)
        after = srv.routes()
        assert after["small_batches"] - before["small_batches"] == len(sizes)
        assert after["one_pass_gathers"] - before["one_pass_gathers"] == (len(sizes) if one_pass else 0)
        assert after["small_rows"] - before["small_rows"] == (len(sizes) if one_pass else 0)
        for it in range(2):
            seeds = [rng.integers(0, N_NODES, 1 + (5 * k + it) % batch).astype(np.int32) for k in range(n_pipes)]
            srv.run_group(list(range(n_pipes)), [0] * n_pipes, seeds=seeds, rng_seeds=[70 + it + k for k in range(n_pipes)], stream=stream)
            for k in range(n_pipes):
                check(k, seeds[k], 70 + it + k)
        # a group that can miss is in line up to 1 MB; eight batches of long rows are more tiles than its share of the device takes
        worst = batch * int(np.prod([1 + f for f in fanout]))
        in_line = cache != "static" or n_pipes * worst * dim * 4 <= 1 << 20
        assert srv.routes()["small_rows"] - after["small_rows"] == (2 * n_pipes if in_line and dim <= 37 else 0)
        srv.status()
    finally:
        srv.close()
        feats.free()
