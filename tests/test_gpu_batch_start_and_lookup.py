"""Batches that start without a launch of their own (parameters and state set up by the first hop) and whose cache lookup
rides in the flag scans: seed counts at the edges of a lookup block, every table, with and without miss lists, and
conditions that must belong to their batch alone."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("table", [0, 1, 2])
@pytest.mark.parametrize("lists", [False, True])
def test_seed_counts_at_block_edges(lmi, oracle, table, lists):
    rng = np.random.default_rng(table)
    n_nodes, batch, dim, fanout = 30_000, 1000, 100, [7, 3]
    indptr, indices = random_graph(rng, n_nodes, 9, hubs=3, hub_deg=900)
    feats = make_features(lmi, rng, n_nodes, dim)
    srv = lmi.Server(batch, fanout, dim, pipes=3, seed=3)
    stream = lmi.stream_create()
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.build_static_cache(n_nodes // 4, table)
        slot = oracle.static_cache_build(indptr, n_nodes // 4)
        bad = None
        for it, n in enumerate([1, 255, 256, 257, 0, 1000, 511]):
            seeds = rng.integers(0, n_nodes, n).astype(np.int32)
            if n == 257:
                seeds[100] = bad = n_nodes + 5
            pipe = 0 if it % 2 else 1
            if lists:
                srv.run_group([pipe, 2], [0, 0], seeds=[seeds, seeds[:n // 2]], rng_seeds=[it + 1, it + 2], stream=stream)
            else:
                srv.run_once(seeds, rng_seed=it + 1, pipe=pipe, stream=stream)
            if n == 257:   # recorded for this batch ...
                with pytest.raises(lmi.LegionError):
                    srv.fetch(pipe=pipe, stream=stream)
                continue
            g = srv.fetch(pipe=pipe, stream=stream)   # ... and for no later one on the same pipe
            o = oracle.sample_batch(indptr, indices, seeds, fanout, it + 1)
            assert_batch_equal(g, o)
            np.testing.assert_array_equal(g.cache_index, slot[o.ids])
            assert g.features.tobytes() == feats.array[o.ids].tobytes()
        assert bad is not None
        routes = srv.routes()
        assert routes["scan_lookups"] == (14 if lists else 7) and routes["small_batches"] == 0
        with pytest.raises(lmi.LegionError):
            srv.status(clear=True)
        srv.status()
    finally:
        srv.close()
        feats.free()
