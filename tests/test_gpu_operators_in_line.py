"""Operators one by one where lookup and gather of a segment are one launch (batches taken in order), at row sizes around a
tile, every table, seed counts with and without work for all tiles, and seeds outside the graph."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("table", [0, 1, 2])
@pytest.mark.parametrize("dim,tile", [(4, 0), (25, 0), (100, 0), (100, 256), (1433, 0)])
def test_segments_looked_up_while_gathered(lmi, oracle, table, dim, tile):
    rng = np.random.default_rng(dim + table)
    n_nodes, batch, fanout = 20_000, 700, [12, 6]
    indptr, indices = random_graph(rng, n_nodes, 12, hubs=3, hub_deg=900)
    feats = make_features(lmi, rng, n_nodes, dim)
    srv = lmi.Server(batch, fanout, dim, pipes=2, seed=3)
    stream = lmi.stream_create()
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.build_static_cache(n_nodes // 5, table)
        slot = oracle.static_cache_build(indptr, n_nodes // 5)
        if tile:
            srv.tune("gather_tile_rows", tile)
        for it, n in enumerate([batch, 700, 0, 1, 257, 300]):
            seeds = rng.integers(0, n_nodes, n).astype(np.int32)
            if it == 4:
                seeds[3] = -5
            pipe = it % 2
            srv.op_batch_generate(seeds, rng_seed=it + 1, pipe=pipe, stream=stream)
            srv.op_cache_lookup(0, pipe=pipe, stream=stream)
            for hop in range(2):
                srv.op_random_sample(hop, pipe=pipe, stream=stream)
                srv.op_cache_lookup(hop + 1, pipe=pipe, stream=stream)
            srv.op_io_submit(pipe=pipe, stream=stream)
            srv.op_io_complete(pipe=pipe, stream=stream)
            if it == 4:
                with pytest.raises(lmi.LegionError):
                    srv.fetch(pipe=pipe, stream=stream)
                v = srv.view(pipe)
                assert lmi.to_host(v.cache_index, n, np.int32)[3] == -1
                continue
            g = srv.fetch(pipe=pipe, stream=stream)
            assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds, fanout, it + 1))
            np.testing.assert_array_equal(g.cache_index, slot[g.ids])
            assert g.features.tobytes() == feats.array[g.ids].tobytes()
        assert srv.routes()["gather_lookups"] == 6 * 3
    finally:
        srv.close()
        feats.free()
