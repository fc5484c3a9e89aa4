"""The gather that serves hits and misses in one pass on the caller's stream: row sizes at the edges of its
16-byte units, tables behind the host link and in HBM, caches that hold nothing, something and everything."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cached", ["nothing", "some", "all"])
@pytest.mark.parametrize("where", ["host", "device"])
@pytest.mark.parametrize("dim,dtype", [(4, np.float32), (5, np.float32), (66, np.float16), (100, np.float32), (1024, np.float32),
                                       (256, np.float32), (1025, np.float32), (1433, np.float32)])
def test_hits_and_misses_in_one_pass(lmi, oracle, dim, dtype, where, cached):
    rng = np.random.default_rng(dim)
    n_nodes, batch, fanout = 20_000, 400, [12, 6]     # the worst case of a batch is above 1 MB for every row size but 16 B
    indptr, indices = random_graph(rng, n_nodes, 12, hubs=3, hub_deg=900)
    feats = make_features(lmi, rng, n_nodes, dim, dtype)
    srv = lmi.Server(batch, fanout, dim, feat_dtype=lmi.F16 if dtype == np.float16 else lmi.F32, pipes=2, seed=3)
    stream, table = lmi.stream_create(), lmi.C.c_void_p()
    try:
        srv.load_graph(indptr, indices)
        if where == "host":
            srv.attach_features(feats)
        else:
            lmi.check(lmi.lib().lmi_device_alloc(feats.nbytes, lmi.C.byref(table)))
            lmi.check(lmi.lib().lmi_copy_to_device(table, feats.ptr, feats.nbytes))
            srv.attach_features_device(table, n_nodes)
        if cached != "nothing":
            srv.build_static_cache(n_nodes if cached == "all" else n_nodes // 5, lmi.TABLE_RANK)
        for it in range(4):
            # each batch is read back on its own stream before the next is issued, so that all but the first are
            # gathered in line; the last holds ids outside the graph, which have no row to read
            seeds = rng.choice(n_nodes, batch if it != 1 else 7, replace=False).astype(np.int32)
            if it == 3:
                seeds[5], seeds[50] = -1, n_nodes
            srv.run_once(seeds, rng_seed=20 + it, pipe=it % 2, stream=stream)
            if it == 3:
                with pytest.raises(lmi.LegionError):
                    srv.fetch(pipe=1, stream=stream)
                v = srv.view(1)
                nc = lmi.to_host(v.node_counter, 16, np.int32)
                ids = lmi.to_host(v.ids, int(nc[11]), np.int32)
                rows = lmi.to_host(v.features, len(ids) * dim, dtype).reshape(len(ids), dim)
                good = (ids >= 0) & (ids < n_nodes)
                assert good.sum() == len(ids) - 2
                assert rows[good].tobytes() == feats.array[ids[good]].tobytes()
                continue
            g = srv.fetch(pipe=it % 2, stream=stream)
            o = oracle.sample_batch(indptr, indices, seeds, fanout, 20 + it)
            assert_batch_equal(g, o)
            assert g.features.tobytes() == feats.array[o.ids].tobytes()
            if cached == "some":
                np.testing.assert_array_equal(g.cache_index, oracle.static_cache_build(indptr, n_nodes // 5)[o.ids])
        listed = cached == "nothing" and where == "host" and feats.array.strides[0] > 4096
        assert srv.routes()["one_pass_gathers"] == (0 if listed else 4)
    finally:
        srv.close()
        feats.free()
        if table:
            lmi.check(lmi.lib().lmi_device_free(table))


@pytest.mark.parametrize("dim", [1024, 1025])
@pytest.mark.parametrize("blocks", [-1, 1, 300])
def test_segments_and_groups_without_a_cache(lmi, oracle, dim, blocks):
    """All rows over the host link: rows of up to 4 096 bytes in one pass, longer ones listed, on any grid."""
    rng = np.random.default_rng(dim)
    n_nodes, batch, fanout = 5_000, 100, [6, 4]
    indptr, indices = random_graph(rng, n_nodes, 12)
    feats = make_features(lmi, rng, n_nodes, dim)
    srv = lmi.Server(batch, fanout, dim, pipes=3, seed=3)
    stream = lmi.stream_create()

    def check(pipe, seeds, key):
        g = srv.fetch(pipe=pipe, stream=stream)
        assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds, fanout, key))
        assert g.features.tobytes() == feats.array[g.ids].tobytes()
        assert (g.cache_index == -1).all()

    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.tune("miss_blocks", blocks)
        for it, n in enumerate([batch, 1, 64]):
            seeds = rng.integers(0, n_nodes, n).astype(np.int32)
            srv.op_batch_generate(seeds, rng_seed=it + 1, pipe=0, stream=stream)
            srv.op_cache_lookup(0, pipe=0, stream=stream)
            for hop in range(2):
                srv.op_random_sample(hop, pipe=0, stream=stream)
                srv.op_cache_lookup(hop + 1, pipe=0, stream=stream)
            srv.op_io_complete(pipe=0, stream=stream)
            check(0, seeds, it + 1)
            srv.run_group([0, 1, 2], [0, 0, 0], seeds=[seeds, seeds[:n // 2], seeds[::-1]], rng_seeds=[7, 8, 9], stream=stream)
            check(0, seeds, 7)
            check(1, seeds[:n // 2], 8)
            check(2, np.ascontiguousarray(seeds[::-1]), 9)
    finally:
        srv.close()
        feats.free()
