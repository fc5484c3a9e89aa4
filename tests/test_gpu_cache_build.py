"""Cache construction: the hot set where its threshold key lies at the edges of the histogram's bins, caches built again in
the same and in other sizes and kinds, and quantised rows around the lengths that stay in registers."""
import numpy as np
import pytest

from test_gpu_parity import make_features

pytestmark = pytest.mark.gpu


def graph_of_degrees(deg):
    indptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
    return indptr, (np.arange(indptr[-1]) % len(deg)).astype(np.int32)


@pytest.mark.parametrize("degrees", [
    [0] * 300,                                             # every key zero
    [7] * 300,                                             # one key
    [1, 0] * 150,
    [40_000, 40_001, 9_000, 8_191, 8_192, 8_193] + [4_096, 4_095, 4_097] * 20 + [3, 2, 1, 0] * 60,
    list(range(300)),
])
def test_hot_set_at_any_threshold_and_rebuilt(lmi, oracle, degrees):
    indptr, indices = graph_of_degrees(degrees)
    n = len(degrees)
    feats = make_features(lmi, np.random.default_rng(0), n, 8)
    srv = lmi.Server(4, [2], 8)
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        for step, cap in enumerate([1, 2, 3, 4, 6, 7, 7, 40, 66, 67, n // 2, n - 1, n, n]):
            (srv.build_int8_cache if step % 5 == 4 else srv.build_static_cache)(cap, step % 3)
            np.testing.assert_array_equal(srv.cache_dump(n), oracle.static_cache_build(indptr, cap))
            if step % 4 == 3:
                srv.build_lru_cache(4, 2)
        srv.build_static_cache(n, 2)
        with pytest.raises(lmi.LegionError):
            srv.build_static_cache(0, 2)
        with pytest.raises(lmi.LegionError):
            srv.cache_dump(n)   # a refused build leaves no cache
        srv.build_static_cache(n, 2)
        srv.run_once(np.arange(4, dtype=np.int32), rng_seed=1)
        g = srv.fetch()
        assert g.features.tobytes() == feats.array[g.ids].tobytes()
    finally:
        srv.close()
        feats.free()


@pytest.mark.parametrize("dim", [256, 258, 768, 770, 1536, 1538])
@pytest.mark.parametrize("dtype", [np.float32, np.float16])
def test_quantised_rows_in_registers_or_not(lmi, oracle, dim, dtype):
    rng = np.random.default_rng(dim)
    n = 64
    indptr, indices = graph_of_degrees([3] * n)
    feats = make_features(lmi, rng, n, dim, dtype)
    feats.array[5] = 0
    srv = lmi.Server(n, [2], dim, feat_dtype=lmi.F16 if dtype is np.float16 else lmi.F32)
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.build_int8_cache(n, 0)
        srv.run_once(np.arange(n, dtype=np.int32), rng_seed=1)
        g = srv.fetch()
        q, scale = oracle.quantize_rows(feats.array)
        want = oracle.dequant_rows(q, scale, dtype)[g.ids]
        assert g.features.tobytes() == np.ascontiguousarray(want).tobytes()
    finally:
        srv.close()
        feats.free()
