"""Every tile of the hop kernel (lane group x threads x nodes per lane group) on both of a tile's edges: batches that are one
node too many for the next smaller tile, repeated seeds among them, and a short last tile."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu

N_NODES, DIM, CUS = 150_000, 4, 256
SHAPES = [(256, 1, 1), (512, 1, 1), (1024, 1, 1), (512, 2, 2), (512, 4, 2), (1024, 4, None)]  # threads, nodes, tiles per CU


@pytest.fixture(scope="module")
def world(lmi):
    rng = np.random.default_rng(11)
    indptr, indices = random_graph(rng, N_NODES, 14, hubs=400, hub_deg=300)
    feats = make_features(lmi, rng, N_NODES, DIM)
    yield rng, indptr, indices, feats
    feats.free()


@pytest.mark.parametrize("shape", range(len(SHAPES)))
@pytest.mark.parametrize("fanout", [3, 7, 13, 29, 50])   # lane groups of 4, 8, 16, 32, 64
def test_tiles_match_the_oracle(lmi, oracle, world, fanout, shape):
    rng, indptr, indices, feats = world
    lanes = 4
    while lanes < fanout:
        lanes *= 2
    if shape == 0:
        batch = 3
    else:   # two batches: a tile per batch more than the tile before may have
        threads, nodes, per_cu = SHAPES[shape - 1]
        batch = per_cu * CUS // 2 * (threads // lanes * nodes) + 1
    srv = lmi.Server(batch, [fanout, 2], DIM, pipes=2, seed=3)
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.build_static_cache(N_NODES // 3, lmi.TABLE_RANK)
        srv.tune("small_edges", 0)
        slot = oracle.static_cache_build(indptr, N_NODES // 3)
        for it in range(2):   # without and with what the kernels noted of the batch before
            seeds = [rng.integers(0, N_NODES, batch).astype(np.int32) for _ in range(2)]
            seeds[1][-1] = seeds[1][0]
            srv.run_group([0, 1], [0, 0], seeds=seeds, rng_seeds=[5 + it, 6 + it])
            threads, nodes, _ = SHAPES[shape]
            routes = srv.routes()
            assert (routes["hop_threads"][0], routes["hop_nodes"][0]) == (threads, threads // lanes * nodes)
            for k in range(2):
                g = srv.fetch(pipe=k)
                assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds[k], [fanout, 2], 5 + it + k))
                np.testing.assert_array_equal(g.cache_index, slot[g.ids])
                assert g.features.tobytes() == feats.array[g.ids].tobytes()
        srv.status()
    finally:
        srv.close()


def test_tiles_behind_a_short_batch(lmi, oracle, world):
    """A full batch takes the same tiles and gathers its rows alike behind a full batch, a short one, and a group whose first
    batch is short; only the fourth short one in a row shapes those behind it."""
    rng, indptr, indices, feats = world
    batch, fanout = 3000, [10, 5]
    srv = lmi.Server(batch, fanout, DIM, pipes=2, seed=3)
    stream = lmi.stream_create()

    def batches(sizes, key, among=np.arange(N_NODES)):
        """Tiles of the hops, and how many of the batches had the last hop's rows gathered by its tiles."""
        before = srv.routes()["tile_rows"]
        seeds = [rng.choice(among, n).astype(np.int32) for n in sizes]
        if len(sizes) == 1:
            srv.run_once(seeds[0], rng_seed=key, stream=stream)
        else:
            srv.run_group([0, 1], [0, 0], seeds=seeds, rng_seeds=[key, key + 1], stream=stream)
        for k in range(len(sizes)):
            g = srv.fetch(pipe=k, stream=stream)
            assert_batch_equal(g, oracle.sample_batch(indptr, indices, seeds[k], fanout, key + k))
            assert g.features.tobytes() == feats.array[g.ids].tobytes()
        r = srv.routes()
        return r["hop_threads"], r["hop_nodes"], r["tile_rows"] - before

    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.tune("small_edges", 0)
        batches([batch], 1)
        one, two = batches([batch], 2), batches([batch, batch], 3)
        for it, before in enumerate([[1], [0], [batch // 5], [1, 1]]):
            batches(before, 10 + it)
            assert batches([batch], 20 + it) == one
        batches([1], 30)
        assert batches([batch, batch], 31) == two
        assert batches([1, batch], 33) == two   # the tiles are those of the larger one, and it leaves its counts
        assert batches([batch, batch], 35) == two
        alone = np.flatnonzero(np.diff(indptr) == 0)   # three of these meet nobody: so would three thousand
        for it in range(3):
            batches([3], 40 + it, alone)
        assert batches([batch], 43) == one
        for it in range(4):
            batches([3], 44 + it, alone)
        assert batches([batch], 48)[0][1] == 256 != one[0][1]
        assert batches([batch], 49) == one
        srv.status()
    finally:
        srv.close()
