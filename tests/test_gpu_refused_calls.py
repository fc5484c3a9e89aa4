"""A call that is refused leaves its pipes and its server as they were: the batch that follows on the same pipes starts from
wiped tables and scan words, whatever the memory of a new server held before."""
import numpy as np
import pytest

from conftest import random_graph
from test_gpu_parity import assert_batch_equal, make_features

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("word", [0, (1 << 32) | 7, (2 << 32) | 7])
@pytest.mark.parametrize("fuse", [0, 1])
def test_a_refused_group_leaves_its_pipes_as_they_were(lmi, oracle, word, fuse):
    rng = np.random.default_rng(fuse)
    n_nodes, batch, dim, fanout = 30_000, 700, 8, [12, 6]
    indptr, indices = random_graph(rng, n_nodes, 12, hubs=3, hub_deg=900)
    feats = make_features(lmi, rng, n_nodes, dim)
    # the new server's buffers come from memory that somebody else has used: as scan words a partial and a whole sum
    junk = np.full(1 << 18, word, np.uint64)
    held = []
    for _ in range(24):
        ptr = lmi.C.c_void_p()
        lmi.check(lmi.lib().lmi_device_alloc(junk.nbytes, lmi.C.byref(ptr)))
        lmi.check(lmi.lib().lmi_copy_to_device(ptr, junk.ctypes.data, junk.nbytes))
        held.append(ptr)
    for ptr in held:
        lmi.check(lmi.lib().lmi_device_free(ptr))
    srv = lmi.Server(batch, fanout, dim, pipes=3, seed=3)
    stream = lmi.stream_create()
    train = rng.choice(n_nodes, 5 * batch, replace=False).astype(np.int32)

    def refused(pipes, counters, seeds=None):
        with pytest.raises(lmi.LegionError):
            srv.run_group(pipes, counters, seeds=seeds, stream=stream)

    def served(pipe, b):
        g = srv.fetch(pipe=pipe, stream=stream)
        assert_batch_equal(g, oracle.sample_batch(indptr, indices, train[b * batch:(b + 1) * batch], fanout, 3 + b))
        assert g.features.tobytes() == feats.array[g.ids].tobytes()

    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.load_idset(lmi.MODE_TRAIN, train)
        srv.tune("fuse_count", fuse)
        # the first batches of the pipes: the second slice lies past the set's end, or has too many seeds
        refused([0, 1], [0, 5])
        refused([1, 0], [0, 0], seeds=[train[:batch], train[:batch + 1]])
        srv.run_once(batch_counter=1, pipe=0, stream=stream)
        served(0, 1)
        srv.run_group([1, 2], [2, 3], stream=stream)
        served(1, 2)
        served(2, 3)
        # where the epochs of the tables run out
        srv.tune("table_epochs", 2)
        for it in range(8):
            refused([0, 1, 2], [0, 1, 5])
            if it % 3 == 2:
                srv.run_group([1, 0], [it % 5, (it + 1) % 5], stream=stream)
                served(1, it % 5)
                served(0, (it + 1) % 5)
            else:
                srv.run_once(batch_counter=it % 5, pipe=it % 2, stream=stream)
                served(it % 2, it % 5)
    finally:
        srv.close()
        feats.free()


def test_a_refused_batch_does_not_age_the_dynamic_cache(lmi, oracle):
    rng = np.random.default_rng(1)
    n_nodes, batch, dim, fanout, sets, ways = 20_000, 300, 16, [8, 4], 200, 4
    indptr, indices = random_graph(rng, n_nodes, 10)
    feats = make_features(lmi, rng, n_nodes, dim)
    host_rows = feats.array.view(np.uint8).reshape(n_nodes, dim * 4)
    srv = lmi.Server(batch, fanout, dim, pipes=2, seed=3)
    cache = oracle.Lru(sets, ways, dim * 4)
    try:
        srv.load_graph(indptr, indices)
        srv.attach_features(feats)
        srv.build_lru_cache(sets, ways)
        for it in range(5):
            with pytest.raises(lmi.LegionError):
                srv.run_once(np.zeros(batch + 1, np.int32), pipe=it % 2)
            with pytest.raises(lmi.LegionError):
                srv.run_once(batch_counter=0, pipe=it % 2)   # no id set
            seeds = rng.choice(n_nodes, batch, replace=False).astype(np.int32)
            srv.run_once(seeds, rng_seed=it + 1, pipe=it % 2)
            o = oracle.sample_batch(indptr, indices, seeds, fanout, it + 1)
            hit = cache.access(o.ids, host_rows)[0]
            g = srv.fetch(pipe=it % 2)
            assert_batch_equal(g, o)
            np.testing.assert_array_equal(g.cache_index, hit)
        keys, use = srv.cache_dump(sets * ways, with_aux=True)
        want = cache.state()
        np.testing.assert_array_equal(keys.ravel(), want[0].ravel())
        np.testing.assert_array_equal(use.ravel(), want[1].ravel())
    finally:
        srv.close()
        feats.free()
