"""The phases of a profiled batch hold all of its kernels, the last hop's fill among them."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,fanout,group", [(8000, [64], 8), (2000, [15, 15], 6)])
def test_phases_add_up_to_the_device_time_of_a_batch(lmi, batch, fanout, group):
    """Groups on one stream, so many edges and so short rows that the last hop's fill is an eighth of the time: the phases sum
    to 0.97 of the time per group here (the rest is what the events between them cost), to 0.85 without the fill."""
    n, dim, passes = 2_000_000, 4, 40
    stream = lmi.stream_create()
    graph = lmi.synth_graph(5, lmi.zipf_cdf(3.5, 400, 100.0), n, 0)
    feats, rows = lmi.HostBuffer((n, dim), np.float32), lmi.C.c_void_p()
    lmi.synth_features(3, feats)
    lmi.check(lmi.lib().lmi_device_alloc(feats.nbytes, lmi.C.byref(rows)))
    lmi.check(lmi.lib().lmi_copy_to_device(rows, feats.ptr, feats.nbytes))
    srv = lmi.Server(batch, fanout, dim, pipes=group, seed=3)
    try:
        srv.attach_graph_device(*graph[:2], n, graph[2])
        srv.attach_features_device(rows, n)
        srv.load_idset(lmi.MODE_TRAIN, np.random.default_rng(1).choice(n, 16 * batch, replace=False).astype(np.int32))

        def serve(count):
            for i in range(count):
                srv.run_group(list(range(group)), [(i + j) % 16 for j in range(group)], stream=stream)
            lmi.check(lmi.lib().lmi_stream_sync(stream))

        srv.profile_enable(1)
        serve(5)
        shares = []
        for _ in range(3):
            srv.profile_read()
            t = time.perf_counter()
            serve(passes)
            wall = (time.perf_counter() - t) * 1e3
            p = srv.profile_read()
            assert p.batches == passes * group and p.sample_launches == passes
            shares.append((p.sample_ms + p.lookup_ms + p.gather_hit_ms + p.gather_miss_ms) / wall)
        assert 0.92 < max(shares) < 1.01, shares
    finally:
        srv.close()
        lmi.check(lmi.lib().lmi_device_free(rows))
        for ptr in graph[:2]:
            lmi.check(lmi.lib().lmi_device_free(ptr))
        feats.free()
