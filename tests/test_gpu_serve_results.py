"""Copying served results to the host: strides that a row does not fit in are refused, and several threads may copy finished
requests of one server at once."""

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _served(requests):
    """A server and the ids of its finished requests: (distance, shots) each."""
    import stim_amd
    from stim_amd import gen
    from stim_amd.serve import Server
    srv = Server(budget_bytes=1 << 30)
    ids = []
    for k, (d, shots) in enumerate(requests):
        text = gen.generate('surface_code:rotated_memory_z', distance=d, rounds=d, after_clifford_depolarization=2e-3,
                            before_measure_flip_probability=2e-3)
        ids.append(srv.submit(stim_amd.Circuit(text).compile_detector_sampler(seed=k), shots, seed=k))
    while not all(srv.done(r) for r in ids):
        srv.step()
    return srv, ids


@pytest.mark.parametrize('shots', [1, 3, 5000])
def test_rows_longer_than_their_stride_are_refused(shots):
    from stim_amd import _native as N
    srv, (r,) = _served([(5, shots)])
    dets, obs = srv.result(r)
    row = dets.shape[1]
    assert row > 1 and obs.shape[1] == 1
    d = np.full((shots, row), 0xA5, dtype=np.uint8)
    o = np.full((shots, 1), 0xA5, dtype=np.uint8)
    copy = N.lib().mfs_server_copy_result
    for dets_stride, obs_stride in [(row - 1, 1), (0, 1), (row, 0)]:
        with pytest.raises(RuntimeError):
            N.check(copy(srv._h, r, d.ctypes.data, dets_stride, o.ctypes.data, obs_stride))
        assert (d == 0xA5).all() and (o == 0xA5).all()
    # A part without a destination has no stride to fit.
    N.check(copy(srv._h, r, d.ctypes.data, row, None, 0))
    assert np.array_equal(d, dets) and (o == 0xA5).all()
    N.check(copy(srv._h, r, None, 0, o.ctypes.data, 1))
    assert np.array_equal(o, obs)


def test_results_copied_by_several_threads_at_once():
    """Requests of one batch and of several, small ones on the compute stream and large ones on the copy stream."""
    srv, ids = _served([(11, 160_001), (3, 501), (9, 60_000), (13, 90_001), (5, 1), (7, 30_003)])
    want = [srv.result(r) for r in ids]
    got = {}
    start = threading.Barrier(len(ids))

    def copy(k):
        start.wait()
        got[k] = [srv.result(ids[k]) for _ in range(3)]

    threads = [threading.Thread(target=copy, args=(k,)) for k in range(len(ids))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    for k, w in enumerate(want):
        for g in got[k]:
            assert np.array_equal(g[0], w[0]) and np.array_equal(g[1], w[1]), k
