"""Copying served results to the host: strides that a row does not fit in are refused."""

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
