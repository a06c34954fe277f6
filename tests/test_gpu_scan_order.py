"""GPU: detection launches that write more than 256 MB with few hits take their tiles XCD by XCD; their rows are those of the generic
scan, whatever the number of tiles leaves over, and do not depend on the launch's size."""

import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _rows(text, variant, shots, calls=1):
    import torch
    import stim_amd
    from stim_amd import _native as N
    s = stim_amd.Circuit(text).compile_detector_sampler(seed=21)
    s.set_engine('symptom')
    if variant == 'generic':
        s.set_scan_variant('generic')
    d = torch.full((shots, (s.num_detectors + 7) // 8), 0xA5, dtype=torch.uint8, device='cuda:0')
    o = torch.full((shots, (s.num_observables + 7) // 8), 0xA5, dtype=torch.uint8, device='cuda:0')
    torch.cuda.synchronize()
    flags = N.MFS_BIT_PACKED | N.MFS_DEVICE_OUTPUT | N.MFS_SEPARATE_OBSERVABLES
    for _ in range(calls):
        N.check(N.lib().mfs_sample(s._h, shots, flags, ctypes.c_void_p(d.data_ptr()), d.stride(0),
                                   ctypes.c_void_p(o.data_ptr()), o.stride(0)))
    return d, o


# Rows of 612 and 1950 bytes: just above 256 MB, and 1 to 7 tiles beyond a multiple of eight.
@pytest.mark.parametrize('d, shots', [(17, 439_000), (17, 32 * 8 * 1800 + 33), (25, 140_000), (25, 16 * 8 * 1200 + 16 * 6 + 5)])
def test_tiles_by_xcd_equal_the_generic_scan(d, shots):
    import torch
    from stim_amd import gen
    text = gen.generate('surface_code:rotated_memory_z', distance=d, rounds=d, after_clifford_depolarization=1e-4,
                        after_reset_flip_probability=1e-4, before_measure_flip_probability=1e-4)
    a = _rows(text, 'fast', shots, 2)
    b = _rows(text, 'generic', shots, 2)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    assert bool(a[0].any())
    few = _rows(text, 'fast', 10_000)
    first = _rows(text, 'fast', shots)
    assert torch.equal(few[0], first[0][:10_000]) and torch.equal(few[1], first[1][:10_000])
