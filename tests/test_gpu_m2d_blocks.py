"""GPU: the whole-record conversion kernel at the edges of its layout (32-column blocks on lanes, 32-shot subtiles
grouped per workgroup): block and word remainders, rows of 1 to 3 trailing bytes, columns of 0 to 12 terms (inline,
summed into slots, and listed where slots do not fit), tight and padded device rows, against the parities
computed with numpy."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _circuit(M, D, O, terms, rng):
    """M results of M qubits, half of them prepared in 1; columns over random results, term counts 0 .. terms."""
    ones = [q for q in range(M) if q % 2]
    text = ['R ' + ' '.join(map(str, range(M)))]
    if ones:
        text.append('X ' + ' '.join(map(str, ones)))
    text.append('M ' + ' '.join(map(str, range(M))))
    cols = []
    for j in range(D + O):
        n = min(M, int(rng.integers(0, terms + 1)) if j else terms)
        idx = rng.choice(M, size=n, replace=False)
        name = 'DETECTOR' if j < D else f'OBSERVABLE_INCLUDE({j - D})'
        text.append(name + ' ' + ' '.join(f'rec[{int(i) - M}]' for i in idx))
        cols.append(idx)
    return '\n'.join(text) + '\n', cols


def _expected(meas, cols):
    out = np.zeros((meas.shape[0], len(cols)), dtype=bool)
    for j, idx in enumerate(cols):
        ref = sum(int(i) % 2 for i in idx) % 2
        out[:, j] = (meas[:, idx].sum(axis=1) + ref) % 2
    return out


@pytest.mark.parametrize('M, D, O, terms, shots', [
    (1, 1, 0, 1, 1), (3, 2, 1, 2, 33), (24, 31, 2, 3, 64), (31, 32, 9, 5, 95), (33, 33, 1, 12, 31),
    (145, 120, 1, 4, 40001), (2049, 2057, 3, 2, 65), (4160, 4095, 1, 6, 70), (16400, 16417, 1, 3, 33),
    (30000, 12000, 2, 8, 40),   # too many long columns for slots next to the record: listed
    # Both sides of the lines between rows on lanes and blocks on lanes: 112 and 113 blocks, 256 and 257 subtiles with 32 and
    # 33 blocks, many shots of few blocks.
    (3584, 3583, 1, 6, 100), (3500, 3585, 2, 6, 100), (1024, 1023, 1, 5, 8192), (1000, 1024, 1, 5, 8193),
    (1000, 1025, 1, 5, 8193), (3, 2, 1, 2, 1600001), (33, 33, 1, 12, 800001),
])
def test_whole_record_kernel_layout_edges(M, D, O, terms, shots):
    import torch
    import stim_amd
    from stim_amd import _native as N
    rng = np.random.default_rng(M + D)
    text, cols = _circuit(M, D, O, terms, rng)
    conv = stim_amd.Circuit(text).compile_m2d_converter()
    assert (conv.num_measurements, conv.num_detectors, conv.num_observables) == (M, D, O)
    conv.set_kernel('whole')
    meas = rng.random((shots, M)) < 0.4
    want = _expected(meas, cols)
    packed = np.packbits(meas, axis=1, bitorder='little')
    d, o = conv.convert(measurements=packed, separate_observables=True)
    np.testing.assert_array_equal(d, want[:, :D])
    np.testing.assert_array_equal(o, want[:, D:])
    got = conv.convert(measurements=packed, append_observables=True, bit_packed=True)
    np.testing.assert_array_equal(got, np.packbits(want, axis=1, bitorder='little'))
    # Device rows: tight, padded to odd and to 16-byte strides.
    row, out_row = packed.shape[1], (D + O + 7) // 8
    for stride in (row, row + 3, (row + 15) // 16 * 16):
        src = torch.zeros((shots, stride), dtype=torch.uint8, device='cuda:0')
        src[:, :row] = torch.from_numpy(packed).to('cuda:0')
        dst = torch.full((shots, out_row + 1), 0xA5, dtype=torch.uint8, device='cuda:0')
        torch.cuda.synchronize()
        flags = N.MFS_BIT_PACKED | N.MFS_DEVICE_OUTPUT | N.MFS_APPEND_OBSERVABLES
        N.check(N.lib().mfs_m2d_convert(conv._h, shots, ctypes.c_void_p(src.data_ptr()), stride, flags,
                                        ctypes.c_void_p(dst.data_ptr()), out_row + 1, None, 0))
        res = dst.cpu().numpy()
        np.testing.assert_array_equal(res[:, :out_row], np.packbits(want, axis=1, bitorder='little'))
        assert (res[:, out_row] == 0xA5).all()   # nothing past a row's last byte


@pytest.mark.parametrize('family, d, r, shots', [('repetition_code:memory', 3, 2, 1), ('surface_code:rotated_memory_z', 3, 3, 33),
                                                 ('surface_code:rotated_memory_x', 5, 4, 40001), ('surface_code:rotated_memory_z', 13, 9, 4099),
                                                 ('surface_code:rotated_memory_z', 25, 3, 321), ('repetition_code:memory', 3, 2, 1700001)])
def test_expanded_records_keep_their_detection_events(family, d, r, shots):
    """Expanded records, with several subtiles per workgroup (many shots) and with one: the reference sample only
    inverts columns, so records with and without it convert to the same detection events; and a call in two parts
    of whole tiles draws the same records."""
    import stim_amd
    from stim_amd import gen
    text = gen.generate(family, distance=d, rounds=r, after_clifford_depolarization=2e-3,
                        before_measure_flip_probability=2e-3, after_reset_flip_probability=2e-3)
    c = stim_amd.Circuit(text)
    rows = {}
    for skip in (False, True):
        s = c.compile_sampler(seed=9, skip_reference_sample=skip)
        s.set_engine('expansion')
        rows[skip] = s.sample(shots, bit_packed=True)
    conv = c.compile_m2d_converter()
    a = conv.convert(measurements=rows[False], append_observables=True)
    b = c.compile_m2d_converter(skip_reference_sample=True).convert(measurements=rows[True], append_observables=True)
    np.testing.assert_array_equal(a, b)
    assert shots == 1 or a.any()
    again = c.compile_sampler(seed=9)
    again.set_engine('expansion')
    if shots > 8192:
        parts = [again.sample(8192, bit_packed=True), again.sample(shots - 8192, bit_packed=True)]
        np.testing.assert_array_equal(np.concatenate(parts), rows[False])
