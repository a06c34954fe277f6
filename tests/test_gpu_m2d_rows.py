"""GPU: conversions with rows on lanes, four blocks a half-wave, at its edges: numbers of blocks that leave one to four in a
group, rows whose last bytes are fewer than 16 or 4, both widths of workgroup and both sides of the lines between them, columns
summed into slots and columns walked as lists, sweep bits, against the parities computed with numpy."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _circuit(M, D, terms, sweep, rng):
    text = [f'R 0 {M - 1}']
    if sweep:
        text += [f'CX sweep[{k}] {k % M}' for k in range(sweep)]
    text.append('M ' + ' '.join(map(str, range(M))))
    cols = [rng.choice(M, size=min(M, int(rng.integers(1, terms + 1))), replace=False) for _ in range(D)]
    text += ['DETECTOR ' + ' '.join(f'rec[{int(i) - M}]' for i in c) for c in cols]
    return '\n'.join(text) + '\n', cols


@pytest.mark.parametrize('M, D, terms, sweep, shots', [
    (1025, 1100, 4, 0, 40), (1055, 1021, 5, 0, 100), (1088, 1120, 3, 0, 8192), (1089, 1057, 9, 0, 8193),   # 33 to 35 blocks
    (5631, 5632, 4, 0, 33), (5633, 5600, 4, 0, 33),                         # 176 and 177 blocks, one subtile a unit
    (3839, 3840, 4, 0, 8300), (3841, 3841, 4, 0, 8300),                     # 120 and 121, up to 512 subtiles
    (4607, 4608, 3, 0, 16500), (4609, 4609, 3, 0, 16500),                   # 144 and 145, beyond
    (65, 70, 3, 0, 742_000), (65, 70, 3, 0, 743_000),                       # many shots of three blocks
    (4000, 1200, 9, 1100, 300), (100, 2200, 9, 37500, 40),                  # sweep bits; no room for slots: lists
])
def test_rows_on_lanes(M, D, terms, sweep, shots):
    import torch
    import stim_amd
    from stim_amd import _native as N
    rng = np.random.default_rng(M * 7 + D)
    text, cols = _circuit(M, D, terms, sweep, rng)
    conv = stim_amd.Circuit(text).compile_m2d_converter()
    conv.set_kernel('whole')
    meas = rng.random((shots, M), dtype=np.float32) < 0.5
    flips = rng.random((shots, sweep), dtype=np.float32) < 0.5
    sent = meas.copy()
    for k in range(sweep):
        meas[:, k % M] ^= flips[:, k]
    want = np.zeros((shots, D), dtype=bool)
    for j, c in enumerate(cols):
        want[:, j] = np.logical_xor.reduce(meas[:, c], axis=1)
    want = np.packbits(want, axis=1, bitorder='little')
    packed = np.packbits(sent, axis=1, bitorder='little')
    sweeps = torch.from_numpy(np.packbits(flips, axis=1, bitorder='little')).to('cuda:0')
    row, out_row = packed.shape[1], want.shape[1]
    for stride in (row, row + 5, (row + 15) // 16 * 16):
        src = torch.zeros((shots, stride), dtype=torch.uint8, device='cuda:0')
        src[:, :row] = torch.from_numpy(packed).to('cuda:0')
        dst = torch.full((shots, out_row + 3), 0xA5, dtype=torch.uint8, device='cuda:0')
        torch.cuda.synchronize()
        N.check(N.lib().mfs_m2d_convert_sweep(
            conv._h, shots, ctypes.c_void_p(src.data_ptr()), stride, ctypes.c_void_p(sweeps.data_ptr()) if sweep else None,
            sweeps.stride(0) if sweep else 0, N.MFS_BIT_PACKED | N.MFS_DEVICE_OUTPUT, ctypes.c_void_p(dst.data_ptr()),
            out_row + 3, None, 0))
        got = dst.cpu().numpy()
        assert np.array_equal(got[:, :out_row], want), stride
        assert (got[:, out_row:] == 0xA5).all()
