"""GPU: conversions of host rows in many batches (every slot and pinned input buffer used again, a ragged last batch) equal
the conversion of the same rows in device memory, and a batch's size accounts for all of its rows' bytes."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _memory(d, r):
    import stim_amd
    from stim_amd import gen
    return stim_amd.Circuit(gen.generate('surface_code:rotated_memory_z', distance=d, rounds=r))


def _swept(results, sweep_bits):
    """`results` measurements of as many qubits; sweep bit k flips qubit k % results. One detector each, and the observable."""
    import stim_amd
    text = ['R ' + ' '.join(map(str, range(results)))]
    for k in range(0, sweep_bits, results):
        text.append('CX ' + ' '.join(f'sweep[{j}] {j % results}' for j in range(k, min(k + results, sweep_bits))))
    text.append('M ' + ' '.join(map(str, range(results))))
    text += [f'DETECTOR rec[-{results - j}]' for j in range(results)]
    text.append('OBSERVABLE_INCLUDE(0) rec[-1]')
    return stim_amd.Circuit('\n'.join(text) + '\n')


def _rows(rng, shots, bits):
    """Packed random rows, padding bits zero."""
    rows = rng.integers(0, 256, size=(shots, (bits + 7) // 8), dtype=np.uint8)
    if bits % 8:
        rows[:, -1] &= (1 << (bits % 8)) - 1
    return rows


def _on_device(conv, meas, sweep=None):
    import torch
    from stim_amd import _native as N
    shots = meas.shape[0]
    m = torch.from_numpy(meas).to('cuda:0')
    w = torch.from_numpy(sweep).to('cuda:0') if sweep is not None else None
    d = torch.zeros((shots, (conv.num_detectors + 7) // 8), dtype=torch.uint8, device='cuda:0')
    o = torch.zeros((shots, (conv.num_observables + 7) // 8), dtype=torch.uint8, device='cuda:0')
    torch.cuda.synchronize()
    p = ctypes.c_void_p
    N.check(N.lib().mfs_m2d_convert_sweep(
        conv._h, shots, p(m.data_ptr()), m.stride(0), p(w.data_ptr()) if w is not None else None,
        w.stride(0) if w is not None else 0, N.MFS_BIT_PACKED | N.MFS_DEVICE_OUTPUT | N.MFS_SEPARATE_OBSERVABLES,
        p(d.data_ptr()), d.stride(0), p(o.data_ptr()), o.stride(0)))
    return d.cpu().numpy(), o.cpu().numpy()


# 211 and 19 bytes a packed row, 145 bytes a bool row: 4 to 6 batches of 16 MiB.
@pytest.mark.parametrize('d, r, shots, bits', [(13, 9, 330_001, True), (5, 5, 480_001, False)])
def test_many_batches_equal_device_rows(d, r, shots, bits):
    from stim_amd import _native as N
    conv = _memory(d, r).compile_m2d_converter()
    M, D, O = conv.num_measurements, conv.num_detectors, conv.num_observables
    assert M % 16
    packed = _rows(np.random.default_rng(d), shots, M)
    want = _on_device(conv, packed)
    if bits:
        for _ in range(2):
            got = conv.convert(measurements=packed, separate_observables=True, bit_packed=True)
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        return
    # One byte per result, rows apart; results as bits (in padded rows) and as bytes.
    rows = np.full((shots, M + 3), 7, dtype=np.uint8)
    rows[:, :M] = np.unpackbits(packed, axis=1, bitorder='little')[:, :M]
    for flag, nd, no in [(N.MFS_BIT_PACKED, (D + 7) // 8, (O + 7) // 8), (0, D, O)]:
        dets = np.full((shots, nd + 2), 0xA5, dtype=np.uint8)
        obs = np.full((shots, no + 1), 0xA5, dtype=np.uint8)
        N.check(N.lib().mfs_m2d_convert(conv._h, shots, rows.ctypes.data, rows.shape[1],
                                        flag | N.MFS_BYTE_INPUT | N.MFS_SEPARATE_OBSERVABLES, dets.ctypes.data,
                                        dets.shape[1], obs.ctypes.data, obs.shape[1]))
        assert (dets[:, nd:] == 0xA5).all() and (obs[:, no:] == 0xA5).all()
        d_bits, o_bits = dets[:, :nd], obs[:, :no]
        if not flag:
            d_bits = np.packbits(d_bits, axis=1, bitorder='little')
            o_bits = np.packbits(o_bits, axis=1, bitorder='little')
        assert np.array_equal(d_bits, want[0]) and np.array_equal(o_bits, want[1])


@pytest.mark.parametrize('results, sweep_bits, shots', [(8, 3001, 200_003), (121, 120, 700_001)])
def test_wide_sweep_rows_are_part_of_a_batch(results, sweep_bits, shots):
    """Rows of 376 bytes of sweep bits beside one byte of results (75 MB), and of 15 beside 16 (21 MB): several batches, and
    staging of a few batches' size only."""
    import torch
    conv = _swept(results, sweep_bits).compile_m2d_converter()
    rng = np.random.default_rng(results)
    meas, sweep = _rows(rng, shots, results), _rows(rng, shots, sweep_bits)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    got = conv.convert(measurements=meas, sweep_bits=sweep, separate_observables=True, bit_packed=True)
    assert free - torch.cuda.mem_get_info()[0] <= 64 << 20    # two slots of 16 MiB in and 16 MiB out
    want = _on_device(conv, meas, sweep)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    # The first and last rows by their parities.
    some = np.r_[0:200, shots - 200:shots]
    m = np.unpackbits(meas[some], axis=1, bitorder='little')[:, :results]
    w = np.unpackbits(sweep[some], axis=1, bitorder='little')[:, :sweep_bits]
    for k in range(sweep_bits):
        m[:, k % results] ^= w[:, k]
    assert np.array_equal(got[0][some], np.packbits(m, axis=1, bitorder='little'))
    assert np.array_equal(got[1][some][:, 0], m[:, -1])
