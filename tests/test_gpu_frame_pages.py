"""The frame kernel's launch shapes: a tile's rows depend on its number alone, not on how many tiles a call has."""

import numpy as np
import pytest

import stim_amd
from stim_amd import gen

pytestmark = pytest.mark.gpu

# Every kind of sparse noise, with as few and as many outcomes as each has, next to sites that share rows.
NOISE = '''
R 0 1 2 3
X_ERROR(0.02) 0 1
PAULI_CHANNEL_1(0.01, 0, 0.03) 2 3
DEPOLARIZE1(0.05) 0 1 2 3
PAULI_CHANNEL_2(0, 0, 0.01, 0, 0, 0, 0, 0.02, 0, 0, 0, 0, 0, 0, 0.01) 0 1 2 3
DEPOLARIZE2(0.1) 1 2
E(0.1) X0 Y1
ELSE_CORRELATED_ERROR(0.2) Z2 X3
HERALDED_ERASE(0.1) 0 1
HERALDED_PAULI_CHANNEL_1(0.01, 0.02, 0.03, 0.04) 2 3
M(0.03) 0 1 2 3
DETECTOR rec[-1]
DETECTOR rec[-2]
DETECTOR rec[-3]
DETECTOR rec[-4]
DETECTOR rec[-5]
DETECTOR rec[-6]
DETECTOR rec[-7]
DETECTOR rec[-8]
'''


def _frame(circuit):
    s = circuit.compile_detector_sampler(seed=77)
    s.set_engine('frame')
    return s


def _clifford(n):
    return gen.random_clifford(n_qubits=n, layers=10, seed=n, px=2e-3, py=1e-3, pz=1e-3, p2=4e-3, mpp_flip=2e-3)


# Tiles of 64 shots (60, 200 and 1500 qubits) and of 32 (5000): one page and several, launches on both sides of the
# lines at 256 and 512 tiles.
@pytest.mark.parametrize('text, few, many', [
    (NOISE * 12, 1000, 64 * 300), (_clifford(60), 64 * 256, 64 * 257), (_clifford(200), 64 * 256 - 5, 64 * 400 + 1),
    (_clifford(1500), 64 * 512, 64 * 513), (_clifford(5000), 32 * 512 - 3, 32 * 513)],
    ids=['noise', 'q60', 'q200', 'q1500', 'q5000'])
def test_rows_do_not_depend_on_the_launch_shape(text, few, many):
    circuit = stim_amd.Circuit(str(text))
    a = _frame(circuit).sample(few, bit_packed=True)
    b = _frame(circuit).sample(many, bit_packed=True)
    assert a.any()
    assert np.array_equal(a, b[:few])


def test_a_tile_that_fills_a_compute_unit():
    n, p, shots = 12000, 0.01, 2048
    qubits = ' '.join(map(str, range(n)))
    circuit = stim_amd.Circuit(f'R {qubits}\nX_ERROR({p}) {qubits}\nM {qubits}\n'
                               + ''.join(f'DETECTOR rec[-{k}]\n' for k in range(1, n + 1)))
    rows = _frame(circuit).sample(shots)
    # Fired entries are binomial: six standard deviations.
    assert abs(int(rows.sum()) - n * shots * p) < 6 * (n * shots * p * (1 - p)) ** 0.5
    # Along one shot and along one detector the counts are binomial too; the largest of that many stays below eight.
    assert abs(rows.sum(axis=1) - n * p).max() < 8 * (n * p * (1 - p)) ** 0.5
    assert abs(rows.sum(axis=0) - shots * p).max() < 8 * (shots * p * (1 - p)) ** 0.5
