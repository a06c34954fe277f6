"""Performance cases: the work that programs have this framework do, through its public entry points.

A case is a dict of plain values; its "kind" names the entry point:

  detect   detector sampler of a memory experiment (CompiledDetectorSampler.sample, or the C ABI's mfs_sample
           with rows that stay in device memory)
  measure  measurement sampler of a memory experiment (CompiledMeasurementSampler.sample, mfs_sample)
  clifford detector or measurement sampler of a random-Clifford circuit (device rows)
  dem      detector-error-model sampler (CompiledDemSampler.sample, mfs_sample)
  m2d      conversion of measurement records to detection events (convert, mfs_m2d_convert)
  batch    BatchSampler over surface codes of several distances, replayed as a graph
  serve    Server: a burst of requests over a resident pool, results copied to the host

"out" says where a call's rows go: "device" (bit-packed rows resident in HBM), "packed" (bit-packed numpy arrays)
or "bool" (one byte per entry, numpy, the default of sample()). Sampled rows are whole numbers under a fixed seed;
exact() therefore has nothing to add.
"""

import gzip
import math
import os
import random

import numpy as np
import torch

import stim_amd
from stim_amd import _native as N
from stim_amd import gen
from stim_amd.batch import BatchSampler
from stim_amd.serve import Server

GOLDEN = os.path.join('tests', 'golden')
FAMILIES = ('surface_code:rotated_memory_z', 'surface_code:rotated_memory_x', 'surface_code:unrotated_memory_z',
            'repetition_code:memory')
DEMS = ('surface_d3_r3_folded', 'color_d5_r3', 'rep_d7_r5', 'surface_d5_r5_folded', 'surface_d25_r25_folded')
ROTATED = FAMILIES[0]


def _memory(family, d, r, p):
    return gen.generate(family, distance=d, rounds=r, after_clifford_depolarization=p, after_reset_flip_probability=p,
                        before_measure_flip_probability=p)


def _dem_text(name):
    path = os.path.join(GOLDEN, 'dems', name + '.dem')
    if os.path.exists(path):
        with open(path) as f:
            return f.read()
    with gzip.open(path + '.gz', 'rt') as f:
        return f.read()


# ------------------------------------------------------------------------------------------------- cases

def listed():
    return [
        # The benchmark's headline: 2^20 shots of the d=25 memory experiment for a decoder on the GPU.
        {'name': 'detect_d25', 'kind': 'detect', 'family': ROTATED, 'd': 25, 'r': 25, 'p': 1e-3, 'shots': 1 << 20,
         'out': 'device'},
        # A small code at a realistic, odd shot count: narrow rows, many shots per workgroup tile.
        {'name': 'detect_d5', 'kind': 'detect', 'family': ROTATED, 'd': 5, 'r': 5, 'p': 1e-3, 'shots': 1000003,
         'out': 'device'},
        # The smallest call: a first look at a small code, sample(1000) with every default.
        {'name': 'detect_first_call', 'kind': 'detect', 'family': ROTATED, 'd': 5, 'r': 5, 'p': 2e-3, 'shots': 1000,
         'out': 'bool'},
        # A decoding loop's call (sinter): bit-packed numpy arrays, separate observables, new arrays each call.
        {'name': 'detect_sinter_d13', 'kind': 'detect', 'family': ROTATED, 'd': 13, 'r': 13, 'p': 3e-3,
         'shots': 131071, 'out': 'packed'},
        # Simulation-bound: a random-Clifford circuit whose fault table would cost more than the call.
        {'name': 'clifford_q5000', 'kind': 'clifford', 'qubits': 5000, 'layers': 20, 'p': 1e-3, 'shots': 16384,
         'records': False},
        # Every measurement result of the d=25 memory experiment, resident in HBM.
        {'name': 'measure_d25', 'kind': 'measure', 'family': ROTATED, 'd': 25, 'r': 25, 'p': 1e-3, 'shots': 1 << 20,
         'out': 'device'},
        # The d=25 model: 356,321 mechanisms of some thirty probabilities.
        {'name': 'dem_d25', 'kind': 'dem', 'model': 'surface_d25_r25_folded', 'shots': 1 << 20, 'out': 'device',
         'errors': False},
        # A decoder's training data: detection events and the mechanisms that fired, as numpy bools.
        {'name': 'dem_d5_errors', 'kind': 'dem', 'model': 'surface_d5_r5_folded', 'shots': 20001, 'out': 'bool',
         'errors': True},
        # Conversion of records that are on the GPU already.
        {'name': 'm2d_d25', 'kind': 'm2d', 'family': ROTATED, 'd': 25, 'r': 25, 'shots': 1 << 20, 'out': 'device',
         'separate': False},
        # Conversion of an experiment's records held in numpy.
        {'name': 'm2d_numpy_d11', 'kind': 'm2d', 'family': ROTATED, 'd': 11, 'r': 11, 'shots': 50001, 'out': 'packed',
         'separate': True},
        # Many circuits of a parameter sweep in one replayed launch.
        {'name': 'batch_16', 'kind': 'batch', 'jobs': 16, 'dmax': 21, 'max_shots': 1000000, 'mix': 7},
        # A burst of requests against a resident pool.
        {'name': 'serve_24', 'kind': 'serve', 'requests': 24, 'max_shots': 100000, 'mix': 3},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def shots_for(row_bytes, out, most):
        # Odd counts mostly; the rows of one call stay under 1.5 GB on the device, 64 MB in numpy arrays.
        cap = (1.5e9 if out == 'device' else 6.4e7) / max(row_bytes, 1)
        n = log_int(200, max(400, min(most, cap)))
        return n + 1 if n % 2 == 0 and rng.random() < 0.8 else n

    p = round(math.exp(rng.uniform(math.log(1e-4), math.log(1e-2))), 7)
    kind = rng.choice(['detect', 'detect', 'detect', 'measure', 'measure', 'dem', 'm2d', 'm2d', 'clifford', 'batch',
                       'serve'])
    if kind in ('detect', 'measure', 'm2d'):
        family = rng.choice(FAMILIES)
        d = rng.randint(3, 51) if family.startswith('rep') else rng.randint(3, 13 if 'unrot' in family else 25)
        r = rng.randint(2, d + 3)
        out = rng.choice(['device', 'device', 'packed', 'bool'])
        bits = d * (r + 1) if family.startswith('rep') else d * d * (r + 1) * (2 if 'unrot' in family else 1)
        shots = shots_for(bits if out == 'bool' else bits / 8, out, 1 << 20)
        case = {'kind': kind, 'family': family, 'd': d, 'r': r, 'shots': shots, 'out': out}
        if kind == 'm2d':
            case['separate'] = rng.random() < 0.5
        else:
            case['p'] = p
        return case
    if kind == 'dem':
        model = rng.choice(DEMS)
        out = rng.choice(['device', 'packed', 'bool'])
        errors = out != 'device' and 'd25' not in model and rng.random() < 0.5
        return {'kind': kind, 'model': model, 'out': out, 'errors': errors,
                'shots': shots_for((2000 if 'd25' in model else 220) * (8 if out == 'bool' else 1), out, 1 << 20)}
    if kind == 'clifford':
        return {'kind': kind, 'qubits': 2 * rng.randint(250, 2500), 'layers': 10 * rng.randint(1, 2), 'p': p,
                'shots': log_int(500, 16384), 'records': rng.random() < 0.5}
    if kind == 'batch':
        return {'kind': kind, 'jobs': rng.randint(2, 16), 'dmax': 2 * rng.randint(2, 10) + 1,
                'max_shots': log_int(20000, 1000000), 'mix': rng.randrange(1 << 20)}
    return {'kind': kind, 'requests': rng.randint(4, 24), 'max_shots': log_int(5000, 100000),
            'mix': rng.randrange(1 << 20)}


# ------------------------------------------------------------------------------- circuits of the mixed cases

def _batch_jobs(case):
    """(distance, p, shots) per job: the batched benchmark's distribution, up to the case's limits."""
    rng = random.Random(case['mix'])
    jobs = []
    for _ in range(case['jobs']):
        d = rng.choice(range(3, case['dmax'] + 1, 2))
        p = gen.log_uniform(rng, 1e-4, 5e-3)
        jobs.append((d, p, int(gen.log_uniform(rng, 1e4, case['max_shots']))))
    return jobs


def _serve_mix(case):
    """Pool of (text, detectors, observables) and requests of (pool index, shots), as the serving benchmark draws
    them: surface and repetition codes and a random-Clifford circuit."""
    rng = random.Random(case['mix'])
    pool = []
    for _ in range(4):
        d = rng.choice(range(3, 18, 2))
        pool.append((_memory(ROTATED, d, d, gen.log_uniform(rng, 1e-4, 1e-2)), d * (d * d - 1)))
    for _ in range(4):
        d = rng.randint(3, 51)
        pool.append((_memory('repetition_code:memory', d, d, gen.log_uniform(rng, 1e-4, 1e-2)), (d - 1) * (d + 1)))
    p = gen.log_uniform(rng, 1e-4, 1e-2)
    pool.append((gen.random_clifford(n_qubits=500, layers=10, seed=case['mix'] & 0xFFFF, px=p / 3, py=p / 3, pz=p / 3,
                                     p2=p, mpp_flip=p), 125))
    requests = [(rng.randrange(len(pool)), int(gen.log_uniform(rng, 1e3, case['max_shots'])))
                for _ in range(case['requests'])]
    return pool, requests


# ------------------------------------------------------------------------------------------------ prepare

def _device_rows(shots, bits, pitch=None):
    return torch.empty((shots, pitch or max((bits + 7) // 8, 1)), dtype=torch.uint8, device='cuda:0')


def _random_rows(shots, bits, pitch, seed):
    """Bit-packed device rows of uniform bits with zero padding. Records of a memory experiment are half random
    already (every first-round check of the other basis), and conversion is the same XORs whatever the bits."""
    g = torch.Generator(device='cuda:0')
    g.manual_seed(seed)
    used = (bits + 7) // 8
    rows = torch.zeros((shots, pitch), dtype=torch.uint8, device='cuda:0')
    rows[:, :used] = torch.randint(0, 256, (shots, used), dtype=torch.uint8, device='cuda:0', generator=g)
    if bits % 8:
        rows[:, used - 1] &= (1 << (bits % 8)) - 1
    return rows


def prepare(case, seed):
    kind = case['kind']
    s = {'case': case}
    if kind in ('detect', 'measure', 'm2d'):
        if (case['family'], case['d'], case['r'], case.get('p', 1e-3)) == (ROTATED, 25, 25, 1e-3):
            circuit = stim_amd.Circuit.from_file(os.path.join(GOLDEN, 'circuits', 'surface_d25_r25.stim'))
        else:
            circuit = stim_amd.Circuit(_memory(case['family'], case['d'], case['r'], case.get('p', 1e-3)))
        if kind == 'detect':
            s['sampler'] = circuit.compile_detector_sampler(seed=seed)
        elif kind == 'measure':
            s['sampler'] = circuit.compile_sampler(seed=seed)
        else:
            s['conv'] = conv = circuit.compile_m2d_converter()
            M = conv.num_measurements
            if case['out'] == 'device':
                s['meas'] = _random_rows(case['shots'], M, 16 * ((M + 127) // 128), seed)
                n = conv.num_detectors + (0 if case['separate'] else conv.num_observables)
                s['dets'] = _device_rows(case['shots'], n)
                s['obs'] = _device_rows(case['shots'], conv.num_observables) if case['separate'] else None
            else:
                rows = _random_rows(case['shots'], M, (M + 7) // 8, seed).cpu().numpy()
                if case['out'] == 'bool':
                    rows = np.unpackbits(rows, axis=1, bitorder='little')[:, :M].astype(np.bool_)
                s['meas'] = np.ascontiguousarray(rows)
            return s
    elif kind == 'clifford':
        p = case['p']
        circuit = stim_amd.Circuit(gen.random_clifford(n_qubits=case['qubits'], layers=case['layers'], seed=5,
                                                       px=p / 3, py=p / 3, pz=p / 3, p2=p, mpp_flip=p))
        s['sampler'] = (circuit.compile_sampler(seed=seed) if case['records']
                        else circuit.compile_detector_sampler(seed=seed))
    elif kind == 'dem':
        s['sampler'] = stim_amd.DetectorErrorModel(_dem_text(case['model'])).compile_sampler(seed=seed)
    elif kind == 'batch':
        jobs = _batch_jobs(case)
        samplers = [stim_amd.Circuit(_memory(ROTATED, d, d, p)).compile_detector_sampler(seed=seed + 1000 * k)
                    for k, (d, p, _) in enumerate(jobs)]
        s['samplers'] = samplers
        s['batch'] = BatchSampler([(x, j[2]) for x, j in zip(samplers, jobs)])
        return s
    else:
        pool, requests = _serve_mix(case)
        s['samplers'] = [stim_amd.Circuit(t).compile_detector_sampler(seed=seed + 1000 * k)
                         for k, (t, _) in enumerate(pool)]
        for x in s['samplers']:
            x.engine_info()
        s['requests'] = [(s['samplers'][c], shots, seed + 7 * k) for k, (c, shots) in enumerate(requests)]
        s['server'] = Server(budget_bytes=4e9)
        return s
    if case.get('out', 'device') == 'device':
        # Rows that a program keeps in device memory and fills again on each call.
        x = s['sampler']
        s['dets'] = _device_rows(case['shots'], x.num_detectors if isinstance(x, stim_amd.CompiledDemSampler)
                                 else _columns(x))
        s['obs'] = None if isinstance(x, stim_amd.CompiledMeasurementSampler) else _device_rows(case['shots'],
                                                                                              x.num_observables)
    return s


def _columns(sampler):
    return (sampler.num_measurements if isinstance(sampler, stim_amd.CompiledMeasurementSampler)
            else sampler.num_detectors)


# ---------------------------------------------------------------------------------------------------- run

def run(s):
    case = s['case']
    kind, out, shots = case['kind'], case.get('out', 'device'), case.get('shots', 0)
    if kind == 'batch':
        return [[d, o] for d, o in s['batch'].run(use_graph=True)]
    if kind == 'serve':
        server = s['server']
        ids = [server.submit(x, n, seed) for x, n, seed in s['requests']]
        while not all(server.done(i) for i in ids):
            server.step()
        results = []
        for i in ids:
            results.append(list(server.result(i)))
            server.release(i)
        return results
    if kind == 'm2d':
        conv = s['conv']
        if out == 'device':
            flags = N.MFS_BIT_PACKED | N.MFS_DEVICE_OUTPUT
            flags |= N.MFS_SEPARATE_OBSERVABLES if case['separate'] else N.MFS_APPEND_OBSERVABLES
            meas, dets, obs = s['meas'], s['dets'], s['obs']
            N.check(N.lib().mfs_m2d_convert(conv._h, shots, meas.data_ptr(), meas.stride(0), flags, dets.data_ptr(),
                                            dets.stride(0), obs.data_ptr() if obs is not None else None,
                                            obs.stride(0) if obs is not None else 0))
            return [dets, obs]
        packed = out == 'packed'
        if case['separate']:
            return list(conv.convert(measurements=s['meas'], separate_observables=True, bit_packed=packed))
        return [conv.convert(measurements=s['meas'], append_observables=True, bit_packed=packed)]
    x = s['sampler']
    if out == 'device':
        dets, obs = s['dets'], s['obs']
        flags = N.MFS_BIT_PACKED | N.MFS_DEVICE_OUTPUT | (N.MFS_SEPARATE_OBSERVABLES if obs is not None else 0)
        N.check(N.lib().mfs_sample(x._h, shots, flags, dets.data_ptr(), dets.stride(0),
                                   obs.data_ptr() if obs is not None else None,
                                   obs.stride(0) if obs is not None else 0))
        return [dets, obs]
    packed = out == 'packed'
    if kind == 'dem':
        return list(x.sample(shots, bit_packed=packed, return_errors=case['errors']))
    if kind == 'measure':
        return [x.sample(shots, bit_packed=packed)]
    if packed:
        return list(x.sample(shots, bit_packed=True, separate_observables=True))
    return [x.sample(shots)]


# --------------------------------------------------------------------------------------------------- work

def _row(bits, out):
    return bits if out == 'bool' else (bits + 7) // 8


def work(case):
    """Bytes of a pass: every input row read once and every output row written once."""
    kind, out, shots = case['kind'], case.get('out', 'device'), case.get('shots', 0)
    if kind == 'batch':
        total = sum(n * ((d * (d * d - 1) + 7) // 8 + 1) for d, _, n in _batch_jobs(case))
    elif kind == 'serve':
        pool, requests = _serve_mix(case)
        total = sum(n * ((pool[c][1] + 7) // 8 + 1) for c, n in requests)
    elif kind == 'dem':
        m = stim_amd.DetectorErrorModel(_dem_text(case['model']))
        total = shots * (_row(m.num_detectors, out) + _row(m.num_observables, out)
                         + (_row(m.num_errors, out) if case['errors'] else 0))
    elif kind == 'clifford':
        q, blocks = case['qubits'], case['layers'] // 10
        products, measured = min(500, q // 4), max(2, int(q * 0.1) // 2 * 2)
        n = blocks * (2 * products + measured) if case['records'] else blocks * products
        total = shots * ((n + 7) // 8 + (0 if case['records'] else 1))
    else:
        c = stim_amd.Circuit(_memory(case['family'], case['d'], case['r'], 1e-3))
        D, O, M = c.num_detectors, c.num_observables, c.num_measurements
        if kind == 'measure':
            total = shots * _row(M, out)
        elif kind == 'm2d':
            total = shots * (_row(M, out) + (_row(D, out) + _row(O, out) if case['separate'] else _row(D + O, out)))
        else:
            total = shots * (_row(D, out) + (0 if out == 'bool' else _row(O, out)))
    return {'bytes': float(total), 'flops': 0.0}


def exact(case, seed):
    return None
