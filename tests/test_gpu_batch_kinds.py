"""Batches and served requests whose jobs run different scans (direct site entries, outcome records, mechanism records, generic):
each scan's jobs are a launch of their own, and every job's rows equal a plain call's, at few tiles a workgroup and at many."""

import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sampler(golden, kind, seed):
    import stim_amd
    from stim_amd import gen
    if kind == 'mechanisms':
        with open(os.path.join(golden.dir, 'dems', 'surface_d5_r5_folded.dem')) as f:
            return stim_amd.DetectorErrorModel(f.read()).compile_sampler(seed=seed)
    if kind == 'records':
        s = stim_amd.Circuit(golden.circuit('color_d5_r3')).compile_detector_sampler(seed=seed)
    else:
        d = {'direct': 5, 'generic': 7, 'large': 13}[kind]
        s = stim_amd.Circuit(gen.generate('surface_code:rotated_memory_z', distance=d, rounds=d,
                                          after_clifford_depolarization=2e-3)).compile_detector_sampler(seed=seed)
    s.engine_info()
    if kind == 'generic':
        s.set_scan_variant('generic')
    return s


JOBS = [('direct', 70001), ('records', 30003), ('mechanisms', 50005), ('generic', 20001), ('direct', 1), ('records', 200000),
        ('mechanisms', 777)]


def _plain(s, shots):
    return s.sample(shots, bit_packed=True, separate_observables=True) if hasattr(s, 'set_engine') else \
        s.sample(shots, bit_packed=True)[:2]


@pytest.mark.parametrize('jobs', [JOBS, JOBS[::-1] + [('large', 1_400_001)], [('records', 5000), ('mechanisms', 5000)]])
def test_mixed_batch_equals_plain_calls(golden, jobs):
    from stim_amd.batch import BatchSampler
    batch = BatchSampler([(_sampler(golden, kind, 100 + k), n) for k, (kind, n) in enumerate(jobs)])
    assert batch.info()['kernel_jobs'] == len(jobs)
    ref = [_sampler(golden, kind, 100 + k) for k, (kind, _) in enumerate(jobs)]
    for replay in range(3):
        got = batch.run(use_graph=replay > 0)
        for k, (s, (_, n)) in enumerate(zip(ref, jobs)):
            for a, b in zip(got[k], _plain(s, n)):
                assert np.array_equal(a.cpu().numpy(), b), (replay, k)


def test_mixed_requests_equal_requests_alone(golden):
    from stim_amd.serve import Server
    kinds = ['direct', 'records', 'mechanisms', 'generic']
    samplers = {kind: _sampler(golden, kind, 7) for kind in kinds}

    def serve(requests, step):
        srv = Server(budget_bytes=1 << 30, step_cost_bytes=step)
        ids = [srv.submit(samplers[kind], shots, seed=seed) for kind, shots, seed in requests]
        while not all(srv.done(r) for r in ids):
            srv.step()
        return [srv.result(r) for r in ids]

    requests = [(kinds[k % 4], [3001, 60000, 1][k % 3], k) for k in range(13)]
    mixed = serve(requests, 1e6)
    for k, request in enumerate(requests):
        (dets, obs), = serve([request], 2e9)
        assert np.array_equal(mixed[k][0], dets) and np.array_equal(mixed[k][1], obs), k
