"""The host pipeline (stim_amd/csrc/host_pipe.h) on streams that are host threads, under ThreadSanitizer and
AddressSanitizer (no GPU needed): rows of calls of several batches through reused slots and pinned input buffers, a call
that ends while another call's kernel is held, an input that is copied while the kernel before it is held, errors
in the middle of a call, and rows of bits that become bytes. A scenario that waits for what is held does not end, and fails by its time limit."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = '/opt/rocm/llvm/bin/clang++'


@pytest.fixture(scope='module', params=['thread', 'address,undefined'])
def driver(request, tmp_path_factory):
    source = os.path.join(ROOT, 'tests', 'sanitize', 'host_pipe_driver.cc')
    if not os.path.exists(CLANG) or not os.path.exists(source):
        pytest.skip('needs ROCm clang++ and the driver source')
    exe = str(tmp_path_factory.mktemp('host_pipe') / 'driver')
    r = subprocess.run([CLANG, '-x', 'c++', '-O1', '-g', '-std=c++17', '-pthread', '-D__HIP_PLATFORM_AMD__',
                        '-I/opt/rocm/include', '-I' + os.path.join(ROOT, 'stim_amd', 'csrc'), '-fsanitize=' + request.param,
                        '-fno-omit-frame-pointer', source, '-o', exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return exe


@pytest.mark.parametrize('scenario', ['rows', 'callers', 'overlap', 'errors', 'bits'])
def test_host_pipeline(driver, scenario):
    r = subprocess.run([driver, scenario], capture_output=True, text=True, timeout=60,
                       env=dict(os.environ, TSAN_OPTIONS='halt_on_error=1:exitcode=25', ASAN_OPTIONS='detect_leaks=1'))
    assert r.returncode == 0 and r.stdout.endswith('ok\n'), r.stdout[-500:] + r.stderr[-4000:]
