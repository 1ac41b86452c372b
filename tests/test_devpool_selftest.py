"""The pool that keeps a bar's device memory for the next one, run on the CPU over a
stand-in allocator (host build with AddressSanitizer): fit, limit, devices apart,
memory given back, threads."""
import os
import subprocess

from scadyn_amd import build


def test_device_pool():
    src, exe = build.SELFTESTS['devpool']
    deps = [os.path.join(build.CSRC, f) for f in (src, 'devpool.hpp')]
    if not os.path.exists(build.LIB):
        build.build()
    if not os.path.exists(exe) or any(os.path.getmtime(d) > os.path.getmtime(exe) for d in deps):
        build.build_selftest(which='devpool')
    env = dict(os.environ, ASAN_OPTIONS='detect_leaks=0')
    r = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-4000:]
    assert ' 0 failures' in r.stdout


def test_device_pool_built_by_the_host_compiler(tmp_path):
    """It optimises less away: reads that the device compiler drops stay and are checked."""
    src = os.path.join(build.CSRC, build.SELFTESTS['devpool'][0])
    exe = str(tmp_path / 'devpool_selftest')
    cmd = ['g++', '-x', 'c++', '-std=c++17', '-g', '-O1', '-fsanitize=address', '-pthread', '-o', exe, src]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    env = dict(os.environ, ASAN_OPTIONS='detect_leaks=0')
    r = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-4000:]
