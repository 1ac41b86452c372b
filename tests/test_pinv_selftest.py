"""The pseudo-inverse of the equivalent-source fit (pinv.hip) against the plain
one-sided Jacobi loops, run on the CPU by the host self-test: random, repeated and
zero columns, odd and even shapes, and the fit's own kind, with and without AVX2.
Tolerance: none, the bits are the same (the two zeros count as equal)."""
import os
import subprocess

from scadyn_amd import build


def test_pinv_matches_plain_loops():
    src, exe = build.SELFTESTS['pinv']
    deps = [os.path.join(build.CSRC, f) for f in (src, 'pinv.hip', 'internal.hpp')]
    if not os.path.exists(build.LIB):
        build.build()
    if not os.path.exists(exe) or any(os.path.getmtime(d) > os.path.getmtime(exe) for d in deps + [build.LIB]):
        build.build_selftest(which='pinv')
    env = dict(os.environ, ASAN_OPTIONS='detect_leaks=0')
    r = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-4000:]
    assert ' 0 failures' in r.stdout
