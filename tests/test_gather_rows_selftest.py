"""The row-group gather kernels' own per-lane steps, run on the CPU (host build with
AddressSanitizer) against a direct evaluation: every wave layout the launcher picks,
row groups of 1 to 6 rows, partial chunks of slots, inactive slots.

Tolerances (relative Frobenius): 1e-13 complex128, 1e-5 complex64, as the older
gather self-test."""
import os
import subprocess

from scadyn_amd import build


def test_row_group_gather():
    src, exe = build.SELFTESTS['gather_rows']
    deps = [os.path.join(build.CSRC, f) for f in (src, 'gather_core.hpp', 'internal.hpp')]
    if not os.path.exists(build.LIB):
        build.build()
    if not os.path.exists(exe) or any(os.path.getmtime(d) > os.path.getmtime(exe) for d in deps):
        build.build_selftest(which='gather_rows')
    env = dict(os.environ, ASAN_OPTIONS='detect_leaks=0')
    r = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-4000:]
    assert r.stdout.splitlines()[-1] == '0 failures'
