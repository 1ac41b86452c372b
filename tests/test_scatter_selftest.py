"""The narrow scatter's own per-lane steps, run on the CPU (host build with
AddressSanitizer) against the sum written out, with workgroups that stride over the
nodes; and launch sizes of grids beyond 2^26 nodes, whose work-items a launch
cannot hold at once.

Tolerances (relative Frobenius over the grid): 1e-14 complex128, 2e-6 complex64
(sums of up to 100 products)."""
import os
import subprocess

from scadyn_amd import build


def test_narrow_scatter():
    src, exe = build.SELFTESTS['scatter']
    deps = [os.path.join(build.CSRC, f) for f in (src, 'scatter_core.hpp', 'internal.hpp')]
    if not os.path.exists(build.LIB):
        build.build()
    if not os.path.exists(exe) or any(os.path.getmtime(d) > os.path.getmtime(exe) for d in deps):
        build.build_selftest(which='scatter')
    env = dict(os.environ, ASAN_OPTIONS='detect_leaks=0')
    r = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-4000:]
    assert ' 0 failures' in r.stdout
