"""The near-zone pair and row kernels' own per-lane steps, run on the CPU (host build
with AddressSanitizer): pair list, row order and each entry's block against the
reference's loops, equal element by element; and a lane's share of two cubes with
more than 2^31 pairs."""
import os
import subprocess

from scadyn_amd import build


def test_pairs_and_rows():
    src, exe = build.SELFTESTS['pairs']
    deps = [os.path.join(build.CSRC, f) for f in (src, 'pairs_core.hpp', 'setup.hpp', 'internal.hpp')]
    if not os.path.exists(build.LIB):
        build.build()
    if not os.path.exists(exe) or any(os.path.getmtime(d) > os.path.getmtime(exe) for d in deps):
        build.build_selftest(which='pairs')
    env = dict(os.environ, ASAN_OPTIONS='detect_leaks=0')
    r = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-4000:]
    assert ' 0 failures' in r.stdout
