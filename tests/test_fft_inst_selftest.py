"""The compiled instances of the register line FFT (fixed tile width, 32-bit lane
offsets), run on the CPU (host build with AddressSanitizer) as the launcher picks
them: bit for bit against the 64-bit instance, and the fused convolution with
octants of FFT(G) around and beyond 2 and 4 GiB against a direct long-double DFT;
and the planner's tile widths.

Tolerances (relative Frobenius): 1e-14 complex128, 2e-6 complex64, as for the
stages themselves."""
import os
import subprocess

from scadyn_amd import build


def test_line_fft_instances():
    src, exe = build.SELFTESTS['fft_inst']
    deps = [os.path.join(build.CSRC, f) for f in (src, 'fft_reg_core.hpp', 'fft.hpp', 'internal.hpp')]
    if not os.path.exists(build.LIB):
        build.build()
    # the planner comes from the library at run time
    if not os.path.exists(exe) or any(os.path.getmtime(d) > os.path.getmtime(exe) for d in deps):
        build.build_selftest(which='fft_inst')
    env = dict(os.environ, ASAN_OPTIONS='detect_leaks=0')
    r = subprocess.run([exe], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-4000:]
    assert ' 0 failures' in r.stdout
