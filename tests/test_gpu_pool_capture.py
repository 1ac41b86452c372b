"""A stream capture of the caller's that is under way while kept device memory is
given back (another thread, up to a second after the call that freed it) stays whole."""
import ctypes
import time

import numpy as np
import pytest

from helpers import A_RADIUS

pytestmark = pytest.mark.gpu


def test_capture_while_memory_is_given_back():
    from scadyn_amd import meshgen, native
    c, e = meshgen.sphere(16)
    c = meshgen.rescale_to_radius(c, e, A_RADIUS)
    native.tmat_solve(c, e, np.full(e.shape[0], 2.5 + 0.01j), 2.0 / A_RADIUS, 3)
    hip = ctypes.CDLL('libamdhip64.so.7')  # loaded with the library
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    held = free.value
    stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    print('[capture] begins', flush=True)
    assert hip.hipStreamBeginCapture(stream, 0) == 0  # 0: forbids such calls in other threads
    time.sleep(2.5)  # kept for one second
    status = ctypes.c_int(-1)
    assert hip.hipStreamIsCapturing(stream, ctypes.byref(status)) == 0
    ended = hip.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert status.value == 1 and ended == 0  # 1: active, not invalidated
    assert hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamDestroy(stream) == 0
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    assert free.value > held + (1 << 28)  # given back all the same
