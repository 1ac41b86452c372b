"""Bars that follow one another use the memory of those before: same results as the
first one, from one thread and from two, and the memory is given back."""
import ctypes
import threading
import time

import numpy as np
import pytest

from helpers import A_RADIUS

pytestmark = pytest.mark.gpu


def free_bytes():
    """Free device memory, from the HIP runtime that the library uses."""
    hip = ctypes.CDLL('libamdhip64.so.7')  # loaded with the library
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def bars():
    """Bars of different sizes and precisions, all with blocks large enough to be kept."""
    from scadyn_amd import meshgen, native
    out = []
    for cells, nmax, prec in ((16, 3, native.PREC_FP64), (18, 2, native.PREC_MIXED), (15, 4, native.PREC_FP64)):
        c, e = meshgen.sphere(cells)
        c = meshgen.rescale_to_radius(c, e, A_RADIUS)
        out.append(((c, e, np.full(e.shape[0], 2.5 + 0.01j), 2.0 / A_RADIUS, nmax), dict(precision=prec)))
    return out


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a[0], b[0])) and np.array_equal(a[1], b[1])


def test_same_results_and_memory_given_back():
    from scadyn_amd import native
    todo = bars()
    print('[bars] one after another', flush=True)
    first = [native.tmat_solve(*a, **o) for a, o in todo]
    for _ in range(2):
        for i in (2, 0, 1, 1, 0):
            a, o = todo[i]
            assert same(native.tmat_solve(*a, **o), first[i])
    print('[bars] two threads', flush=True)
    bad = []

    def run(order):
        for i in order:
            a, o = todo[i]
            if not same(native.tmat_solve(*a, **o), first[i]):
                bad.append(i)
    th = [threading.Thread(target=run, args=(o,)) for o in ((0, 1, 2, 0), (2, 2, 1, 0))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    time.sleep(2.5)  # kept for one second
    free = free_bytes()  # the runtime has all it holds by now
    a, o = todo[0]
    native.tmat_solve(*a, **o)
    assert free_bytes() < free - (1 << 28)
    time.sleep(2.5)
    assert free_bytes() > free - (1 << 26)
    op = native.Operator(*a[:4], **o)
    T = op.tmatrix(a[4])
    op.close()
    assert same(T, first[0])
    assert free_bytes() < free - (1 << 28)
    time.sleep(2.5)
    assert free_bytes() > free - (1 << 26)


def test_the_request_loop_keeps_nothing():
    from scadyn_amd import native
    a, o = bars()[0]
    sv = native.Server()
    sv.wait(sv.submit(*a, **o))
    time.sleep(2.5)
    free = free_bytes()
    sv.wait(sv.submit(*a, **o))
    time.sleep(0.2)  # the worker retires the request
    assert free_bytes() > free - (1 << 26)
    sv.close()
