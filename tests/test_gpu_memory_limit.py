"""A batch that does not fit the card is refused, every time it is asked for, and the
operator works on: nothing of the failed workspace is used.  Two small balls far
apart: 384 tets on a large grid."""
import ctypes

import numpy as np
import pytest

from helpers import A_RADIUS, rel

pytestmark = pytest.mark.gpu


def free_bytes():
    """Free device memory, from the HIP runtime that the library uses."""
    hip = ctypes.CDLL('libamdhip64.so.7')  # loaded with the library
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_refused_batch_leaves_the_operator_usable():
    from scadyn_amd import meshgen, native
    c, e = meshgen.sphere(4)
    c = meshgen.rescale_to_radius(c, e, A_RADIUS)
    c, e = np.vstack([c, c + 40.0 * A_RADIUS]), np.vstack([e, e + c.shape[0]])
    op = native.Operator(c, e, np.full(e.shape[0], 2.5 + 0.01j), 2.0 / A_RADIUS, precision=native.PREC_MIXED)
    x = np.random.default_rng(5).standard_normal((2, 2, 3 * e.shape[0]))
    x = x[0] + 1j * x[1]
    y = op.matvec(x)
    inf = op.info()
    grid = 64 * inf['Lx'] * inf['Ly'] * inf['Nz']  # bytes of one vector's grid; a workspace holds two
    op.matvec(x[:1])
    nrhs = int(0.7 * free_bytes() / grid)  # one fits, two do not
    print(f'[memory-limit] {nrhs} vectors, {2 * nrhs * grid / 2**30:.0f} GiB of grids', flush=True)
    wide = np.zeros((nrhs, 3 * e.shape[0]), complex)
    for prec in (native.PREC_FP64, native.PREC_MIXED):
        with pytest.raises(native.ScadynError) as ex:
            op.matvec(wide, precision=prec)
        assert ex.value.code == native.ERR_MEMORY
    assert rel(op.matvec(x), y) < 1e-15
    assert rel(op.matvec(x, precision=native.PREC_MIXED), y) < 1e-5
    op.close()
