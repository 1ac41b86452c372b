"""An operator used while a resumable job on it is unfinished: products and another
job take buffers of their own, and neither's results change."""
import numpy as np
import pytest

from helpers import rel, sphere_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
def test_calls_between_the_steps_of_a_job(precision):
    from scadyn_amd import native
    c, e, param, k = sphere_case(n_cells=6)
    prec = native.PREC_MIXED if precision == 'mixed' else native.PREC_FP64
    x = np.random.default_rng(2).standard_normal((2, 3, 3 * e.shape[0]))
    x = x[0] + 1j * x[1]
    ref = native.Operator(c, e, param, k, precision=prec)
    y, T, it = ref.matvec(x), *ref.tmatrix_cols(5, np.arange(70))
    U, iu = ref.tmatrix_cols(3, np.arange(12))
    ref.close()
    op = native.Operator(c, e, param, k, precision=prec)
    print(f'[live-job] {precision}', flush=True)
    a = native.TJob(op, 5, np.arange(70), spread=8)
    a.advance(1)
    assert rel(op.matvec(x), y) < 1e-13
    b = native.TJob(op, 3, np.arange(12))
    left = True
    while left:
        left = a.advance(10) < 70
        b.advance(1)
        assert rel(op.matvec(x), y) < 1e-13
    b.advance(12)
    for job, V, iv in ((a, T, it), (b, U, iu)):
        W, iw = job.result()
        assert np.array_equal(iv, iw)
        assert rel(W, V) < 1e-9
        job.close()
    assert rel(op.matvec(x), y) < 1e-13
    op.close()
