"""The gather's rule on width and mesh: batches of 1 to 9 vectors on meshes of 6.7
thousand to 0.2 million tets, on both sides of each line of the rule, against other
kernels of the same sums: complex128 against the vectors in a batch of 33, 1e-13;
complex64 against complex64 in that batch, 2e-6, as the other widths."""
import numpy as np
import pytest

from helpers import rel, sphere_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n_cells,lo,hi', [(12, 4096, 8192), (14, 8192, 1 << 16), (30, 1 << 16, 3 << 16),
                                           (40, 3 << 16, 1 << 18)])
def test_gather_widths(n_cells, lo, hi):
    from scadyn_amd import native
    c, e, param, k = sphere_case(n_cells=n_cells)
    assert lo <= e.shape[0] < hi
    print(f'[gather-rule] {e.shape[0]} tets', flush=True)
    a = native.Operator(c, e, param, k, precision=native.PREC_MIXED)
    x = np.random.default_rng(6).standard_normal((2, 33, 3 * e.shape[0]))
    x = x[0] + 1j * x[1]
    for prec, tol in ((native.PREC_FP64, 1e-13), (native.PREC_MIXED, 2e-6)):
        ref = a.matvec(x, precision=prec)
        for wide in (1, 2, 3, 4, 5, 6, 7, 8, 9):
            y = a.matvec(x[:wide], precision=prec)
            for r in range(wide):
                assert rel(y[r], ref[r]) < tol
    a.close()


@pytest.mark.parametrize('wide', [8, 31, 70])
def test_matrix_core_gather_needs_half_a_chunk(wide):
    """gather_kernel = 1 on widths whose last 64-slot chunk is less than half full: the
    vector kernel, hence its bits."""
    from scadyn_amd import native
    c, e, param, k = sphere_case(n_cells=8)
    print(f'[gather-rule] matrix cores, {wide} vectors', flush=True)
    a = native.Operator(c, e, param, k, precision=native.PREC_MIXED)
    b = native.Operator(c, e, param, k, precision=native.PREC_MIXED, gather_kernel=1)
    x = np.random.default_rng(8).standard_normal((2, wide, 3 * e.shape[0]))
    x = x[0] + 1j * x[1]
    assert np.array_equal(a.matvec(x, precision=native.PREC_MIXED), b.matvec(x, precision=native.PREC_MIXED))
    a.close()
    b.close()


# rows to a gather group: 2.0, 3.3 and 3.9 to 4.3 (a flattened body), and 2 on a small mesh
@pytest.mark.parametrize('n_cells,stretch,grid_size', [(18, (1, 1, 1), 1.2), (18, (1, 1, 1), 1.5),
                                                       (18, (2, 2, 0.25), 1.8), (18, (0.4, 0.4, 2.5), 1.8),
                                                       (10, (1, 1, 1), 1.2)])
def test_gather_widths_with_few_rows_to_a_group(n_cells, stretch, grid_size):
    """Complex128 widths of 1 to 32 against the vectors in a batch of 33, 1e-13 of the
    largest element times what the near zone cancels; complex64 widths, whose sums have
    one order from 5 vectors on, likewise in single precision."""
    from scadyn_amd import native
    c, e, param, k = sphere_case(n_cells=n_cells)
    c = c * np.array(stretch)
    print(f'[gather-rule] {e.shape[0]} tets, {stretch}, grid {grid_size}', flush=True)
    a = native.Operator(c, e, param, k, precision=native.PREC_MIXED, grid_size=grid_size)
    x = np.random.default_rng(7).standard_normal((2, 33, 3 * e.shape[0]))
    x = x[0] + 1j * x[1]
    ref = a.matvec(x, precision=native.PREC_FP64)
    single = a.matvec(x, precision=native.PREC_MIXED)
    lost = max(rel(single[r], ref[r]) for r in range(33))  # what single precision loses here
    double = max(1e-13, lost * 2.0 ** -29 * 16)  # 29 bits more, and a wide margin
    for wide in (1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 17, 20, 24, 25, 31, 32):
        y = a.matvec(x[:wide], precision=native.PREC_FP64)
        z = a.matvec(x[:wide], precision=native.PREC_MIXED)
        for r in range(wide):
            assert rel(y[r], ref[r]) < double
            assert rel(z[r], ref[r]) < 16 * lost
    a.close()
