"""The scatter's rule on width and grid size: two small balls far apart give grids of
30 thousand to 1.2 million nodes with 384 tets, on both sides of each line of the
rule.  A batch against its vectors one at a time: another kernel, another order of
the same sums of about 20 terms; complex128 1e-13, as the other widths."""
import numpy as np
import pytest

from helpers import A_RADIUS, rel

pytestmark = pytest.mark.gpu


def two_balls(gap):
    from scadyn_amd import meshgen
    c, e = meshgen.sphere(4)
    c = meshgen.rescale_to_radius(c, e, A_RADIUS)
    return np.vstack([c, c + gap * A_RADIUS]), np.vstack([e, e + c.shape[0]])


@pytest.mark.parametrize('gap,lo,hi', [(5.0, 0, 1 << 15), (6.0, 1 << 15, 1 << 16), (9.0, 1 << 16, 1 << 17),
                                       (12.0, 1 << 17, 3 << 17), (17.0, 3 << 17, 1 << 19), (24.0, 1 << 19, 1 << 21)])
def test_scatter_widths(gap, lo, hi):
    from scadyn_amd import native
    c, e = two_balls(gap)
    param = np.full(e.shape[0], 2.5 + 0.01j)
    a = native.Operator(c, e, param, 2.0 / A_RADIUS)
    inf = a.info()
    nodes = inf['Nx'] * inf['Ny'] * inf['Nz']
    print(f'[scatter-rule] gap {gap}: {nodes} nodes', flush=True)
    assert lo <= nodes < hi
    b = native.Operator(c, e, param, 2.0 / A_RADIUS)
    x = np.random.default_rng(4).standard_normal((2, 25, 3 * e.shape[0]))
    x = x[0] + 1j * x[1]
    one = np.concatenate([b.matvec(x[r:r + 1]) for r in range(25)])
    for wide in (2, 3, 5, 6, 9, 13, 17, 25):
        y = a.matvec(x[:wide])
        for r in range(wide):
            assert rel(y[r], one[r]) < 1e-13
    a.close()
    b.close()


@pytest.mark.parametrize('n_cells,nx', [(14, 32), (30, 64)])
def test_scatter_widths_on_lines_of_a_multiple_of_32(n_cells, nx):
    """The same on a body whose lines have 32 or 64 nodes."""
    from helpers import sphere_case
    from scadyn_amd import native
    case = sphere_case(n_cells=n_cells)
    a = native.Operator(*case)
    assert a.info()['Nx'] == nx
    print(f'[scatter-rule] {nx} nodes along x', flush=True)
    x = np.random.default_rng(5).standard_normal((2, 25, 3 * case[1].shape[0]))
    x = x[0] + 1j * x[1]
    one = np.concatenate([a.matvec(x[r:r + 1]) for r in range(25)])
    for wide in (2, 3, 4, 5, 7, 8, 11, 12, 15, 16, 23, 24, 25):
        y = a.matvec(x[:wide])
        for r in range(wide):
            assert rel(y[r], one[r]) < 1e-13
    a.close()
