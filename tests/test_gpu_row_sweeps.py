"""Row sweeps of the block MGS with 6 and 8 vectors a pass, where their workgroups are
limited: fewer row groups than the limit, more, and so many that each sweeps 16."""
import numpy as np
import pytest

from helpers import sphere_case

pytestmark = pytest.mark.gpu


# row groups (3 N rows, 256 // slots to a group) and workgroups: 204 and 204, 269 and
# 256, 2,052 and 256, 4,104 and 257, 13,248 and 828
@pytest.mark.parametrize('cells,slots', [(6, 20), (7, 20), (12, 30), (12, 64), (14, 90)])
@pytest.mark.parametrize('bs', [6, 8])
def test_wide_blocks(cells, slots, bs):
    """Iteration counts within one, solutions within 1e-8 (both converged to 1e-10)."""
    from scadyn_amd import native
    case = sphere_case(n_cells=cells)
    n = 3 * case[1].shape[0]
    print(f'[sweeps] {cells} cells, {n} rows, {slots} slots, {bs} vectors a pass', flush=True)
    rng = np.random.default_rng(5)
    rhs = rng.standard_normal((slots, n)) + 1j * rng.standard_normal((slots, n))
    out = []
    for b in (1, bs):
        op = native.Operator(*case, tol=1e-10, restart=6, mgs_block=b, batch=slots)
        out.append(op.solve(rhs))
        op.close()
    (xa, ia), (xb, ib) = out
    assert np.max(np.abs(ia.astype(int) - ib.astype(int))) <= 1
    assert np.max(np.linalg.norm(xb - xa, axis=1) / np.linalg.norm(xa, axis=1)) < 1e-8
