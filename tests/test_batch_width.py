"""Slots of an automatic batch: the footprint query sizes the width that the solve
takes.  The width by its rule, written out: up to 64 columns one batch, above the
equal generations of at most 128 slots with the least sum of slots and half the lanes
of their 64-slot chunks, the fewest where two are equal."""
import numpy as np
import pytest

from helpers import rel, sphere_case


def width(ncols):
    if ncols <= 64:
        return ncols
    best = None
    for gen in range(-(-ncols // 128), -(-ncols // 32) + 1):
        b = -(-ncols // gen)
        cost = gen * (2 * b + 64 * -(-b // 64))
        if best is None or cost < best[0]:
            best = (cost, b)
    return best[1]


def columns(nmax):
    return 2 * ((nmax + 1) ** 2 - 1)


def test_rule():
    assert [width(n) for n in (6, 64, 70, 96, 126, 128, 160)] == [6, 64, 70, 96, 126, 128, 54]
    assert all(1 <= width(n) <= 128 for n in range(1, 881))


@pytest.mark.parametrize('nmax', range(1, 21))
def test_footprint_sizes_the_width_that_runs(nmax):
    from scadyn_amd import native
    c, e, p, k = sphere_case()
    for precision in (native.PREC_FP64, native.PREC_MIXED):
        auto = native.footprint(c, e, p, nmax, precision=precision)
        w = width(columns(nmax))
        assert auto == native.footprint(c, e, p, nmax, precision=precision, batch=w)
        if w > 1:
            assert auto > native.footprint(c, e, p, nmax, precision=precision, batch=w - 1)


@pytest.mark.gpu
@pytest.mark.parametrize('nmax', [4, 5, 6, 7, 8])
def test_solve_takes_that_width(nmax):
    from scadyn_amd import native
    c, e, p, k = sphere_case()
    print(f'[batch-width] {columns(nmax)} columns', flush=True)
    op = native.Operator(c, e, p, k)
    op.tmatrix(nmax)
    assert op.info()['batch'] == width(columns(nmax))
    op.close()


@pytest.mark.gpu
@pytest.mark.parametrize('first,nmax,slots', [(64, 5, 70),   # 64 and 6 would cost 1.4 times one batch of 70
                                              (64, 7, 64),   # two batches of 64 within 2% of one of 126
                                              (100, 5, 100), # holds them all
                                              (64, 4, 64)])
def test_width_does_not_depend_on_the_call_before(first, nmax, slots):
    """A workspace of `first` slots, from a product, then a T-matrix."""
    from scadyn_amd import native
    c, e, p, k = sphere_case()
    print(f'[batch-width] {columns(nmax)} columns after a product of {first}', flush=True)
    op = native.Operator(c, e, p, k)
    op.matvec(np.ones((first, 3 * e.shape[0]), complex))
    assert op.info()['batch'] == first
    T, it = op.tmatrix(nmax)
    assert op.info()['batch'] == slots
    fresh = native.Operator(c, e, p, k)
    Tf, itf = fresh.tmatrix(nmax)
    assert np.array_equal(it, itf)
    for a, b in zip(T, Tf):
        assert rel(a, b) < 1e-9
    op.close()
    fresh.close()
