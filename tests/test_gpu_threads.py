"""Operators made in two threads at once: each has the projections, near-zone blocks
and products of one made alone, bit for bit."""
import threading

import numpy as np
import pytest

from helpers import sphere_case

pytestmark = pytest.mark.gpu


def test_operators_made_at_once():
    from scadyn_amd import native
    todo = [sphere_case(n_cells=n, ka=ka) for n, ka in ((10, 2.0), (13, 1.5), (9, 2.5), (12, 1.0))]
    x = [np.random.default_rng(i).standard_normal((2, 3 * c[1].shape[0])) + 0j for i, c in enumerate(todo)]

    def make(i):
        op = native.Operator(*todo[i])
        out = op.export('S'), op.export('blocks'), op.matvec(x[i])
        op.close()
        return out
    alone = [make(i) for i in range(len(todo))]
    bad = []

    def run(order):
        for i in order:
            for what, a, b in zip(('S', 'blocks', 'product'), make(i), alone[i]):
                if not np.array_equal(a, b):
                    bad.append((i, what))
    print('[threads] two threads', flush=True)
    th = [threading.Thread(target=run, args=(o * 8,)) for o in ([0, 1, 2, 3], [3, 1, 0, 2])]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
