"""How a batch splits a request into lane chunks and wave items: every order
at which the split changes, and item budgets that only the widest chunks fit."""
import numpy as np
import pytest

from oracle import oracle as O
from superman_amd import _lib
from superman_amd.batch import BatchEngine, to_permanent

from conftest import rel_err

TOL = 1e-10  # the bar of the dense kernels against the oracle


def make(kind, n, seed=0):
    rng = np.random.default_rng([n, seed])
    if kind == "int":
        return (rng.random((n, n)) < 0.5).astype(float)
    a = rng.standard_normal((n, n))
    return a + 1j * rng.standard_normal((n, n)) if kind == "complex" else a


@pytest.mark.parametrize("kind,wide", [("real", 10), ("complex", 9), ("int", 10)])
@pytest.mark.parametrize("n", [1, 2, 3, 8, 13, 16, 17, 22, 28])
def test_item_budget_of_the_widest_chunks(kind, wide, n):
    # one item fewer than the widest chunks take is refused, that many are not
    B = n - 1
    L = 0 if n == 1 else 1 if n == 2 else max(2, min(wide, B - 6))
    items = max(1, 2 ** (B - L) // 64)
    with BatchEngine(dry_run=True, max_items=items) as eng:
        assert eng.try_submit(kind, make(kind, n))[0] == 0
    if items > 1:
        with BatchEngine(dry_run=True, max_items=items - 1) as eng:
            assert eng.try_submit(kind, make(kind, n))[0] == _lib.SPM_ENOMEM


@pytest.mark.gpu
@pytest.mark.parametrize("max_items", [None, 2])
@pytest.mark.parametrize("kind", ["real", "complex", "int"])
def test_orders_where_the_split_changes(kind, max_items):
    # 11 | 12 | 13: one wave, two waves, four; 16 | 17: chunks grow from 2^5;
    # 18 .. 21: up to each kind's longest; two items: the widest chunks
    orders = [3, 7, 8, 11, 12, 13, 16, 17] + ([] if max_items else [18, 19, 20, 21])
    reqs = [(kind, make(kind, n, 1), n) for n in orders]
    with BatchEngine(**({"max_items": max_items} if max_items else {})) as eng:
        st, res = eng.run_raw(reqs)
        assert st == 0
        for (_, a, n), r in zip(reqs, res):
            p = to_permanent(r, kind)
            if kind == "int":
                assert p.exact == O.int_exact(a.astype(np.int64))[0], n
                continue
            q = O.complex_dd(a) if kind == "complex" else O.dense_dd(a)
            ref = complex(q[0] + q[1], q[2] + q[3]) if kind == "complex" else q[0] + q[1]
            assert rel_err(p.value, ref) <= TOL, n
        assert eng.counters() == {"late_publish": 0, "retried": 0}
