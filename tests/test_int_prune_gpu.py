"""Exact walk over the subsets with no zero row (SPM_INT_WALK_PRUNED):
bit-exact against the int128 oracle at the edges of its layout, and against
closed forms where the oracle is too slow."""
import math

import numpy as np
import pytest

from oracle import oracle as O
from superman_amd import _lib, api

pytestmark = pytest.mark.gpu


def pruned(a):
    with api.DensePlan(np.asarray(a, dtype=np.int64), "exact", int_walk="pruned") as p:
        info, r = p.info(), p.run()
        assert p.run().exact == r.exact  # lists and counters are back to 0
    return r.exact, info["kernel"]


def pattern(n, per_row, seed, values=(1,)):
    rng = np.random.default_rng(seed)
    a = np.zeros((n, n), dtype=np.int64)
    p = rng.permutation(n)
    for i in range(n):
        a[i, p[i]] = 1
        a[i, rng.choice(np.delete(np.arange(n), p[i]), per_row - 1, replace=False)] = 1
    return a * rng.choice(values, (n, n))


# 13: one node; 14, 18: prefixes but no list; 19: the first order with a list
# (first_group 3); 16 | 17: 4 and 8 dwords of 8-bit fields; 25 and 26: a
# group of 6 columns filled and one begun
@pytest.mark.parametrize("n", [13, 14, 16, 17, 18, 19, 24, 25])
@pytest.mark.parametrize("kind", ["half01", "even4", "odd3", "signed"])
def test_vs_oracle(n, kind):
    rng = np.random.default_rng(100 * n + len(kind))
    a = {"half01": lambda: (rng.random((n, n)) < 0.5).astype(np.int64),
         "even4": lambda: pattern(n, 4, n),                    # every row can be zero
         "odd3": lambda: pattern(n, 3, n),                     # no row ever is
         "signed": lambda: pattern(n, 4, n, (-3, -2, -1, 1, 2, 3))}[kind]()
    ref, st = O.int_exact(a)
    assert st == 0
    v, k = pruned(a)
    assert v == ref and k.startswith("int_prune_kernel<1")


@pytest.mark.parametrize("n,values", [(13, (150, -100, 77)), (14, (-90, 40, 127)), (17, (-9, 40, 7, 25))])
def test_wide_fields(n, values):
    # rows past 8 bits: 16-bit fields, row products in 64 bits; some rows'
    # zero masks do not fit and their zeros come out of the product
    a = pattern(n, 3, n, values)
    ref, st = O.int_exact(a)
    assert st == 0
    v, k = pruned(a)
    assert v == ref
    assert k.startswith("int_prune_kernel<%d" % (1 if 2 * np.abs(a).sum(1).max() <= 255 else 2))


def test_zero_lines():
    a = pattern(20, 4, 1)
    a[3, :] = 0
    assert pruned(a)[0] == 0
    b = pattern(20, 4, 2)
    b[:, 7] = 0
    assert pruned(b)[0] == 0


@pytest.mark.parametrize("n", [33, 36, 37, 42, 43, 49, 63])
def test_identity_plus_cycle(n):
    # launches for up to 7 column groups; 12 and 16 dwords of 8-bit fields
    a = np.eye(n, dtype=np.int64) + np.roll(np.eye(n, dtype=np.int64), 1, axis=1)
    assert pruned(a)[0] == 2


def test_wide_fields_many_dwords():
    # I + 300 P, P the n-cycle: 1 + 300^n outgrows 128 bits, so the cycle
    # entry is 300 in one row only
    for n in (17, 33):
        a = np.eye(n, dtype=np.int64) + np.roll(np.eye(n, dtype=np.int64), 1, axis=1)
        a[2, 3] = 300
        v, k = pruned(a)
        assert v == 301 and k.startswith("int_prune_kernel<2, %d>" % (16 if n == 17 else 24))


def test_like_rows_overfill_the_lists():
    # four blocks of ones J_8, order 32: rows of a block are zero together, so
    # far more prefixes survive than the row-independence estimate that sizes
    # the lists; what does not fit is walked where it is found
    n = 32
    a = np.zeros((n, n), dtype=np.int64)
    for b in range(4):
        a[8 * b:8 * b + 8, 8 * b:8 * b + 8] = 1
    rng = np.random.default_rng(8)
    a = a[rng.permutation(n)][:, rng.permutation(n)]
    assert pruned(a)[0] == math.factorial(8) ** 4


def test_refused():
    for a in (np.ones((12, 12), dtype=np.int64), np.diag([1 << 17] * 2 + [1] * 12)):
        with pytest.raises(_lib.SpmError) as e:
            pruned(a)
        assert e.value.status == _lib.SPM_ERANGE


def test_automatic_choice():
    for a, pre in ((pattern(36, 4, 1), "int_prune"), (pattern(36, 3, 1), "int_small"), (pattern(16, 4, 1), "int_small"),
                   ((np.random.default_rng(3).random((30, 30)) < 0.5).astype(np.int64), "int_prune")):
        with api.DensePlan(a, "exact") as p:
            assert p.info()["kernel"].startswith(pre)
