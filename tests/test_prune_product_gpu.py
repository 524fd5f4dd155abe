"""The pruned walk's row products at the ends of their ranges: sums that just
fit signed bytes and that just do not, 16 rows within 64 bits and beyond, and
lanes whose 64 settings all survive; exact against the int128 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from superman_amd import api

pytestmark = pytest.mark.gpu


def check(a):
    with api.DensePlan(a, "exact", int_walk="pruned") as p:
        got = [p.run().exact for _ in range(2)]
    ref, st = O.int_exact(a)
    assert st == 0 and got == [ref, ref]


def pattern(n, per_row):
    rng = np.random.default_rng([n, per_row])
    a = np.zeros((n, n), dtype=np.int64)
    for i in range(n):
        a[i, rng.choice(n, per_row, replace=False)] = 1
        a[i, i] = 1
    return a


def wide_row(n, total, last):
    r = np.zeros(n, dtype=np.int64)
    r[: n - 1] = total // (n - 1)
    r[0] += total - r.sum()
    r[n - 1] = last
    return r


# y from -128 to 127, from -127 to 128; past a byte altogether (190 to 210);
# the same below zero
@pytest.mark.parametrize("total,last", [(255, -1), (255, 1), (10, 200), (10, -201)])
@pytest.mark.parametrize("n,per_row", [(13, 4), (18, 3), (20, 5)])
def test_byte_range(n, per_row, total, last):
    a = pattern(n, per_row)
    a[n // 2] = wide_row(n, total, last)
    check(a)


# 16 rows of up to 2^3, 2^4 and 2^5: within and beyond 64 bits
@pytest.mark.parametrize("n", [13, 17, 20])
@pytest.mark.parametrize("top", [1, 2, 4])
def test_product_width(n, top):
    rng = np.random.default_rng([n, top])
    a = rng.integers(0, top + 1, (n, n))
    check(a)


@pytest.mark.parametrize("n", [13, 15, 19])
def test_every_subset_survives(n):
    a = np.ones((n, n), dtype=np.int64)
    a[:, -1] = 3  # odd row sums
    assert (a.sum(1) % 2 == 1).all()
    check(a)
