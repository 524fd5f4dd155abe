"""Dense matrices whose rows are integers of different scales: the walk's row
sums are exact row by row, so the products and the permanent come out exact
where they fit 53 bits.  Scaling the rows to a column of ones would round them."""
import math

import numpy as np
import pytest

from oracle import oracle as O
from superman_amd import api

pytestmark = pytest.mark.gpu


def scaled_rows(n, seed, step):
    rng = np.random.default_rng([n, seed])
    a = rng.integers(3, 8, (n, n)).astype(np.int64)
    a[:, -1] += 1 - a.sum(1) % 2  # odd row sums: no term is 0
    e = np.arange(n) * step - n * step // 2
    return a, e


@pytest.mark.parametrize("precision", ["kahan", "dd"])
@pytest.mark.parametrize("n,step", [(6, 1), (6, 60), (7, 25), (8, 9), (8, -14)])
def test_real(n, step, precision):
    a, e = scaled_rows(n, 1, step)
    ref, st = O.int_exact(a)
    # every term 2^n prod |x_i| <= prod sum_j a_ij, and 2^n of them
    assert st == 0 and math.prod(int(v) for v in a.sum(1)) << n < 1 << 53
    m = a * np.exp2(e)[:, None]
    assert api.dense_f64(m, precision).value == ref * 2.0 ** int(e.sum())
    assert api.dense_f64_noalloc(m, precision).value == ref * 2.0 ** int(e.sum())


@pytest.mark.parametrize("precision", ["kahan", "dd"])
@pytest.mark.parametrize("n,step", [(6, 60), (8, 9)])
def test_complex(n, step, precision):
    a, e = scaled_rows(n, 2, step)
    ref, st = O.int_exact(a)
    assert st == 0 and math.prod(int(v) for v in a.sum(1)) << n < 1 << 53
    turn = np.array([1, 1j, -1, -1j])
    z = a * np.exp2(e)[:, None] * turn[np.arange(n) % 4][:, None]  # perm = i^(0 + ... + n-1) perm(a)
    assert api.dense_c128(z, precision).value == ref * 2.0 ** int(e.sum()) * turn[n * (n - 1) // 2 % 4]


def test_one_exact_row_decides():
    # an integer row among others needs a power of two in the column that is
    # scaled to ones; row n-2 of a complex matrix is multiplied by the others'
    # entries of that column instead, and its last row is left as it is
    n = 12
    for i in (5, n - 2, n - 1):
        for row in (np.full(n, 3.0), np.full(n, 4.0), np.r_[4.0, np.full(n - 1, 3.0)]):
            m = np.random.default_rng(5).standard_normal((n, n))
            m[:, 0] = 1.5 + m[:, 0] % 0.25
            m[i] = row
            two = row[0] == 4.0
            for a, pair in ((m, two), (m * (1 + 0j), two if i == 5 else i == n - 1)):
                with api.DensePlan(a) as p:
                    assert ("_pair_kernel" in p.info()["kernel"]) == pair, (i, row[0], a.dtype)
