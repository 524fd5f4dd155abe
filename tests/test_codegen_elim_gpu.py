"""Generated real kernels that sum the inner columns out (orders from 26):
value, sum |term| and error estimate against the dense kernels on the same
matrix, and closed forms."""
import numpy as np
import pytest

from conftest import rel_err
from superman_amd import api

pytestmark = pytest.mark.gpu


def pattern(n, per_row, seed):
    rng = np.random.default_rng(seed)
    a = np.zeros((n, n))
    p = rng.permutation(n)
    for i in range(n):
        a[i, p[i]] = rng.standard_normal()
        a[i, rng.choice(np.delete(np.arange(n), p[i]), per_row - 1, replace=False)] = rng.standard_normal(per_row - 1)
    return a


def banded(n, w, seed):
    rng = np.random.default_rng(seed)
    i, j = np.indices((n, n))
    return np.where(np.abs(i - j) <= w, rng.standard_normal((n, n)), 0.0)


def summed_out(a, precision="kahan"):
    return "inner columns summed out" in api.codegen_source_real(a, precision).split("\n")[0]


def check(a, precision="kahan"):
    g = api.sparse_codegen_real(a, precision)
    d = api.dense_f64(a, "kahan")
    # err_est is each result's own estimate; plain sums carry none
    assert abs(g.value - d.value) <= d.err_est + (g.err_est if precision == "kahan" else d.err_est)
    if precision == "kahan":  # positive sums: no cancellation
        assert rel_err(g.abs_sum, d.abs_sum) <= 1e-10


@pytest.mark.parametrize("precision", ["kahan", "dd"])
@pytest.mark.parametrize("n,per_row", [(26, 2), (26, 4), (26, 7), (27, 3), (30, 5), (31, 8)])
def test_matches_the_dense_kernel(n, per_row, precision):
    a = pattern(n, per_row, 100 * n + per_row)
    assert summed_out(a, precision) == ((n, per_row) != (26, 7))  # 6 columns at most: the walk is as cheap
    check(a, precision)


@pytest.mark.parametrize("n,w", [(26, 1), (28, 2), (29, 3)])
def test_banded(n, w):
    a = banded(n, w, n)
    assert summed_out(a) == (w <= 2)  # 7 columns tied by a row: tables past the limit
    check(a)


def test_patterns_that_keep_the_walk():
    full = np.random.default_rng(1).standard_normal((26, 26))  # every row in every column: nothing to factor
    assert not summed_out(full) and not summed_out(pattern(25, 3, 1))
    check(full)
    z = pattern(26, 4, 5)
    z[:, 3] = 0.0  # an empty column comes first in the order
    assert not summed_out(z)
    r = api.sparse_codegen_real(z)  # perm = 0
    assert abs(r.value) <= r.err_est


def test_some_rows_full():
    a = pattern(28, 3, 9)
    a[4, :] = np.random.default_rng(2).standard_normal(28)
    a[:, 11] += 0.5
    check(a)


@pytest.mark.parametrize("n", [36, 40])
def test_triangular_closed_form(n):
    rng = np.random.default_rng(n)
    a = np.diag(rng.uniform(0.5, 2.0, n))
    for i in range(n - 1):
        a[i, rng.choice(np.arange(i + 1, n), size=min(2, n - 1 - i), replace=False)] = rng.uniform(-1, 1)
    r = api.sparse_codegen_real(a)
    assert abs(r.value - np.prod(np.diag(a))) <= r.err_est
