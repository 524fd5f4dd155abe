"""Dense real permanents two subsets per step (dense_pair_kernel): the
matrix scaled so that one column is all ones, against the double-double
oracle and against the one-subset kernel on matrices that keep it."""
import numpy as np
import pytest

from conftest import rel_err
from oracle import oracle as O
from superman_amd import api

pytestmark = pytest.mark.gpu

TOL = 1e-10  # the bar of the dense kernels against the oracle


def run(a, precision="kahan", chunk=None):
    with api.DensePlan(a, precision) as p:
        if chunk is not None:
            p.set_log2_chunk(chunk)
        return p.run(), p.info()["kernel"]


def dd(a):
    hi, lo = O.dense_dd(a)
    return hi + lo


@pytest.mark.parametrize("precision", ["kahan", "dd"])
@pytest.mark.parametrize("n", [5, 6, 7, 8, 11, 16, 21])
def test_edges_of_the_orders(n, precision):
    # 5: below the pair kernel; every chunk length down to the one that the
    # one-subset kernel walks (2)
    a = np.random.default_rng(n).standard_normal((n, n))
    ref = dd(a)
    for chunk in [None] + list(range(2, n)):
        r, k = run(a, precision, chunk)
        assert k.startswith("dense_pair_kernel" if n >= 6 and chunk != 2 else "dense_f64_kernel"), (chunk, k)
        assert rel_err(r.value, ref) <= TOL, (chunk, r.value, ref)


def test_matrices_that_keep_one_subset_per_step():
    rng = np.random.default_rng(1)
    z = rng.standard_normal((12, 12))
    z[rng.permutation(12), np.arange(12)] = 0.0       # a zero in every column
    ints = rng.integers(2, 10, (12, 12)).astype(float)  # exact row sums that quotients would lose
    tiny = rng.standard_normal((12, 12))
    tiny[rng.permutation(12), np.arange(12)] *= 1e-30   # every column's quotients spread too far
    for a in (z, ints, tiny):
        r, k = run(a)
        assert k.startswith("dense_f64_kernel")
        assert rel_err(r.value, dd(a)) <= TOL


def test_exact_columns_of_powers_of_two():
    rng = np.random.default_rng(2)
    a = rng.integers(2, 10, (9, 9)).astype(float)
    a[:, 4] = 2.0 ** rng.integers(-3, 4, 9) * rng.choice([-1, 1], 9)
    r, k = run(a)
    # every quotient and sum is exact: the only roundings are the products'
    assert k.startswith("dense_pair_kernel") and rel_err(r.value, dd(a)) <= 1e-14
    b = np.ones((10, 10))
    r, k = run(b)
    assert k.startswith("dense_pair_kernel") and r.value == 3628800.0


def test_row_scales_far_apart():
    # rows 2^+-400: the quotients do not see them, the result does
    a = np.random.default_rng(3).standard_normal((14, 14))
    e = np.array([400, -400] * 7) + np.arange(14)
    r, _ = run(a)
    s, k = run(np.ldexp(a, e[:, None]))
    assert k.startswith("dense_pair_kernel")
    assert (s.hi, s.lo, s.abs_sum) == tuple(np.ldexp(v, int(e.sum())) for v in (r.hi, r.lo, r.abs_sum))


@pytest.mark.parametrize("n", [10, 17, 20])
def test_same_sums_as_one_subset_per_step(n):
    # a zero put into every column but one keeps the pair kernel; a zero in
    # that one too takes the other kernel on nearly the same matrix
    rng = np.random.default_rng(40 + n)
    a = rng.random((n, n))
    a[rng.permutation(n)[:n - 1], np.arange(1, n)] = 0.0
    r, k = run(a)
    assert k.startswith("dense_pair_kernel")
    b = a.copy()
    b[5, 0] = 0.0
    c = a.copy()
    c[5, 1:] = 0.0  # perm(a) = perm(b) + perm(c) by row 5; c has one entry there
    q, kq = run(b)
    assert kq.startswith("dense_f64_kernel")
    t, _ = run(np.delete(np.delete(c, 5, 0), 0, 1))
    assert abs(r.value - (q.value + a[5, 0] * t.value)) <= r.err_est + q.err_est + abs(a[5, 0]) * t.err_est
    assert r.abs_sum >= abs(r.value)
