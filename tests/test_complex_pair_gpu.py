"""Dense complex permanents two subsets per step (dense_c128_pair_kernel)
against the double-double oracle and the one-subset kernel."""
import numpy as np
import pytest

from conftest import rel_err
from oracle import oracle as O
from superman_amd import api

pytestmark = pytest.mark.gpu

TOL = 1e-10  # the bar of the dense kernels against the oracle


def gauss(n, seed):
    rng = np.random.default_rng([n, seed])
    return (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(2)


def dd(z):
    q = O.complex_dd(z)
    return complex(q[0] + q[1], q[2] + q[3])


def run(z, precision="kahan", chunk=None):
    with api.DensePlan(z, precision) as p:
        if chunk is not None:
            p.set_log2_chunk(chunk)
        return p.run(), p.info()["kernel"]


@pytest.mark.parametrize("precision", ["kahan", "dd"])
@pytest.mark.parametrize("n", [5, 6, 7, 9, 14, 17])
def test_edges_of_the_orders(n, precision):
    # 17 | 16 rows: one and two column parts; every chunk length down to the
    # one that the one-subset kernel walks (2)
    z = gauss(n, 1)
    ref = dd(z)
    sums = {}
    for chunk in [None] + list(range(2, n)):
        r, k = run(z, precision, chunk)
        pair = n >= 6 and chunk != 2
        assert k.startswith("dense_c128_pair_kernel" if pair else "dense_c128_kernel")
        assert rel_err(r.value, ref) <= TOL
        sums[pair] = r.abs_sum
    if precision == "kahan" and len(sums) == 2:
        # the moduli are bounded in the same L1 norms: equal but for roundings
        assert rel_err(sums[True], sums[False]) <= 1e-12


def test_matrices_that_keep_one_subset_per_step():
    rng = np.random.default_rng(2)
    z = gauss(11, 2)
    z[rng.permutation(9), np.arange(9)] = 0.0  # a zero in rows 0..8 of columns 0..8
    z[[0, 1], [9, 10]] = 0.0
    ints = (rng.integers(2, 9, (11, 11)) + 1j * rng.integers(2, 9, (11, 11))).astype(complex)
    for a in (z, ints):
        r, k = run(a)
        assert k.startswith("dense_c128_kernel") and rel_err(r.value, dd(a)) <= TOL


def test_zeros_in_the_last_two_rows_and_unit_columns():
    z = gauss(12, 3)
    z[10:, :] *= np.random.default_rng(3).random((2, 12)) < 0.5  # any entry of these rows may be 0
    r, k = run(z)
    assert k.startswith("dense_c128_pair_kernel") and rel_err(r.value, dd(z)) <= TOL
    rng = np.random.default_rng(4)
    g = (rng.integers(-3, 4, (9, 9)) + 1j * rng.integers(-3, 4, (9, 9))).astype(complex)
    g[:, 5] = rng.choice([1, -1, 1j, -2j], 9)  # exact quotients: only products round
    r, k = run(g)
    assert k.startswith("dense_c128_pair_kernel") and rel_err(r.value, dd(g)) <= 1e-14


def test_conjugate_and_scaled_rows():
    z = gauss(13, 5)
    r, _ = run(z)
    c, _ = run(np.conj(z))
    assert rel_err(c.value, r.value.conjugate()) <= TOL
    s, k = run(z * np.ldexp(1.0, np.arange(-130, 130, 20))[:, None])
    assert k.startswith("dense_c128_pair_kernel")
    assert rel_err(s.value, r.value * 2.0 ** float(np.arange(-130, 130, 20).sum())) <= TOL
