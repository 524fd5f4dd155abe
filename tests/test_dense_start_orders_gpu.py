"""The one-subset dense walk on both sides of the order where its chunk starts
change (36 | 37): I + 2 P, P the n-cycle, has permanent 1 + 2^n, and every
column has a zero, so no column can be scaled to ones."""
import numpy as np
import pytest

from superman_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [36, 37])
def test_two_permutations(n):
    a = np.eye(n) + 2.0 * np.roll(np.eye(n), 1, axis=1)
    with api.DensePlan(a, "kahan") as p:
        assert p.info()["kernel"].startswith("dense_f64_kernel")
        r = p.run()
    with api.DensePlan(a, "dd") as p:
        plain = p.run()
    assert abs(r.value - (1 + 2.0**n)) <= r.err_est
    # plain sums: at most 2^20 terms (a lane's) added in FP64, each addition half
    # an ulp of a partial sum of at most sum |term|
    assert abs(plain.value - (1 + 2.0**n)) <= r.err_est + 2.0**20 * 2.0**-53 * r.abs_sum
