"""The pruned walk's tables (prune_tables_kernel) where their sizes end: one
zero mask per row up to all that fit, 8- and 16-bit fields, a last column
group of one column and of six; exact against the int128 oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from superman_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [13, 18, 19, 20])  # 12 = 2 groups, 17, 18 = 3 groups, 19 columns
@pytest.mark.parametrize("scale,kernel", [(1, 1), (12, 1), (90, 2)])
def test_dense_rows(n, scale, kernel):
    # three rows 12 or 90 times as wide (8 and 16 bits): more masks than fit,
    # those of the last tested rows are dropped
    rng = np.random.default_rng(1000 * n + scale)
    a = (rng.random((n, n)) < (0.9 if scale == 1 else 0.5)).astype(np.int64)
    a[:, 0] = 1  # a tested row in every even row sum
    a[:3] *= scale
    with api.DensePlan(a, "exact", int_walk="pruned") as p:
        assert p.info()["kernel"].startswith("int_prune_kernel<%d" % kernel)
        got = [p.run().exact for _ in range(2)]
    a[:3] //= scale
    base, st = O.int_exact(a)
    ref = scale**3 * base
    assert st == 0 and got == [ref, ref]


def test_no_masks():
    # odd row sums throughout: no row is ever zero, no masks at all
    a = np.eye(14, dtype=np.int64) + np.roll(np.eye(14, dtype=np.int64), 1, 1) + np.roll(np.eye(14, dtype=np.int64), 5, 1)
    with api.DensePlan(a, "exact", int_walk="pruned") as p:
        assert p.run().exact == O.int_exact(a)[0]
