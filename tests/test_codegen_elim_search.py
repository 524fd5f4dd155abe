"""The search for the inner columns a generated real kernel sums out (host
only): a pattern whose rows are too full for it is given up before its tables
are spelled out, and sparse ones keep their choice."""
import time

import numpy as np
import pytest

from superman_amd import api


def head(a, precision="kahan"):
    return api.codegen_source_real(a, precision).split("\n")[0]


def pattern(n, per_row):
    rng = np.random.default_rng([n, per_row])
    a = np.zeros((n, n))
    p = rng.permutation(n)
    for i in range(n):
        a[i, p[i]] = 1.0
        a[i, rng.choice(np.delete(np.arange(n), p[i]), per_row - 1, replace=False)] = 1.0
    return a * rng.standard_normal((n, n))


@pytest.mark.parametrize("n,share", [(36, 1.0), (40, 1.0), (63, 1.0), (40, 0.5)])
def test_full_patterns_are_given_up_at_once(n, share):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) * (rng.random((n, n)) < share)
    a[np.arange(n), np.arange(n)] = 1.0
    t0 = time.perf_counter()
    assert "suffix-product" in head(a)
    assert time.perf_counter() - t0 < 1.0  # milliseconds; 8-15 s with the tables written first


@pytest.mark.parametrize("n,per_row,columns,ops", [(26, 3, 6, 36), (30, 4, 10, 449), (36, 5, 16, 980), (38, 7, 10, 670),
                                                          (40, 4, 16, 732), (63, 3, 16, 197)])
def test_choice_of_sparse_patterns(n, per_row, columns, ops):
    assert f"{columns} inner columns summed out in {ops} operations" in head(pattern(n, per_row))
