"""Generated integer kernels that sieve the chunks' prefixes before walking
them (orders from 24, patterns whose rows are completed outside a chunk):
bit-exact against the int128 oracle, the search over column groups and
closed forms."""
import numpy as np
import pytest

from oracle import oracle as O
from superman_amd import api

pytestmark = pytest.mark.gpu


def pattern(n, per_row, seed, values=(1,)):
    rng = np.random.default_rng(seed)
    a = np.zeros((n, n), dtype=np.int64)
    p = rng.permutation(n)
    for i in range(n):
        a[i, p[i]] = 1
        a[i, rng.choice(np.delete(np.arange(n), p[i]), per_row - 1, replace=False)] = 1
    return a * rng.choice(values, (n, n))


def is_sieved(a):
    return "queue[at & 127u]" in api.codegen_source(a)


# 24: the first sieved order (a block per part, every task its own part);
# 27, 28: batches of one and two parts; 33 and 34: whole blocks, and batches
# of 64 from 36 on; 31: terms tested per block
@pytest.mark.parametrize("n,per_row,values", [(24, 4, (1,)), (24, 2, (1, -1)), (25, 4, (-2, -1, 1, 2)), (27, 4, (1,)),
                                              (28, 6, (1,)), (31, 4, (1,)), (33, 4, (-1, 1)), (34, 6, (1,)),
                                              (36, 4, (1,)), (37, 6, (1,)), (41, 4, (1,))])
def test_sieved_kernels_are_exact(n, per_row, values):
    a = pattern(n, per_row, 10 * n + per_row, values)
    if n <= 25:
        ref, st = O.int_exact(a)
        assert st == 0
    else:
        with api.DensePlan(a, "exact", int_walk="pruned") as q:
            ref = q.run().exact
    assert is_sieved(a)
    with api.CodegenPlan(a) as p:
        assert p.run().exact == ref
        assert p.run().exact == ref


def test_rows_never_zero_keep_the_whole_walk():
    a = pattern(26, 3, 1)  # odd row sums
    assert not is_sieved(a)
    with api.DensePlan(a, "exact", int_walk="fp64") as q:
        assert api.sparse_codegen(a).exact == q.run().exact
    assert not is_sieved(pattern(23, 4, 1))


@pytest.mark.parametrize("n", [26, 40, 47])
def test_triangular_closed_form(n):
    # ones on the diagonal and 3 more per row above it: perm = 1
    rng = np.random.default_rng(n)
    a = np.eye(n, dtype=np.int64)
    for i in range(n - 1):
        above = np.arange(i + 1, n)
        a[i, rng.choice(above, size=min(3, above.size), replace=False)] = 1
    assert api.sparse_codegen(a).exact == 1
