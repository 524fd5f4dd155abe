"""Where a chunk's start takes its columns from: per lane below chunk + 6, for
the whole wave above; one wave, two, four and many, real, complex and the two
dense integer walks."""
import numpy as np
import pytest

from conftest import rel_err
from oracle import oracle as O
from superman_amd import api

pytestmark = pytest.mark.gpu

TOL = 1e-10  # the bar of the dense kernels against the oracle


# walked columns outside a chunk: 5 | 6 (half a wave, one), 7, 8, 11 (2, 4, 32)
@pytest.mark.parametrize("outside", [5, 6, 7, 8, 11])
@pytest.mark.parametrize("n", [13, 16, 17])
@pytest.mark.parametrize("kind", ["real", "real zeros", "complex", "complex zeros"])
def test_dense(kind, n, outside):
    rng = np.random.default_rng([n, outside])
    a = rng.standard_normal((n, n))
    if kind.startswith("complex"):
        a = a + 1j * rng.standard_normal((n, n))
    if kind.endswith("zeros"):  # no column without zeros: one subset per step
        for j in range(n):
            a[(j + np.arange(0, n, n // 3)) % n, j] = 0
    with api.DensePlan(a) as p:
        p.set_log2_chunk(max(2, n - 1 - outside))
        assert ("pair" in p.info()["kernel"]) == (not kind.endswith("zeros") and n - 1 - outside > 2)
        v = p.run().value
    q = O.complex_dd(a) if kind.startswith("complex") else O.dense_dd(a)
    ref = complex(q[0] + q[1], q[2] + q[3]) if kind.startswith("complex") else q[0] + q[1]
    assert rel_err(v, ref) <= TOL


@pytest.mark.parametrize("walk", ["fp64", "int32"])
@pytest.mark.parametrize("n", [8, 9, 10, 12, 15, 18, 21])
def test_integer(n, walk):
    a = (np.random.default_rng(n).random((n, n)) < 0.6).astype(np.int64)
    with api.DensePlan(a, "exact", int_walk=walk) as p:
        assert p.run().exact == O.int_exact(a)[0]
