"""Batches whose integer items take a kernel of their own behind the fused one."""
import numpy as np
import pytest

from superman_amd import api
from superman_amd.batch import BatchEngine

pytestmark = pytest.mark.gpu


def make(kind, n, seed):
    rng = np.random.default_rng([n, seed])
    if kind == "int":
        return (rng.random((n, n)) < 0.5).astype(float)
    a = rng.standard_normal((n, n))
    return a + 1j * rng.standard_normal((n, n)) if kind == "complex" else a


# 28 requests of order 26: past the line; 2: below it
@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("others", [0, 9])
def test_much_integer_work(others, use_graph):
    few = [("int", make("int", 26, s)) for s in range(2)]
    rest = [(k, make(k, n, 7)) for n in (5, 14, 21) for k in ("real", "complex", "int")][:others]
    many = [("int", make("int", 26 - s % 2, s)) for s in range(28)] + rest
    with BatchEngine(use_graph=use_graph) as eng:
        exact = {}
        alone = [eng.run([q])[0] for q in rest]
        for reqs in (few, many, few, many, many):  # each slot changes over and back
            res = eng.run(reqs)
            for i, ((kind, a), r) in enumerate(zip(reqs, res)):
                if kind == "int":
                    key = a.tobytes()
                    if key not in exact:
                        exact[key] = api.int_exact(a).exact
                    assert r.exact == exact[key], i
            for r, p in zip(res[28:], alone):  # the same bits whatever else is in the batch
                assert (r.hi, r.lo, r.exact) == (p.hi, p.lo, p.exact)
        assert eng.counters() == {"late_publish": 0, "retried": 0}
