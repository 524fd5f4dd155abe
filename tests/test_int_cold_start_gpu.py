"""The FP64 integer walk on both sides of the order where its chunk starts change
(31 | 32), against the pruned walk, which shares no code with it."""
import numpy as np
import pytest

from superman_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("density", [0.3, 0.45])
@pytest.mark.parametrize("n", [30, 31, 32, 33])
def test_fp64_walk(n, density):
    a = (np.random.default_rng(n).random((n, n)) < density).astype(np.int64)
    got = []
    for walk in ("fp64", "pruned"):
        with api.DensePlan(a, "exact", int_walk=walk) as p:
            got += [p.run().exact for _ in range(2)]
    assert len(set(got)) == 1 and got[0] is not None
