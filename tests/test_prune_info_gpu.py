"""What a pruned integer plan says of itself: the grid of its node kernel, and
the launches of a run."""
import numpy as np
import pytest

from superman_amd import api

pytestmark = pytest.mark.gpu


# 13 and 18: the node kernel alone behind the tables; 24 and 36: one and two lists before it
@pytest.mark.parametrize("n,launches", [(13, 2), (18, 2), (24, 3), (36, 4)])
def test_grid_and_launches(n, launches):
    a = np.eye(n, dtype=np.int64) + np.roll(np.eye(n, dtype=np.int64), 1, axis=1)
    with api.DensePlan(a, "exact", int_walk="pruned") as p:
        info, r = p.info(), p.run()
    assert r.exact == 2 and r.launches == launches
    assert info["grid"] >= 1 and info["block"] == 512 and info["log2_chunk"] == 0
    assert info["tasks"] == 1 << (n - 1 - 6 * launches)
