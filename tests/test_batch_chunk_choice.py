"""A chunk size that the caller sets is taken as it is; the engine's own gives
way to the split of small requests and to the item budget."""
import numpy as np

from superman_amd import _lib
from superman_amd.batch import BatchEngine


def make(kind, n):
    a = np.random.default_rng(n).standard_normal((n, n))
    return a + 1j * a.T if kind == "complex" else a


def batches(eng, kind, n, count):
    rc, _, _, stats = eng.replay([(kind, make(kind, n))] * count, np.zeros(count))
    assert rc == 0
    return stats.batches


def test_chunk_size_of_the_caller():
    # order 20 complex: 2^19 subsets; chunks of 2^11 are 4 items of 64, of 2^7
    # 64 items; the engine's own split of such a request takes 16
    with BatchEngine(dry_run=True, max_items=16, slots=1) as eng:
        assert batches(eng, "complex", 20, 8) == 8
        t = eng.tuning
        t.waves_per_cu = 8
        eng.tuning = t  # the chunk sizes written back as they were read
        assert batches(eng, "complex", 20, 8) == 8
        t.log2_chunk["complex"] = 11
        eng.tuning = t
        assert batches(eng, "complex", 20, 8) == 2
        t.log2_chunk["complex"] = 7
        eng.tuning = t
        assert eng.try_submit("complex", make("complex", 20))[0] == _lib.SPM_ENOMEM
        assert batches(eng, "real", 20, 8) == 8  # the other kinds keep the engine's
        t.log2_chunk["complex"] = 8  # the default's value, set: 32 items
        eng.tuning = t
        assert eng.try_submit("complex", make("complex", 20))[0] == _lib.SPM_ENOMEM
