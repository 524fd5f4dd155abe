"""A chunk size that the caller sets is an upper limit, and the one that counts
for the item budget; the engine's own also gives way to that."""
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
    # order 20 complex, 2^19 subsets: the engine's 2^8 steps are 32 items of 64
    # chunks, more than the budget, and give way to 2^9, the split's limit
    with BatchEngine(dry_run=True, max_items=16, slots=1) as eng:
        assert batches(eng, "complex", 20, 4) == 4
        t = eng.tuning
        t.waves_per_cu = 8
        eng.tuning = t  # the chunk sizes written back as they were read
        assert batches(eng, "complex", 20, 4) == 4
        for steps, st in ((11, 0), (9, 0), (7, _lib.SPM_ENOMEM), (8, _lib.SPM_ENOMEM)):
            t.log2_chunk["complex"] = steps  # (8 is the default's value, now set)
            eng.tuning = t
            assert eng.try_submit("complex", make("complex", 20))[0] == st, steps
            while eng.poll() or eng.progress():
                pass
        assert batches(eng, "real", 20, 4) == 4  # the other kinds keep the engine's
    with BatchEngine(dry_run=True, max_items=64, slots=1) as eng:
        t = eng.tuning
        t.log2_chunk["complex"] = 13  # split to 2^9 steps all the same: 4 requests a batch
        eng.tuning = t
        assert batches(eng, "complex", 20, 8) == 2
        t.log2_chunk["complex"] = 7  # as short as it is set: one request a batch
        eng.tuning = t
        assert batches(eng, "complex", 20, 8) == 8
