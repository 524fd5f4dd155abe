"""The pruned walk on matrices whose entries are small but for one column: its
entries are in no field (the column is walked by no subset) and in the rows'
values all the same, so products of two or four rows outgrow 32 bits.  The
layout's product mode must form them exactly, or leave the matrix to the other
walks."""
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O
from superman_amd import _lib, api

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="session")
def layout(tmp_path_factory):
    """matrix -> (field bytes, mode, [(o, width)]) or None, from prune_plan."""
    out = str(tmp_path_factory.mktemp("prune") / "prune_plan")
    pkg = os.path.join(ROOT, "superman_amd")
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(pkg, "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "prune_plan_main.cpp"), "-L" + pkg, "-lsuperman_amd",
                    "-Wl,-rpath," + pkg, "-Wl,--allow-shlib-undefined", "-o", out], check=True)

    def run(a):
        text = "%d %s\n" % (a.shape[0], " ".join(str(int(v)) for v in a.ravel()))
        t = subprocess.run([out], input=text, capture_output=True, text=True, check=True).stdout.split()
        if t[0] == "none":
            return None
        v = [int(x) for x in t]
        return v[0], v[2], list(zip(v[3::2], v[4::2]))

    return run


def column(n, rows, value, per_row=3, seed=0):
    """per_row ones a row, one column of ones with `value` in `rows` rows."""
    rng = np.random.default_rng([n, rows, per_row, seed])
    a = np.zeros((n, n), dtype=np.int64)
    for i in range(n):
        a[i, rng.choice(n - 1, per_row, replace=False)] = 1
    a[:, n - 1] = 1
    a[rng.choice(n, rows, replace=False), n - 1] = value
    return a[:, rng.permutation(n)]


def groups(fb, mode, fields):
    """Index sets that one product() of this mode forms in 32 and in 64 bits."""
    run = lambda k: [list(range(i, i + k)) for i in range(0, fields, k)]  # noqa: E731
    if fb == 2:
        return [], run(4 if mode == 1 else 2)
    if mode == 0:
        return run(2), run(4)
    wide = run(8)
    return run(4), wide if mode == 1 else [x + y for x, y in zip(wide[: len(wide) // 2], wide[len(wide) // 2:])]


@pytest.mark.parametrize("value", [1, 3, 300, 92681, 92683, -92683, 200001, (1 << 20) + 1, -(1 << 24)])
@pytest.mark.parametrize("n,rows", [(13, 2), (16, 16), (20, 3), (24, 2), (24, 4), (32, 5), (40, 3), (43, 2), (44, 2),
                                    (63, 2)])
def test_products_fit_their_words(layout, n, rows, value):
    p = layout(column(n, rows, value))
    if p is None:  # no 16-bit layout past order 43, or the column is walked and outgrows 16 bits
        assert abs(value) > 46341 and (n > 43 or rows == n)
        return
    fb, mode, field = p
    top = [max(abs(o), abs(o + w), 1) for o, w in field]
    narrow, wide = groups(fb, mode, len(field))
    for bits, sets in ((31, narrow), (63, wide)):
        for g in sets:
            prod = 1
            for i in g:
                prod *= top[i]
            assert prod < 1 << bits, (fb, mode, g)


@pytest.mark.gpu
@pytest.mark.parametrize("value", [92681, 92683, -92683, 200001, 300001, 400001])
@pytest.mark.parametrize("n,rows,per_row", [(13, 2, 3), (18, 3, 3), (20, 4, 3), (24, 3, 3), (26, 2, 3)])
def test_exact(n, rows, per_row, value):
    a = column(n, rows, value, per_row)
    ref, st = O.int_exact(a)
    assert st == 0
    for walk in ("pruned", "auto", "int32"):
        with api.DensePlan(a, "exact", int_walk=walk) as p:
            assert p.run().exact == ref, walk
    assert api.int_exact(a).exact == ref
    assert api.permanent(a.astype(np.float64)).exact == ref


@pytest.mark.gpu
def test_order_28_and_refused_orders():
    a = column(28, 2, 92683)
    ref, st = O.int_exact(a)
    assert st == 0 and api.int_exact(a).exact == ref
    with api.DensePlan(a, "exact", int_walk="pruned") as p:
        assert p.run().exact == ref
    b = np.eye(44, dtype=np.int64) + np.roll(np.eye(44, dtype=np.int64), 1, axis=1)
    b[:, 7] += 1
    b[:4, 7] = 92683
    with pytest.raises(_lib.SpmError) as e:
        api.DensePlan(b, "exact", int_walk="pruned")
    assert e.value.status == _lib.SPM_ERANGE
