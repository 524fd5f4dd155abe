"""Plan memory from a pool (csrc/workspace.cpp): plans that live at once,
more than the pool keeps, in any order, on several threads and streams, give
the results of a plan alone."""
import ctypes
import threading

import numpy as np
import pytest

from superman_amd import api

pytestmark = pytest.mark.gpu


def matrix(kind, n, seed):
    rng = np.random.default_rng([n, seed])
    if kind == "real":
        return rng.standard_normal((n, n))
    if kind == "complex":
        return rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    return (rng.random((n, n)) < 0.5).astype(np.int64)


def plan(kind, a):
    return api.DensePlan(a, "exact" if kind == "int" else "kahan")


def value(r):
    return r.exact if r.exact is not None else (r.hi, r.lo, r.abs_sum)


CASES = [(k, n) for n in (3, 9, 14, 19, 26) for k in ("real", "complex", "int") if (k, n) != ("complex", 26)]


def test_plans_alive_together():
    alone = {}
    for k, n in CASES:
        with plan(k, matrix(k, n, 1)) as p:
            alone[k, n] = value(p.run())
    plans = {c: plan(c[0], matrix(*c, 1)) for c in CASES}
    rng = np.random.default_rng(0)
    for _ in range(3):
        for i in rng.permutation(len(CASES)):
            assert value(plans[CASES[i]].run()) == alone[CASES[i]]
    for i in rng.permutation(len(CASES)):  # dropped and made again in another order
        plans.pop(CASES[i]).close()
        with plan(CASES[i][0], matrix(*CASES[i], 1)) as p:
            assert value(p.run()) == alone[CASES[i]]


def test_calls_on_threads_and_streams():
    hip = ctypes.CDLL("libamdhip64.so")
    want = {(k, n, s): value(plan(k, matrix(k, n, s)).run()) for k, n in CASES if n < 26 for s in range(2)}
    bad = []

    def work(t):
        stream = ctypes.c_void_p()
        if hip.hipStreamCreate(ctypes.byref(stream)) != 0:
            bad.append((t, "hipStreamCreate"))
            return
        for rep in range(6):
            for k, n, s in sorted(want)[t::4]:
                a = matrix(k, n, s)
                f = {"real": api.dense_f64, "complex": api.dense_c128, "int": api.int_exact}[k]
                r = f(a, stream=stream.value if rep % 2 else None)
                if value(r) != want[k, n, s]:
                    bad.append((t, k, n, s))
        hip.hipStreamDestroy(stream)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_device_time_is_reported():
    with api.DensePlan(matrix("real", 28, 3), "kahan") as p:
        r = [p.run() for _ in range(3)]
    for q in r:
        assert 0.05 < q.kernel_ms < 1e3 * q.seconds + 0.05
