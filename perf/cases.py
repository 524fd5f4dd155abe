"""The work that a user of this framework has it do, as cases that can be
timed and checked: one-shot calls from the smallest order to the order-40
permanent, plans kept for a matrix, every kind of matrix (real, complex, 0/1
and integer, sparse integer, sparse real) and a batch of mixed requests.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the matrix (host memory, as every entry point takes
                        it) and the plan or engine a program keeps for it
    run(state)          one call through the public entry points
    work(case)          bytes and flops one pass cannot do without
    exact(case, seed)   what run() returns, from plain numpy / torch in 64 bits
"""
import math

import numpy as np
import torch

from superman_amd import api
from superman_amd.batch import BatchEngine

# ---------------------------------------------------------------- cases
LISTED = [
    # the smallest call: latency and launches are all of it
    {"name": "real_n8_call", "op": "real", "n": 8, "dist": "uniform", "precision": "kahan", "plan": False},
    # the benchmark's small dense matrix: one call on a fresh matrix
    {"name": "real_n24_call", "op": "real", "n": 24, "dist": "uniform", "precision": "kahan", "plan": False},
    # an odd order with the reference's plain FP64 precision
    {"name": "real_n33_dd", "op": "real", "n": 33, "dist": "normal", "precision": "dd", "plan": False},
    # the headline: dense order 40, compensated, the matrix resident in a plan
    {"name": "real_n40_plan", "op": "real", "n": 40, "dist": "normal", "precision": "kahan", "plan": True},
    # a small complex matrix (boson-sampling amplitude), one call
    {"name": "complex_n21_call", "op": "complex", "n": 21, "dist": "gauss", "precision": "kahan", "plan": False},
    # the benchmark's Haar-random unitary block
    {"name": "complex_n32_haar", "op": "complex", "n": 32, "dist": "haar", "precision": "kahan", "plan": False},
    # a dense 0/1 matrix (bipartite perfect matchings), counted exactly through the automatic choice
    {"name": "int01_n30_auto", "op": "int", "n": 30, "density": 0.5, "vmax": 1},
    # sparse 0/1, order 40, about 4 entries per row: one exact call
    {"name": "sparse01_n40_exact", "op": "sparse_int", "n": 40, "per_row": 4, "how": "exact"},
    # the same kind of matrix through a kernel generated for its pattern and kept
    {"name": "sparse01_n40_codegen", "op": "sparse_int", "n": 40, "per_row": 4, "how": "codegen"},
    # and through the whole preprocessing pipeline (pruning, components, compressions)
    {"name": "sparse01_n40_decomposed", "op": "sparse_int", "n": 40, "per_row": 4, "how": "decomposed"},
    # a sparse real matrix through its generated kernel
    {"name": "sparse_real_n36_codegen", "op": "sparse_real", "n": 36, "per_row": 5, "precision": "kahan"},
    # a batch of mixed requests (half real, 30 % complex, 20 % 0/1), one synchronous call
    {"name": "batch_mixed_256", "op": "batch", "count": 256, "n_lo": 8, "n_hi": 24},
]


def listed():
    return [dict(c) for c in LISTED]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["real", "real", "real", "complex", "complex", "int", "sparse_int", "sparse_int", "sparse_real",
                     "batch"])
    if op == "real":
        n = rng.randint(4, 38)
        dist = "normal" if n > 26 else rng.choice(["uniform", "normal"])
        return {"op": op, "n": n, "dist": dist, "precision": rng.choice(["kahan", "kahan", "dd"]),
                "plan": rng.random() < 0.4}
    if op == "complex":
        n = rng.randint(4, 33)
        return {"op": op, "n": n, "dist": "haar" if n > 28 else rng.choice(["gauss", "haar"]),
                "precision": rng.choice(["kahan", "kahan", "dd"]), "plan": rng.random() < 0.4}
    if op == "int":
        if rng.random() < 0.5:
            return {"op": op, "n": rng.randint(8, 32), "density": round(rng.uniform(0.3, 0.7), 2), "vmax": 1}
        return {"op": op, "n": rng.randint(6, 20), "density": round(rng.uniform(0.2, 0.35), 2),
                "vmax": rng.choice([2, 3, 5])}
    if op == "sparse_int":
        how = rng.choice(["exact", "codegen", "decomposed"])
        per_row = rng.choice([4, 6]) if how == "codegen" else rng.randint(3, 6)
        n = rng.randint(24, 36 if per_row % 2 else 40)
        if how == "decomposed":
            n, per_row = rng.randint(30, 40), min(per_row, 4)
        return {"op": op, "n": n, "per_row": per_row, "how": how}
    if op == "sparse_real":
        return {"op": op, "n": rng.randint(26, 38), "per_row": rng.randint(3, 7),
                "precision": rng.choice(["kahan", "kahan", "dd"])}
    return {"op": op, "count": _log_int(rng, 24, 512), "n_lo": rng.randint(4, 10), "n_hi": rng.randint(14, 25)}


# ---------------------------------------------------------------- inputs
def _rng(seed, *key):
    return np.random.default_rng([seed & 0x7FFFFFFF, *key])


def _pattern(rng, n, per_row):
    """0/1: a random permutation plus per_row - 1 further entries per row."""
    a = np.zeros((n, n))
    p = rng.permutation(n)
    for i in range(n):
        a[i, p[i]] = 1.0
        others = np.delete(np.arange(n), p[i])
        a[i, rng.choice(others, per_row - 1, replace=False)] = 1.0
    return a


def _matrix(case, seed):
    op, n = case["op"], case["n"]
    rng = _rng(seed, n)
    if op == "real":
        return rng.random((n, n)) if case["dist"] == "uniform" else rng.standard_normal((n, n))
    if op == "complex":
        if case["dist"] == "gauss":
            return (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(2.0)
        m = 2 * n
        z = (rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))) / np.sqrt(2.0)
        q, r = np.linalg.qr(z)
        d = np.diag(r)
        return np.ascontiguousarray((q * (d / np.abs(d))[None, :])[:n, :n])
    if op == "int":
        nz = rng.random((n, n)) < case["density"]
        if case["vmax"] == 1:
            return nz.astype(np.float64)
        nz[np.arange(n), rng.permutation(n)] = True
        v = rng.integers(1, case["vmax"] + 1, (n, n)) * rng.choice([-1, 1], (n, n))
        return (v * nz).astype(np.int64)
    if op == "sparse_int":
        return _pattern(rng, n, case["per_row"])
    return _pattern(rng, n, case["per_row"]) * rng.standard_normal((n, n))  # sparse_real


def _requests(case, seed):
    count = case["count"]
    rng = _rng(seed, count)
    kinds = ["real"] * (count // 2) + ["complex"] * (3 * count // 10)
    kinds += ["int"] * (count - len(kinds))
    out = []
    for k in rng.permutation(count):
        n = int(rng.integers(case["n_lo"], case["n_hi"] + 1))
        if kinds[k] == "real":
            a = rng.random((n, n))
        elif kinds[k] == "complex":
            a = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(2.0)
        else:
            a = (rng.random((n, n)) < 0.5).astype(np.float64)
        out.append((kinds[k], a))
    return out


def prepare(case, seed):
    op = case["op"]
    if op == "batch":
        return {"case": case, "engine": BatchEngine(), "requests": _requests(case, seed)}
    a = _matrix(case, seed)
    s = {"case": case, "a": a, "plan": None}
    if op in ("real", "complex") and case["plan"]:
        s["plan"] = api.DensePlan(a, case["precision"])
    elif op == "sparse_int" and case["how"] == "codegen":
        s["plan"] = api.CodegenPlan(a)
    elif op == "sparse_real":
        s["plan"] = api.CodegenRealPlan(a, case["precision"])
    return s


# ---------------------------------------------------------------- one pass
def _real(r):
    return {"value": np.float64(r.value), "abs_sum": np.float64(r.abs_sum)}


def _complex(r):
    return {"value": np.complex128(r.value), "abs_sum": np.float64(r.abs_sum)}


def _words(values):
    """Exact integers as (high, low) 64-bit words."""
    w = [((v >> 64) & (2**64 - 1), v & (2**64 - 1)) for v in values]
    return np.array(w, dtype=np.uint64).reshape(len(w), 2).view(np.int64)


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "batch":
        res = s["engine"].run(s["requests"])
        kinds = [k for k, _ in s["requests"]]
        return {"real": np.array([r.value for r, k in zip(res, kinds) if k == "real"], dtype=np.float64),
                "complex": np.array([r.value for r, k in zip(res, kinds) if k == "complex"], dtype=np.complex128),
                "int": _words([r.exact for r, k in zip(res, kinds) if k == "int"])}
    if op in ("real", "complex"):
        r = s["plan"].run() if s["plan"] is not None else api.permanent(s["a"], case["precision"])
        return _complex(r) if op == "complex" else _real(r)
    if op == "sparse_real":
        return _real(s["plan"].run())
    if op == "int":
        r = api.permanent(s["a"]) if case["vmax"] == 1 else api.int_exact(s["a"])
    elif case["how"] == "exact":
        r = api.int_exact(s["a"])
    elif case["how"] == "codegen":
        r = s["plan"].run()
    else:
        r = api.permanent_decomposed(s["a"])
    if r.exact is None:  # beyond the 128-bit range: an FP64 permanent
        return _real(r)
    return {"exact": _words([r.exact])}


# ---------------------------------------------------------------- work
def work(case):
    """The matrix read once, the result written once, and the flops of the
    Gray-code Ryser formula: per subset one add and one multiply per row
    (complex: 2 + 6); sparse ones add only the flipped column's entries.  An
    exact integer permanent multiplies out only the terms with no zero row,
    a vanishing share here."""
    op = case["op"]
    if op == "batch":
        per = [(0.5 * 2 + 0.3 * 8 + 0.2 * 1) * n * 2.0 ** (n - 1) for n in range(case["n_lo"], case["n_hi"] + 1)]
        byt = [(0.7 * 8 + 0.3 * 16) * n * n + 88 for n in range(case["n_lo"], case["n_hi"] + 1)]
        return {"bytes": case["count"] * sum(byt) / len(byt), "flops": case["count"] * sum(per) / len(per)}
    n = case["n"]
    subsets = 2.0 ** (n - 1)
    per = {"real": 2.0 * n, "complex": 8.0 * n, "int": 1.0 * n, "sparse_int": case.get("per_row", 0),
           "sparse_real": 2.0 * case.get("per_row", 0)}[op]
    return {"bytes": (16.0 if op == "complex" else 8.0) * n * n + 88, "flops": per * subsets}


# ---------------------------------------------------------------- exact values
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _two_sum(a, b):
    s = a + b
    t = s - a
    return s, (a - (s - t)) + (b - t)


def _split(a):
    c = a * 134217729.0
    h = c - (c - a)
    return h, a - h


def _dd_add(a, b):
    s, e = _two_sum(a[0], b[0])
    e = e + (a[1] + b[1])
    h = s + e
    return h, e - (h - s)


def _dd_mul(a, b):
    p = a[0] * b[0]
    ah, al = _split(a[0])
    bh, bl = _split(b[0])
    e = ((ah * bh - p) + ah * bl + al * bh) + al * bl
    e = e + (a[0] * b[1] + a[1] * b[0])
    h = p + e
    return h, e - (h - p)


def _row_start(row):
    """a_{i,n-1} - rowsum / 2, as an unevaluated pair of doubles."""
    terms = [float(row[-1])] + [-0.5 * float(v) for v in row]
    hi = math.fsum(terms)
    return hi, math.fsum(terms + [-hi])


def _subset_parity(bits, device):
    k = torch.arange(1 << bits, device=device)
    par = torch.zeros(1 << bits, dtype=torch.int64, device=device)
    for j in range(bits):
        par ^= (k >> j) & 1
    return 1.0 - 2.0 * par.double()


def _ryser_dd(parts, n):
    """perm of the real (one part) or complex (re, im) matrix in pairs of
    doubles: 2 (-1)^(n-1) sum_S (-1)^|S| prod_i x_i(S)."""
    dev = _device()
    cplx = len(parts) == 2
    bits = n - 1
    low = min(bits, 18 if cplx else 20)
    sign = _subset_parity(low, dev)
    idx = torch.arange(1 << low, device=dev)
    total = [[], []]
    starts = [[_row_start(m[i]) for i in range(n)] for m in parts]
    for high in range(1 << (bits - low)):
        neg = bin(high).count("1") & 1
        prod = None
        for i in range(n):
            x = []
            for m, st in zip(parts, starts):
                h, l = st[i]
                base = [h, l] + [float(m[i][low + j]) for j in range(bits - low) if (high >> j) & 1]
                bh = math.fsum(base)
                v = (torch.full((1 << low,), bh, device=dev, dtype=torch.float64),
                     torch.full((1 << low,), math.fsum(base + [-bh]), device=dev, dtype=torch.float64))
                for j in range(low):
                    on = ((idx >> j) & 1).double() * float(m[i][j])
                    v = _dd_add(v, (on, torch.zeros_like(on)))
                x.append(v)
            if prod is None:
                prod = x
            elif not cplx:
                prod = [_dd_mul(prod[0], x[0])]
            else:
                t = _dd_mul(prod[1], x[1])
                re = _dd_add(_dd_mul(prod[0], x[0]), (-t[0], -t[1]))
                im = _dd_add(_dd_mul(prod[0], x[1]), _dd_mul(prod[1], x[0]))
                prod = [re, im]
        for c, (h, l) in enumerate(prod):
            v = (h * sign, l * sign)
            while v[0].numel() > 1:
                half = v[0].numel() // 2
                v = _dd_add((v[0][:half], v[1][:half]), (v[0][half:], v[1][half:]))
            f = -1.0 if neg else 1.0
            total[c] += [f * float(v[0][0]), f * float(v[1][0])]
    f = 2.0 if (n - 1) % 2 == 0 else -2.0
    return [f * math.fsum(t) for t in total[:len(parts)]]


def _ryser_f64(a, n):
    """The same sum in plain FP64 / complex128 (orders too large for pairs)."""
    dev = _device()
    dt = torch.complex128 if np.iscomplexobj(a) else torch.float64
    t = torch.tensor(a, dtype=dt, device=dev)
    bits = n - 1
    low = min(bits, 22)
    start = t[:, -1] - 0.5 * t.sum(1)
    sign = _subset_parity(low, dev)
    tab = torch.zeros((n, 1), dtype=dt, device=dev) + start[:, None]
    for j in range(low):
        tab = torch.cat([tab, tab + t[:, j:j + 1]], dim=1)
    sums = torch.zeros((), dtype=dt, device=dev)
    ah = t[:, low:bits]
    for high in range(1 << (bits - low)):
        on = torch.tensor([(high >> j) & 1 for j in range(bits - low)], dtype=torch.float64, device=dev)
        base = (ah * on.to(dt)).sum(1)
        p = tab[0] + base[0]
        for i in range(1, n):
            p = p * (tab[i] + base[i])
        s = (p * sign).sum()
        sums = sums - s if bin(high).count("1") & 1 else sums + s
    f = 2.0 if (n - 1) % 2 == 0 else -2.0
    return f * sums.item()


def _sparse_perm(a):
    """Expansion row by row over the sets of used columns (sets that can no
    longer be completed are dropped): no cancellation but the matrix's own."""
    n = a.shape[0]
    rows = [set(np.flatnonzero(a[i])) for i in range(n)]
    left, opened, order = set(range(n)), set(), []
    while left:
        i = min(left, key=lambda r: (len(rows[r] - opened), r))
        order.append(i)
        opened |= rows[i]
        left.discard(i)
    last = {j: max(k for k, i in enumerate(order) if j in rows[i]) for j in range(n) if any(j in r for r in rows)}
    masks, vals = np.zeros(1, dtype=np.int64), np.ones(1)
    for k, i in enumerate(order):
        must = 0
        for j, at in last.items():
            if at <= k:
                must |= 1 << int(j)
        nm, nv = [], []
        for j in rows[i]:
            bit = np.int64(1) << np.int64(j)
            ok = (masks & bit) == 0
            m = masks[ok] | bit
            v = vals[ok] * a[i, j]
            keep = (m & must) == must
            nm.append(m[keep])
            nv.append(v[keep])
        masks, vals = np.concatenate(nm), np.concatenate(nv)
        if masks.size == 0:
            return 0.0
        if masks.size > 12_000_000:
            return None
        at = np.argsort(masks, kind="stable")
        masks, vals = masks[at], vals[at]
        first = np.flatnonzero(np.concatenate([[True], masks[1:] != masks[:-1]]))
        masks, vals = masks[first], np.add.reduceat(vals, first)
    return float(vals.sum())


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        req = _requests(case, seed)
        if max(a.shape[0] for _, a in req) > 25 or case["count"] > 300:
            return None
        re, cx = [], []
        for k, a in req:
            if k == "real":
                re.append(_ryser_f64(a, a.shape[0]))
            elif k == "complex":
                cx.append(_ryser_f64(a, a.shape[0]))
        return {"real": np.array(re, dtype=np.float64), "complex": np.array(cx, dtype=np.complex128), "int": None}
    if op in ("int", "sparse_int"):
        return None  # whole numbers
    a, n = _matrix(case, seed), case["n"]
    if op == "sparse_real":
        v = _sparse_perm(a)
        return None if v is None else {"value": np.float64(v), "abs_sum": None}
    if op == "real":
        v = _ryser_dd([a.tolist()], n)[0] if n <= 25 else _ryser_f64(a, n) if n <= 34 else None
        return None if v is None else {"value": np.float64(v), "abs_sum": None}
    if n <= 21:
        v = complex(*_ryser_dd([a.real.tolist(), a.imag.tolist()], n))
    else:
        v = _ryser_f64(a, n) if n <= 32 else None
    return None if v is None else {"value": np.complex128(v), "abs_sum": None}
