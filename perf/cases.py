"""The framework's work, as cases that can be timed and compared.

A case is a dict of plain values; `prepare` makes what a user's program holds
before the call (device inputs, workspaces, plans, a server), `run` makes one
pass through the public entry points and returns the whole results, `exact`
gives the same results in 64 bits from plain torch, and `work` the bytes and
operations one pass cannot do without.

Every factorisation overwrites its input, so a pass copies the kept input into
the working buffer first, as a program that still needs A (for a residual, a
later solve, the next step) does.

Kinds:
  qr     one QR, A <- Q and R, with kept workspaces: `form` the precision form,
         `plan` a graph-captured plan instead of an eager call
  panel  one tall panel of at most 32 columns by itself
  batch  many independent matrices in one persistent launch
  gels   one least-squares solve, min ||A X - B||
  serve  a burst of least-squares requests through the server

Inputs are what the factorisation meets in regression, orthogonalisation and
polar-decomposition callers: Gaussian or uniform entries, taller than wide, and
for square matrices a Gaussian plus a multiple of the identity (a shifted or
regularised operator), so that Q is determined by the data.
"""
import math

import torch

import later_amd as later


def listed():
    return [
        # The smallest call: one small regression block, default (reference)
        # options, ragged on both sides.  Launch latency.
        {"name": "reference 1000x100", "kind": "qr", "form": "reference", "m": 1000, "n": 100, "pad": 0,
         "dist": "uniform", "plan": False},
        # One tall panel alone: the building block a caller's own blocked QR
        # uses, FP32 block Gram-Schmidt tree.
        {"name": "panel 16384x32", "kind": "panel", "m": 16384, "n": 32, "fp64": 0, "pad": 0},
        # The documented 8192 x 1024 workload in the reference's own form.
        {"name": "reference 8192x1024", "kind": "qr", "form": "reference", "m": 8192, "n": 1024, "pad": 0,
         "dist": "uniform", "plan": False},
        # Odd sizes and a leading dimension that aligns nothing, accurate form.
        {"name": "mixed 3001x333 ld+3", "kind": "qr", "form": "mixed", "m": 3001, "n": 333, "pad": 3,
         "dist": "normal", "plan": False},
        # The same 8192 x 1024 workload, accurate form, replayed from a plan as
        # a program does that factors one shape again and again.
        {"name": "mixed 8192x1024 plan", "kind": "qr", "form": "mixed", "m": 8192, "n": 1024, "pad": 0,
         "dist": "uniform", "plan": True},
        # Plain FP32 (no 16-bit operands anywhere) on an ordinary wide matrix.
        {"name": "fp32 8192x4096", "kind": "qr", "form": "fp32", "m": 8192, "n": 4096, "pad": 0,
         "dist": "normal", "plan": False},
        # Tall and skinny, the two documented shapes: accurate form, and FP8
        # first-pass projections.
        {"name": "mixed 1048576x128", "kind": "qr", "form": "mixed", "m": 1048576, "n": 128, "pad": 0,
         "dist": "normal", "plan": False},
        {"name": "fp8 262144x256", "kind": "qr", "form": "fp8", "m": 262144, "n": 256, "pad": 0,
         "dist": "normal", "plan": False},
        # The largest: the square 16384 workload, accurate form, from a plan.
        {"name": "mixed 16384x16384 plan", "kind": "qr", "form": "mixed", "m": 16384, "n": 16384, "pad": 0,
         "dist": "shifted", "plan": True},
        # Many small and medium matrices at once, sizes spread as in the
        # documented batch (m over [64, 4096], n up to 256).
        {"name": "batch 1024", "kind": "batch", "form": "mixed", "count": 1024, "mlo": 64, "mhi": 4096, "nhi": 256},
        # One least-squares solve with several right-hand sides.
        {"name": "gels 4096x512 k16", "kind": "gels", "form": "mixed", "m": 4096, "n": 512, "k": 16},
        # Least-squares requests of mixed sizes arriving together.
        {"name": "serve 16", "kind": "serve", "count": 16, "mlo": 128, "mhi": 16384, "nlo": 16, "nhi": 512},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["qr", "qr", "qr", "tall", "panel", "batch", "gels", "serve"])
    if kind == "qr":
        # From a block of a few columns to a few thousand, from barely taller
        # than wide to long.
        n = _logint(rng, 17, 3000)
        m = min(_logint(rng, int(1.5 * n) + 8, 64 * n), (1 << 25) // n)
        return {"kind": "qr", "form": rng.choice(["reference", "fp32", "mixed", "mixed"]), "m": max(m, int(1.5 * n)),
                "n": n, "pad": rng.choice([0, 0, 1, 4, 7]), "dist": rng.choice(["uniform", "normal"]),
                "plan": rng.random() < 0.3}
    if kind == "tall":
        m = _logint(rng, 40000, 700000)
        return {"kind": "qr", "form": rng.choice(["reference", "mixed", "mixed", "bf16", "fp8"]), "m": m,
                "n": rng.randint(33, 256), "pad": rng.choice([0, 0, 3]), "dist": rng.choice(["uniform", "normal"]),
                "plan": False}
    if kind == "panel":
        return {"kind": "panel", "m": _logint(rng, 100, 400000), "n": rng.randint(5, 32), "fp64": rng.choice([0, 0, 1, 2]),
                "pad": rng.choice([0, 0, 1])}
    if kind == "batch":
        return {"kind": "batch", "form": rng.choice(["mixed", "fp32"]), "count": _logint(rng, 16, 1024), "mlo": 64,
                "mhi": _logint(rng, 256, 4096), "nhi": rng.randint(32, 256)}
    if kind == "gels":
        n = _logint(rng, 17, 1000)
        return {"kind": "gels", "form": rng.choice(["mixed", "fp32"]), "m": _logint(rng, 2 * n, 32 * n), "n": n,
                "k": rng.randint(1, 16)}
    return {"kind": "serve", "count": rng.randint(2, 16), "mlo": 128, "mhi": _logint(rng, 512, 16384), "nlo": 16,
            "nhi": rng.randint(32, 512)}


# --------------------------------------------------------------------------
# Inputs, from the seed alone
# --------------------------------------------------------------------------
def _sizes(case, seed):
    """(m, n, k) of every matrix of a batch or a burst: m log-uniform, n
    uniform up to m / 2, k right-hand sides.  The sizes belong to the case
    (the same for every seed); the entries belong to the seed."""
    import random
    rng = random.Random(1000003 * case["count"] + case["mhi"])
    out = []
    for _ in range(case["count"]):
        m = _logint(rng, case["mlo"], case["mhi"])
        n = rng.randint(min(case.get("nlo", 16), m // 2), min(m // 2, case["nhi"]))
        out.append((m, n, rng.randint(1, 16)))
    return out


def _matrix(m, n, seed, mat, dist="normal", pad=0):
    A = later.colmajor(m, n, ld=m + pad)
    if dist == "uniform":
        return later.generate_uniform(m, n, seed=seed % (1 << 31), mat=mat, out=A)
    later.generate_normal(m, n, seed=seed % (1 << 31), mat=mat, out=A)
    if dist == "shifted":
        A.diagonal().add_(2.0 * math.sqrt(m))
    return A


def _rhs(A, k, seed, mat):
    """B = A X0 + noise: an ordinary regression's right-hand sides."""
    m, n = A.shape
    B = later.colmajor(m, k)
    X0 = _matrix(n, k, seed, mat + 1)
    B.copy_(A @ X0 + 1e-3 * _matrix(m, k, seed, mat + 2))
    return B


def _flat(sizes):
    """Column-major matrices of the given sizes side by side in one buffer
    each for A and R (a batch's own storage)."""
    na, nr = sum(m * n for m, n, _ in sizes), sum(n * n for _, n, _ in sizes)
    fa, fr = torch.zeros(na, device="cuda"), torch.zeros(nr, device="cuda")
    As, Rs, pa, pr = [], [], 0, 0
    for m, n, _ in sizes:
        As.append(fa[pa:pa + m * n].view(n, m).t())
        Rs.append(fr[pr:pr + n * n].view(n, n).t())
        pa += m * n
        pr += n * n
    return fa, fr, As, Rs


class _Serving:
    """A server with its requests' inputs; closed with the program's state."""

    def __init__(self, case, seed):
        self.sizes = _sizes(case, seed)
        self.A = [_matrix(m, n, seed, 8 * i) for i, (m, n, _) in enumerate(self.sizes)]
        self.B = [_rhs(a, k, seed, 8 * i) for i, (a, (_, _, k)) in enumerate(zip(self.A, self.sizes))]
        torch.cuda.synchronize()  # the server's streams read them
        self.server = later.Server(slots=8, hbm_budget_bytes=2 << 30)

    def __del__(self):
        try:
            self.server.close()
        except Exception:
            pass


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        return {"case": case, "serving": _Serving(case, seed)}
    if kind == "batch":
        sizes = _sizes(case, seed)
        src, _, srcs, _ = _flat(sizes)
        for i, a in enumerate(srcs):
            later.generate_uniform(a.shape[0], a.shape[1], seed=seed % (1 << 31), mat=i, out=a)
        fa, fr, As, Rs = _flat(sizes)
        return {"case": case, "src": src, "a": fa, "r": fr, "plan": later.BatchWg(As, Rs, later.opts(case["form"]))}
    m, n = case["m"], case["n"]
    if kind == "panel":
        A = _matrix(m, n, seed, 0, "uniform", case["pad"])
        work = torch.empty(later.caqr_panel_workspace(m, n, case["fp64"]), device="cuda", dtype=torch.float32)
        return {"case": case, "src": A, "a": later.colmajor(m, n, ld=m + case["pad"]), "r": later.colmajor(n, n),
                "work": work}
    if kind == "gels":
        A = _matrix(m, n, seed, 0)
        return {"case": case, "src": A, "b": _rhs(A, case["k"], seed, 8), "a": later.colmajor(m, n),
                "o": later.opts(case["form"])}
    o = later.opts(case["form"])
    s = {"case": case, "src": _matrix(m, n, seed, 0, case["dist"], case["pad"]),
         "a": later.colmajor(m, n, ld=m + case["pad"]), "r": later.colmajor(n, n), "o": o,
         "work": later.workspace(m, n, o), "hwork": later.hworkspace(m, n, o)}
    if case["plan"]:
        s["plan"] = later.Plan(s["a"], s["r"], o, work=s["work"], hwork=s["hwork"])
    return s


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "serve":
        v = state["serving"]
        ids = [v.server.submit(a, b) for a, b in zip(v.A, v.B)]
        while v.server.poll():
            pass
        out = [v.server.fetch(i, m, n, k) for i, (m, n, k) in zip(ids, v.sizes)]
        for i in ids:
            v.server.release(i)
        return out
    state["a"].copy_(state["src"])
    if kind == "batch":
        state["plan"].execute()
        return {"q": state["a"], "r": state["r"]}
    if kind == "panel":
        later.caqr_panel(state["a"], state["r"], fp64=case["fp64"], work=state["work"])
        return {"q": state["a"], "r": state["r"]}
    if kind == "gels":
        X, R = later.gels(state["a"], state["b"], state["o"])
        return {"x": X, "q": state["a"], "r": R}
    if "plan" in state:
        state["plan"].execute()
    else:
        later.rgsqrf(state["a"], state["r"], state["o"], work=state["work"], hwork=state["hwork"])
    return {"q": state["a"], "r": state["r"]}


# --------------------------------------------------------------------------
# What a pass cannot do without, and the results in 64 bits
# --------------------------------------------------------------------------
def work(case):
    """Reads A once, writes Q and R once; Gram-Schmidt's 2 m n^2 operations,
    and for a solve Q^T B and the triangular solve."""
    if case["kind"] in ("batch", "serve"):
        sizes = _sizes(case, 0)
    else:
        sizes = [(case["m"], case["n"], case.get("k", 0))]
    solve = case["kind"] in ("gels", "serve")
    b = sum(4 * (2 * m * n + n * n) + (4 * k * (m + n) if solve else 0) for m, n, k in sizes)
    f = sum(2 * m * n * n + ((2 * m * n + n * n) * k if solve else 0) for m, n, k in sizes)
    return {"bytes": b, "flops": f}


def _qr64(A):
    """A = Q R in 64 bits with R's diagonal positive: Cholesky QR, twice."""
    Q = A.double().t().contiguous().t()
    R = None
    for _ in range(2):
        L = torch.linalg.cholesky(Q.t().contiguous() @ Q)
        I = torch.eye(L.shape[0], device=L.device, dtype=L.dtype)
        Q = Q @ torch.linalg.solve_triangular(L, I, upper=False).t()
        R = L.t().contiguous() if R is None else L.t().contiguous() @ R
    return Q, torch.triu(R)


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        v = _Serving(case, seed)
        out = []
        for a, b in zip(v.A, v.B):
            Q, R = _qr64(a)
            out.append([torch.linalg.solve_triangular(R, Q.t().contiguous() @ b.double(), upper=True), R])
        return out
    if kind == "batch":
        s = prepare(case, seed)
        q, r, p = torch.empty_like(s["a"], dtype=torch.float64), torch.empty_like(s["r"], dtype=torch.float64), [0, 0]
        for m, n, _ in _sizes(case, seed):
            Q, R = _qr64(s["src"][p[0]:p[0] + m * n].view(n, m).t())
            q[p[0]:p[0] + m * n] = Q.t().reshape(-1)
            r[p[1]:p[1] + n * n] = R.t().reshape(-1)
            p[0] += m * n
            p[1] += n * n
        return {"q": q, "r": r}
    if kind == "gels":
        A = _matrix(case["m"], case["n"], seed, 0)
        Q, R = _qr64(A)
        B = _rhs(A, case["k"], seed, 8)
        return {"x": torch.linalg.solve_triangular(R, Q.t().contiguous() @ B.double(), upper=True), "q": Q, "r": R}
    Q, R = _qr64(_matrix(case["m"], case["n"], seed, 0, case.get("dist", "uniform"), case["pad"]))
    return {"q": Q, "r": R}
