"""What is timed: the solves and factorizations that programs built on this library make,
through its public entry points (`elemental_amd.device` for data resident in HBM, the C API of
`include/El.h` for host buffers).

A case is a dict of plain values. `kind` selects the entry point:

  solve        device.gesv        one system, B overwritten with the solution
  lu           device.getrf + getrs, the factors kept and solved with
  hpd          device.posv        Cholesky factor and solve
  mixed        device.gesv_mixed  low-precision LU with FP64 refinement
  hpd_mixed    device.posv_mixed  the same for HPD systems
  batched_hpd  device.potrf_vbatched + potrs_vbatched, or one PosvGraph replay
  batched_lu   device.gesv_mixed_batched
  host         ElLinearSolve_d    the drop-in C call on host buffers

The factorizations work in place, so a pass that may be repeated first refreshes its working
matrix from the caller's, as El::LinearSolve and El::HPDSolve do. The leading dimension is the
height plus `pad`.
"""
import ctypes
import math

import numpy as np
import torch

import elemental_amd
from elemental_amd import device as dev

_DTYPE = {"f64": torch.float64, "f32": torch.float32}
_EXACT_ORDER = 6144  # largest order whose LAPACK solution takes a few seconds on host cores


def listed():
    return [
        # the smallest call: one small dense system, where the chain of launches is the cost
        {"name": "solve_small", "kind": "solve", "n": 200, "nrhs": 1, "pad": 0, "kappa": 0.0},
        # an ordinary LU that is kept and solved with: n = 1024, one right-hand side
        {"name": "lu_ordinary", "kind": "lu", "n": 1024, "nrhs": 1, "pad": 0, "orient": 0,
         "kappa": 0.0},
        # a ragged submatrix (odd leading dimension) and a transposed solve of several
        # right-hand sides, as sensitivity and adjoint computations make
        {"name": "lu_ragged_adjoint", "kind": "lu", "n": 3001, "nrhs": 7, "pad": 2, "orient": 1,
         "kappa": 0.0},
        # a large FP64 system by the plain path
        {"name": "solve_large", "kind": "solve", "n": 16384, "nrhs": 1, "pad": 0,
         "kappa": 100.0},
        # HPD system n = 16384 with 16 right-hand sides, FP64
        {"name": "hpd_large", "kind": "hpd", "n": 16384, "nrhs": 16, "pad": 0, "dtype": "f64",
         "uplo": 0},
        # an FP32 HPD system of ragged order held in its upper triangle
        {"name": "hpd_f32_ragged", "kind": "hpd", "n": 4700, "nrhs": 3, "pad": 4,
         "dtype": "f32", "uplo": 1},
        # the mixed-precision headline: n = 32768, kappa = 100, one right-hand side, fp16 factors
        {"name": "mixed_large", "kind": "mixed", "n": 32768, "nrhs": 1, "kappa": 100.0,
         "factor": "fp16"},
        # the mixed HPD solve, several right-hand sides refined as one block
        {"name": "hpd_mixed", "kind": "hpd_mixed", "n": 8192, "nrhs": 16, "factor": "fp16"},
        # thousands of HPD systems of uneven sizes in one launch, FP64
        {"name": "batched_hpd", "kind": "batched_hpd", "count": 3000, "nmin": 16, "nmax": 512,
         "dtype": "f64", "graph": 0},
        # small FP32 systems refilled and replayed through the captured graph
        {"name": "batched_hpd_f32_graph", "kind": "batched_hpd", "count": 5000, "nmin": 16,
         "nmax": 128, "dtype": "f32", "graph": 1},
        # many nonsymmetric systems of uneven sizes and conditioning, 4 right-hand sides each
        {"name": "batched_lu", "kind": "batched_lu", "count": 300, "nmin": 64, "nmax": 1024,
         "kmax": 1e4, "nrhs": 4},
        # the drop-in call of a C or C++ program: host matrices in, solution out
        {"name": "host_solve", "kind": "host", "n": 2000, "nrhs": 1},
    ]


def _log_int(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    n = min(max(n, lo), hi)
    # half of the sizes as they fall (mostly odd against every tile), half on multiples of 32
    return n if rng.random() < 0.5 or n < 64 else n // 32 * 32


def draw(rng):
    kind = rng.choice(["solve", "solve", "lu", "lu", "hpd", "hpd", "mixed", "hpd_mixed",
                       "batched_hpd", "batched_hpd", "batched_lu", "host"])
    if kind == "solve":
        return {"kind": kind, "n": _log_int(rng, 64, 12288), "nrhs": rng.choice([1, 1, 2, 5, 16]),
                "pad": rng.choice([0, 0, 1, 8]), "kappa": rng.choice([0.0, 100.0])}
    if kind == "lu":
        return {"kind": kind, "n": _log_int(rng, 64, 8192), "nrhs": rng.choice([1, 3, 8, 64]),
                "pad": rng.choice([0, 0, 1, 2, 16]), "orient": rng.choice([0, 0, 1]),
                "kappa": rng.choice([0.0, 100.0])}
    if kind == "hpd":
        return {"kind": kind, "n": _log_int(rng, 64, 12288), "nrhs": rng.choice([1, 4, 16, 33]),
                "pad": rng.choice([0, 0, 1, 4]), "dtype": rng.choice(["f64", "f64", "f32"]),
                "uplo": rng.choice([0, 0, 1])}
    if kind == "mixed":
        return {"kind": kind, "n": _log_int(rng, 2048, 20480), "nrhs": rng.choice([1, 1, 1, 4]),
                "kappa": round(10.0 ** rng.uniform(1, 3), 1),
                "factor": rng.choice(["fp16", "fp16", "bf16", "fp32"])}
    if kind == "hpd_mixed":
        return {"kind": kind, "n": _log_int(rng, 2048, 12288), "nrhs": rng.choice([1, 4, 16]),
                "factor": rng.choice(["fp16", "fp16", "bf16"])}
    if kind == "batched_hpd":
        return {"kind": kind, "count": _log_int(rng, 200, 4000), "nmin": 16,
                "nmax": rng.choice([64, 128, 200, 256, 384, 512]),
                "dtype": rng.choice(["f64", "f32"]), "graph": rng.choice([0, 1])}
    if kind == "batched_lu":
        return {"kind": kind, "count": _log_int(rng, 50, 400), "nmin": 64,
                "nmax": rng.choice([256, 512, 1000]), "kmax": rng.choice([1e2, 1e4]),
                "nrhs": rng.choice([1, 4])}
    return {"kind": kind, "n": _log_int(rng, 100, 4096), "nrhs": rng.choice([1, 3])}


# ------------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, dtype=torch.float64, device="cuda", generator=g)


def _colmajor(m, n, pad, dtype=torch.float64):
    """An uninitialised column-major m x n matrix of leading dimension m + pad."""
    return torch.empty((n, m + pad), dtype=dtype, device="cuda").t()[:m]


def _colmajor_of(a, pad, dtype=torch.float64):
    t = _colmajor(a.shape[0], a.shape[1], pad, dtype)
    t.copy_(a)
    return t


def _mixer(n, g):
    """An orthogonal n x n matrix: the cosine transform with its rows permuted and its rows and
    columns signed at random. Products of two of them around a diagonal have the entries and
    singular values of a randsvd matrix, without a QR of order n."""
    j = torch.arange(n, dtype=torch.float64, device="cuda")
    c = j[:, None] * (2.0 * j[None, :] + 1.0)
    c.remainder_(4.0 * n).mul_(math.pi / (2.0 * n)).cos_().mul_(math.sqrt(2.0 / n))
    c[0] *= math.sqrt(0.5)
    c = c[torch.randperm(n, device="cuda", generator=g)]
    signs = torch.randint(0, 2, (2, n), device="cuda", generator=g).to(torch.float64) * 2 - 1
    return c.mul_(signs[0][:, None]).mul_(signs[1][None, :])


def _sigma(n, kappa):
    """Singular values falling geometrically from 1 to 1/kappa."""
    return kappa ** (-torch.arange(n, dtype=torch.float64, device="cuda") / max(n - 1, 1))


def _general(n, nrhs, kappa, seed):
    """(A, B, X): a Gaussian system (kappa 0, X unknown) or one of condition kappa."""
    g = _gen(seed)
    b = _randn(g, n, nrhs)
    if kappa == 0.0:
        return _randn(g, n, n), b, None
    u, v = _mixer(n, g), _mixer(n, g)
    sig = _sigma(n, kappa)
    x = v.t() @ ((u @ b) / sig[:, None])
    a = u.t() @ v.mul_(sig[:, None])
    return a, b, x


def _hpd(n, nrhs, seed):
    """G G^T / n + I and its right-hand sides, G Gaussian."""
    g = _gen(seed)
    b = _randn(g, n, nrhs)
    m = _randn(g, n, n)
    a = m @ m.t() / n
    a.diagonal().add_(1.0)
    return a, b


def _hpd_batch(case, seed):
    """Sizes and widths (the batch's structure, a part of the case) and, from the seed, the flat
    FP64 matrices (column-major, one after another) and right-hand sides."""
    g = _gen(seed)
    rng = np.random.default_rng([case["count"], case["nmin"], case["nmax"]])
    ns = rng.integers(case["nmin"], case["nmax"] + 1, size=case["count"])
    ws = rng.integers(1, 9, size=case["count"])
    ao = np.concatenate([[0], np.cumsum(ns * ns)])
    bo = np.concatenate([[0], np.cumsum(ns * ws)])
    a = torch.empty(int(ao[-1]), dtype=torch.float64, device="cuda")
    b = _randn(g, int(bo[-1]))
    for n, idx in _by_order(ns):
        m = _randn(g, len(idx), n, n)
        p = torch.bmm(m, m.transpose(1, 2).contiguous()) / n
        p.diagonal(dim1=1, dim2=2).add_(1.0)
        for k, i in enumerate(idx):
            a[ao[i]:ao[i + 1]] = p[k].reshape(-1)
    return ns, ws, ao, bo, a, b


def _by_order(ns):
    order = np.argsort(ns, kind="stable")
    cuts = np.flatnonzero(np.diff(ns[order])) + 1
    return [(int(ns[part[0]]), part) for part in np.split(order, cuts)]


def _lu_batch(case, seed):
    """Lists A, B, X of systems of uneven order and condition (both a part of the case)."""
    rng = np.random.default_rng([case["count"], case["nmin"], case["nmax"]])
    out = []
    for i in range(case["count"]):
        n = int(round(math.exp(rng.uniform(math.log(case["nmin"]), math.log(case["nmax"])))))
        kappa = 10.0 ** rng.uniform(1, math.log10(case["kmax"]))
        out.append(_general(n, case["nrhs"], kappa, seed * 100003 + i))
    return [list(v) for v in zip(*out)]


def _flat(mats):
    """Column-major matrices one after another."""
    return torch.cat([t.t().reshape(-1) for t in mats])


# ------------------------------------------------------------------------ the timed calls
def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case, "kind": kind}
    if kind in ("solve", "lu", "mixed"):
        a, b, _ = _general(case["n"], case["nrhs"], case["kappa"], seed)
        pad = case.get("pad", 0)
        st["A"], st["B"] = _colmajor_of(a, pad), _colmajor_of(b, pad)
        st["X"] = _colmajor(case["n"], case["nrhs"], pad)
        if kind != "mixed":
            st["F"] = _colmajor(case["n"], case["n"], pad)
    elif kind in ("hpd", "hpd_mixed"):
        dtype = _DTYPE[case.get("dtype", "f64")]
        a, b = _hpd(case["n"], case["nrhs"], seed)
        pad = case.get("pad", 0)
        st["A"], st["B"] = _colmajor_of(a, pad, dtype), _colmajor_of(b, pad, dtype)
        st["X"] = _colmajor(case["n"], case["nrhs"], pad, dtype)
        if kind == "hpd":
            st["F"] = _colmajor(case["n"], case["n"], pad, dtype)
    elif kind == "batched_hpd":
        dtype = _DTYPE[case["dtype"]]
        ns, ws, ao, bo, a, b = _hpd_batch(case, seed)
        st["A"], st["B"] = a.to(dtype), b.to(dtype)
        st["F"], st["X"] = torch.empty_like(st["A"]), torch.empty_like(st["B"])
        mats = [st["F"][ao[i]:ao[i + 1]].view(int(n), int(n)).t() for i, n in enumerate(ns)]
        rhs = [st["X"][bo[i]:bo[i + 1]].view(int(ws[i]), int(n)).t() for i, n in enumerate(ns)]
        st["factors"], st["rhs"] = dev.Batch(mats, dtype), dev.Batch(rhs, dtype)
        if case["graph"]:
            st["graph"] = dev.PosvGraph(st["factors"], st["rhs"])
    elif kind == "batched_lu":
        a, b, x = _lu_batch(case, seed)
        st["A"] = [_colmajor_of(t, 0) for t in a]
        st["B"] = [_colmajor_of(t, 0) for t in b]
        # the solutions side by side in one buffer
        st["sol"] = torch.empty(sum(t.numel() for t in x), dtype=torch.float64, device="cuda")
        parts = st["sol"].split([t.numel() for t in x])
        st["X"] = [p.view(t.shape[1], t.shape[0]).t() for p, t in zip(parts, x)]
    else:
        a, b, _ = _general(case["n"], case["nrhs"], 0.0, seed)
        st["A"] = np.asfortranarray(a.cpu().numpy())
        st["B"] = np.asfortranarray(b.cpu().numpy())
        st["X"] = np.empty_like(st["B"], order="F")
        st["lib"] = elemental_amd.load()
        st["hA"], st["hX"] = _attach(st["lib"], st["A"]), _attach(st["lib"], st["X"])
    return st


def _attach(lib, a):
    """An ElMatrix_d handle over a Fortran-ordered numpy array."""
    h = ctypes.c_void_p()
    if lib.ElMatrixCreate_d(ctypes.byref(h)) != 0:
        raise RuntimeError("ElMatrixCreate_d failed")
    m, n = a.shape
    if lib.ElMatrixAttach_d(h, m, n, ctypes.c_void_p(a.ctypes.data), max(m, 1)) != 0:
        raise RuntimeError("ElMatrixAttach_d failed")
    return h


def run(state):
    case, kind = state["case"], state["kind"]
    if kind == "solve":
        state["F"].copy_(state["A"])
        state["X"].copy_(state["B"])
        info = dev.gesv(state["F"], state["X"])
        return state["X"], info
    if kind == "lu":
        state["F"].copy_(state["A"])
        state["X"].copy_(state["B"])
        dests, info = dev.getrf(state["F"])
        dev.getrs(state["F"], dests, state["X"], orient=case["orient"])
        return state["F"], state["X"], dests, info
    if kind == "hpd":
        state["F"].copy_(state["A"])
        state["X"].copy_(state["B"])
        info = dev.posv(state["F"], state["X"], uplo=case["uplo"])
        return state["F"], state["X"], info
    if kind == "mixed":
        dev.gesv_mixed(state["A"], state["B"], state["X"], factor=case["factor"])
        return state["X"]
    if kind == "hpd_mixed":
        dev.posv_mixed(state["A"], state["B"], state["X"], factor=case["factor"])
        return state["X"]
    if kind == "batched_hpd":
        state["F"].copy_(state["A"])
        state["X"].copy_(state["B"])
        if case["graph"]:
            info = state["graph"].launch()
        else:
            info = dev.potrf_vbatched(state["factors"])
            dev.potrs_vbatched(state["factors"], state["rhs"])
        return state["F"], state["X"], info
    if kind == "batched_lu":
        dev.gesv_mixed_batched(state["A"], state["B"], state["X"])
        return state["sol"]
    state["X"][...] = state["B"]
    if state["lib"].ElLinearSolve_d(state["hA"], state["hX"]) != 0:
        raise RuntimeError("ElLinearSolve_d failed")
    return state["X"]


# ------------------------------------------------------------- bytes, flops and references
def work(case):
    kind = case["kind"]
    if kind == "batched_hpd":
        # expectations over the uniform sizes, 4.5 right-hand sides on average
        n = np.arange(case["nmin"], case["nmax"] + 1, dtype=np.float64)
        c, size = float(case["count"]), 8.0 if case["dtype"] == "f64" else 4.0
        return {"bytes": c * size * float(np.mean(1.5 * n * n + 2 * 4.5 * n)),
                "flops": c * float(np.mean(n ** 3 / 3.0 + 2.0 * 4.5 * n * n))}
    if kind == "batched_lu":
        # expectations over orders uniform in their logarithm
        lo, hi = float(case["nmin"]), float(case["nmax"])
        span, c, w = math.log(hi / lo), float(case["count"]), case["nrhs"]
        n1, n2, n3 = (hi - lo) / span, (hi ** 2 - lo ** 2) / (2 * span), (hi ** 3 - lo ** 3) / (3 * span)
        return {"bytes": c * 8.0 * (n2 + 2 * w * n1),
                "flops": c * (2.0 / 3.0 * n3 + 2.0 * w * n2)}
    n, w = float(case["n"]), float(case["nrhs"])
    size = 4.0 if case.get("dtype") == "f32" else 8.0
    if kind in ("hpd", "hpd_mixed"):
        out = 0.5 * n * n if kind == "hpd" else 0.0
        return {"bytes": size * (0.5 * n * n + out + 2 * n * w),
                "flops": n ** 3 / 3.0 + 2.0 * w * n * n}
    out = n * n if kind == "lu" else 0.0
    return {"bytes": size * (n * n + out + 2 * n * w),
            "flops": 2.0 / 3.0 * n ** 3 + 2.0 * w * n * n}


def exact(case, seed):
    kind = case["kind"]
    if kind == "batched_lu":
        return _flat(_lu_batch(case, seed)[2])
    if kind == "batched_hpd":
        ns, ws, ao, bo, a, b = _hpd_batch(case, seed)
        dtype = _DTYPE[case["dtype"]]
        a, b = a.to(dtype).to(torch.float64), b.to(dtype).to(torch.float64)
        f, x = a.clone(), torch.empty_like(b)
        for n, idx in _by_order(ns):
            m = torch.stack([a[ao[i]:ao[i + 1]].view(n, n) for i in idx])
            r = torch.zeros(len(idx), n, 8, dtype=torch.float64, device="cuda")
            for k, i in enumerate(idx):
                r[k, :, :int(ws[i])] = b[bo[i]:bo[i + 1]].view(int(ws[i]), n).t()
            # the row-major storage read as given: its transpose is the column-major matrix
            l = torch.linalg.cholesky(m.transpose(1, 2).contiguous())
            s = torch.cholesky_solve(r, l)
            for k, i in enumerate(idx):
                lower = torch.tril(l[k]) + torch.triu(m[k].t(), 1)
                f[ao[i]:ao[i + 1]] = lower.t().reshape(-1)
                x[bo[i]:bo[i + 1]] = s[k, :, :int(ws[i])].t().reshape(-1)
        return f, x, None
    n = case["n"]
    if kind == "mixed":
        return _general(n, case["nrhs"], case["kappa"], seed)[2]
    if kind == "solve" and case["kappa"] != 0.0:
        return _general(n, case["nrhs"], case["kappa"], seed)[2], None
    if n > _EXACT_ORDER:
        return None
    if kind in ("hpd", "hpd_mixed"):
        dtype = _DTYPE[case.get("dtype", "f64")]
        a, b = _hpd(n, case["nrhs"], seed)
        a, b = a.to(dtype).to(torch.float64).cpu(), b.to(dtype).to(torch.float64).cpu()
        upper = bool(case.get("uplo", 0))
        # the factorization reads one triangle; mirror it for the reference
        t = torch.triu(a) if upper else torch.tril(a)
        sym = t + t.t() - torch.diag(torch.diagonal(a))
        l = torch.linalg.cholesky(sym)
        x = torch.cholesky_solve(b, l)
        if kind == "hpd_mixed":
            return x
        f = l.t() + torch.tril(a, -1) if upper else l + torch.triu(a, 1)
        return f, x, None
    a, b, _ = _general(n, case["nrhs"], case.get("kappa", 0.0), seed)
    a, b = a.cpu(), b.cpu()
    if kind == "lu":
        f, piv = torch.linalg.lu_factor(a)
        x = torch.linalg.lu_solve(f, piv, b, adjoint=bool(case["orient"]))
        return f, x, None, None
    x = torch.linalg.solve(a, b)
    return (x, None) if kind == "solve" else x.numpy()
