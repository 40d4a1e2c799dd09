"""Performance cases of the Cholesky path: the calls that programs make of it.

A case is a dict of plain values.  `listed()` gives the fixed cases, `draw`
one more of the same ranges; `prepare` makes what a program holds before the
call (inputs on the GPU, the handle, the descriptors, the tuned batch
schedule), `run` is one pass through the public entry points, `work` the
bytes and operations that the pass cannot do without, and `exact` the result
in 64 bits from plain torch.

Kinds:
    posv      A X = B from scratch (pposv): one SPD / Hermitian system
    potrf     a factorization alone (ppotrf), for a program that keeps the factor
    potrs     solves with a kept factor (ppotrs)
    mixed     pposv_mixed: FP32 or split-product factor, FP64 refinement
    vbatched  many small systems of uneven order in one call (pposv_vbatched)
    gp        Gaussian-process likelihoods with their gradients, all problems in one call
    grad      Cholesky, solve and log-determinant composed under torch.autograd

The routines work in place, so a pass that must be repeatable copies its
inputs into the working buffers first, as a program does that still needs A.
"""
import math

import numpy as np
import torch

import libddla_amd as dd
from libddla_amd import autograd as ag

DEVICE = "cuda"
TORCH = {"s": torch.float32, "d": torch.float64, "c": torch.complex64, "z": torch.complex128}
NUMPY = {"s": np.float32, "d": np.float64, "c": np.complex64, "z": np.complex128}
ITEM = {"s": 4, "d": 8, "c": 8, "z": 16}

_HANDLE = []


def handle():
    """The program's one handle, on torch's current stream."""
    if not _HANDLE:
        _HANDLE.append(dd.Handle(dd.Backend.GPU))
        _HANDLE[0].set_stream(torch.cuda.current_stream().cuda_stream)
    return _HANDLE[0]


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: one right-hand side of a filter or a Newton step, where launches and the return count
        {"name": "posv_d_96", "kind": "posv", "type": "d", "n": 96, "nrhs": 1, "uplo": "L", "pad": 0, "delta": 1.0},
        # an ordinary system: the order and right-hand sides of the reference's own CPU-handle case
        {"name": "posv_d_2048", "kind": "posv", "type": "d", "n": 2048, "nrhs": 16, "uplo": "L", "pad": 0,
         "delta": 1.0},
        # the largest: the benchmark's headline system
        {"name": "posv_d_32768", "kind": "posv", "type": "d", "n": 32768, "nrhs": 64, "uplo": "L", "pad": 0,
         "delta": 0.1},
        # a complex Hermitian system of an odd order (electronic-structure and antenna-array programs)
        {"name": "posv_z_1999", "kind": "posv", "type": "z", "n": 1999, "nrhs": 16, "uplo": "L", "pad": 0,
         "delta": 1.0},
        # FP32 factor of an odd order, upper triangle, inside a larger parent matrix
        {"name": "potrf_s_7001_upper", "kind": "potrf", "type": "s", "n": 7001, "uplo": "U", "pad": 23,
         "delta": 1.0},
        # FP32 complex factor, kept for later solves
        {"name": "potrf_c_4500", "kind": "potrf", "type": "c", "n": 4500, "uplo": "L", "pad": 0, "delta": 1.0},
        # repeated solves with a kept factor
        {"name": "potrs_d_8192", "kind": "potrs", "type": "d", "n": 8192, "nrhs": 64, "uplo": "L", "side": "L",
         "delta": 0.1},
        # mixed precision at the benchmark's middle size: split half-precision updates, FP64 refinement
        {"name": "mixed_fp16x3_16384", "kind": "mixed", "factor": 3, "n": 16384, "nrhs": 64, "uplo": "L",
         "delta": 4e-2},
        # the benchmark's batch: 4096 systems of orders 32 to 512, FP64
        {"name": "vbatched_d_4096", "kind": "vbatched", "type": "d", "batch": 4096, "lo": 32, "hi": 512,
         "orders": 3, "nrhs": 1},
        # a smaller FP32 batch of smaller systems
        {"name": "vbatched_s_1500", "kind": "vbatched", "type": "s", "batch": 1500, "lo": 20, "hi": 300,
         "orders": 5, "nrhs": 1},
        # the benchmark's Gaussian-process fit: 16 likelihoods and their gradients
        {"name": "gp_16x4096", "kind": "gp", "batch": 16, "n": 4096},
        # a differentiable solve and log-determinant in a training step
        {"name": "grad_d_1500", "kind": "grad", "n": 1500, "nrhs": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["posv", "posv", "posv", "potrf", "potrf", "potrs", "mixed", "vbatched", "vbatched", "gp",
                       "grad"])
    if kind in ("posv", "potrf"):
        t = rng.choice(["d", "d", "d", "s", "z", "c"])
        case = {"kind": kind, "type": t, "n": _log_int(rng, 64, 12000 if t in "sd" else 4500),
                "uplo": rng.choice("LLU"), "pad": rng.choice([0, 0, 1, 23]), "delta": rng.choice([0.1, 1.0])
                if t in "dz" else 1.0}
        if kind == "posv":
            case["nrhs"] = _log_int(rng, 1, 128)
        return case
    if kind == "potrs":
        return {"kind": kind, "type": rng.choice("dds"), "n": _log_int(rng, 128, 12000),
                "nrhs": _log_int(rng, 1, 600), "uplo": rng.choice("LLU"), "side": rng.choice("LLR"), "delta": 1.0}
    if kind == "mixed":
        return {"kind": kind, "factor": rng.randrange(4), "n": _log_int(rng, 2048, 16384),
                "nrhs": _log_int(rng, 1, 64), "uplo": "L", "delta": rng.choice([4e-2, 4e-4])}
    if kind == "vbatched":
        lo, hi = rng.choice([(8, 64), (20, 300), (32, 512), (100, 400)])
        return {"kind": kind, "type": rng.choice("ds"), "batch": _log_int(rng, 200, 4096), "lo": lo, "hi": hi,
                "orders": rng.randrange(1 << 30), "nrhs": rng.choice([1, 1, 3])}
    if kind == "gp":
        return {"kind": kind, "batch": rng.randint(2, 16), "n": _log_int(rng, 200, 4096)}
    return {"kind": kind, "n": _log_int(rng, 200, 3000), "nrhs": _log_int(rng, 1, 32)}


# ---------------------------------------------------------------------------
# Inputs (torch alone, from the seed)
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _spd(n, ld, t, delta, gen):
    """Storage (n, ld) of the column-major A = G G^H / n + delta I, G of normals; a copied matrix, padding zero."""
    dtype = TORCH[t]
    g = torch.randn(n, n, dtype=dtype, device=DEVICE, generator=gen)
    m = torch.mm(g, g.mH.contiguous() if t in "cz" else g.t())
    del g
    m.div_(n)
    m.diagonal().add_(delta)
    if t in "cz":
        m.diagonal().imag.zero_()
    if ld == n:
        return m.t().contiguous() if t in "cz" else m
    a = torch.zeros(n, ld, dtype=dtype, device=DEVICE)
    a[:, :n] = m.t()
    return a


def _dense(case, seed):
    """(A, B) of a posv / potrf / potrs / mixed case; B's storage is (columns, rows)."""
    gen = _generator(seed)
    n, t = case["n"], case.get("type", "d")
    a = _spd(n, n + case.get("pad", 0), t, case["delta"], gen)
    if "nrhs" not in case:
        return a, None
    rows, cols = (n, case["nrhs"]) if case.get("side", "L") == "L" else (case["nrhs"], n)
    return a, torch.randn(cols, rows, dtype=TORCH[t], device=DEVICE, generator=gen)


def _factor_storage(a, n, uplo):
    """Storage of the factor in the triangle uplo of `a` (its other triangle and padding kept), by torch."""
    m = a[:, :n].t()  # M(i, j) = a[j, i]
    if uplo == "U":
        m = m.mH  # the stored triangle as a lower one, which is the one that torch reads
    wide = m.to(torch.complex128 if a.is_complex() else torch.float64)
    low = torch.linalg.cholesky(wide.contiguous())
    out = a.to(wide.dtype)
    out[:, :n] = (torch.triu(low.t()) + torch.tril(out[:, :n], -1) if uplo == "L"
                  else torch.tril(low.conj()) + torch.triu(out[:, :n], 1))
    return out, low


def _orders(case):
    """The members' orders: uniform, and the case's own (a batch has the same shape for every seed)."""
    return np.random.RandomState(case["orders"]).randint(case["lo"], case["hi"] + 1, size=case["batch"])


def _batch_inputs(case, seed):
    """(orders, A arena, B arena): the members one after another, column-major, leading dimension n_i."""
    gen = _generator(seed)
    sizes = _orders(case)
    dtype, nrhs = TORCH[case["type"]], case["nrhs"]
    a = torch.empty(int((sizes.astype(np.int64) ** 2).sum()), dtype=dtype, device=DEVICE)
    b = torch.randn(int(sizes.sum()) * nrhs, dtype=dtype, device=DEVICE, generator=gen)
    at = 0
    for n in sizes.tolist():
        g = torch.randn(n, n, dtype=dtype, device=DEVICE, generator=gen)
        m = a[at:at + n * n].view(n, n)
        torch.mm(g, g.t(), out=m)
        m.div_(n)
        m.diagonal().add_(0.5)
        at += n * n
    return sizes, a, b


class _Arena:
    """Device memory of a VBatch as an array (keeps the VBatch alive)."""

    def __init__(self, vb, ptr, count, typestr):
        self.vb = vb
        self.__cuda_array_interface__ = {"shape": (int(count),), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}


def _arena(vb, device, count, dtype):
    return torch.as_tensor(_Arena(vb, device.ptr.value, count, np.dtype(dtype).str), device=DEVICE)


def _gp_inputs(case, seed):
    """RBF kernels of points uniform in the unit cube (l = 0.2, s = 1, jitter 1e-2) and normal targets."""
    gen = _generator(seed)
    batch, n = case["batch"], case["n"]
    k = torch.empty(batch, n, n, dtype=torch.float64, device=DEVICE)
    for b in range(batch):
        x = torch.rand(n, 3, dtype=torch.float64, device=DEVICE, generator=gen)
        sq = x.square().sum(1)
        d2 = (sq[:, None] + sq[None, :] - 2.0 * torch.mm(x, x.t())).clamp_min_(0.0)
        d2 = 0.5 * (d2 + d2.t())
        k[b] = torch.exp(d2 / (-2.0 * 0.2 ** 2))
        k[b].diagonal().add_(1e-2)
    return k, torch.randn(batch, n, dtype=torch.float64, device=DEVICE, generator=gen)


def _grad_inputs(case, seed):
    gen = _generator(seed)
    a = _spd(case["n"], case["n"], "d", 1.0, gen)
    a = 0.5 * (a + a.t())
    b = torch.randn(case["n"], case["nrhs"], dtype=torch.float64, device=DEVICE, generator=gen)
    w = torch.randn(case["n"], case["nrhs"], dtype=torch.float64, device=DEVICE, generator=gen)
    return a, b, w


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def _wrap(h, storage, rows, cols):
    return dd.DistributedMatrix.from_torch(h, storage, rows, cols, 512, 512)


def prepare(case, seed):
    h = handle()
    kind = case["kind"]
    s = {"kind": kind, "h": h, "case": case}
    if kind in ("posv", "potrf", "potrs", "mixed"):
        n = case["n"]
        s["a0"], s["b0"] = _dense(case, seed)
        s["a"] = s["a0"].clone()
        s["A"] = _wrap(h, s["a"], n, n)
        if s["b0"] is not None:
            s["b"] = s["b0"].clone()
            cols, rows = s["b"].shape
            s["B"] = _wrap(h, s["b"], rows, cols)
        if kind == "potrs":  # the kept factor
            _, info = dd.ppotrf(s["A"], case["uplo"])
            assert info == 0
            del s["a0"]
    elif kind == "vbatched":
        sizes, s["a0"], s["b0"] = _batch_inputs(case, seed)
        vb = dd.VBatch(h, sizes, nrhs=case["nrhs"], dtype=NUMPY[case["type"]])
        s["vb"] = vb
        s["a"] = _arena(vb, vb.A, s["a0"].numel(), vb.dtype)
        s["b"] = _arena(vb, vb.B, s["b0"].numel(), vb.dtype)
        s["info"] = _arena(vb, vb.info, vb.batch, np.int32)
        s["logdet"] = _arena(vb, vb.logdet, vb.batch, np.float64)
        s["a"].copy_(s["a0"])
        s["b"].copy_(s["b0"])
        dd.pposv_vbatched_tune(vb, "L")  # times the schedules on copies of this batch
    elif kind == "gp":
        k, y = _gp_inputs(case, seed)
        s["k"], s["y"] = k.requires_grad_(True), y.requires_grad_(True)
    else:
        a, b, s["w"] = _grad_inputs(case, seed)
        s["a"], s["b"] = a.requires_grad_(True), b.requires_grad_(True)
    return s


def run(s):
    kind, case, h = s["kind"], s["case"], s["h"]
    if kind == "posv":
        s["a"].copy_(s["a0"])
        s["b"].copy_(s["b0"])
        _, info = dd.pposv(s["A"], s["B"], case["uplo"])
        return {"factor": s["a"], "x": s["b"], "info": info}
    if kind == "potrf":
        s["a"].copy_(s["a0"])
        _, info = dd.ppotrf(s["A"], case["uplo"])
        return {"factor": s["a"], "info": info}
    if kind == "potrs":
        s["b"].copy_(s["b0"])
        dd.ppotrs(s["A"], s["B"], case["uplo"], case["side"])
        return {"x": s["b"]}
    if kind == "mixed":
        s["a"].copy_(s["a0"])
        s["b"].copy_(s["b0"])
        _, _, info = dd.pposv_mixed(s["A"], s["B"], case["uplo"], factor=case["factor"], tol=1e-14, max_iter=30)
        return {"x": s["b"], "info": info}
    if kind == "vbatched":
        s["a"].copy_(s["a0"])
        s["b"].copy_(s["b0"])
        dd.pposv_vbatched(s["vb"], "L")
        return {"factors": s["a"], "x": s["b"], "logdet": s["logdet"], "info": s["info"]}
    if kind == "gp":
        loss = ag.gp_negative_log_likelihood_batched(s["k"], s["y"], h)
        dk, dy = torch.autograd.grad(loss.sum(), (s["k"], s["y"]))
        return {"loss": loss.detach(), "dk": dk, "dy": dy}
    low = ag.cholesky(s["a"], h)
    x = ag.cholesky_solve(s["b"], low, h)
    loss = (s["w"] * x).sum() + ag.cholesky_logdet(low, h)
    da, db = torch.autograd.grad(loss, (s["a"], s["b"]))
    return {"loss": loss.detach(), "x": x.detach(), "da": da, "db": db}


# ---------------------------------------------------------------------------
# work and exact
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "vbatched":
        n = _orders(case).astype(np.float64)
        es, m = ITEM[case["type"]], case["batch"]
        return {"bytes": float(m * es * (np.mean(n * (n + 1)) + 2 * case["nrhs"] * np.mean(n))),
                "flops": float(m * np.mean(n ** 3 / 3 + 2 * n ** 2 * case["nrhs"]))}
    n = float(case["n"])
    if kind == "gp":
        # factor, inverse (n^3/3 each to L^-1 and to K^-1); K read, dK written
        return {"bytes": case["batch"] * 8 * (n * (n + 1) / 2 + n * n + 2 * n), "flops": case["batch"] * n ** 3}
    nrhs = case.get("nrhs", 0)
    if kind == "grad":
        # factor n^3/3; its adjoint L^-T Phi(L^T Lbar) L^-1 with the triangles used: n^3; the solves 8 n^2 nrhs
        return {"bytes": 8 * (n * (n + 1) / 2 + n * n + 4 * n * nrhs), "flops": 4 * n ** 3 / 3 + 8 * n * n * nrhs}
    t = case.get("type", "d")
    mult, es = (4 if t in "cz" else 1), ITEM[t]
    tri, b = es * n * (n + 1) / 2, 2 * es * n * nrhs
    if kind == "potrs":
        return {"bytes": tri + b, "flops": mult * 2 * n * n * nrhs}
    if kind == "mixed":
        return {"bytes": tri + b, "flops": n ** 3 / 3 + 2 * n * n * nrhs}
    return {"bytes": 2 * tri + b, "flops": mult * (n ** 3 / 3 + 2 * n * n * nrhs)}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("posv", "potrf", "potrs", "mixed"):
        n = case["n"]
        a, b = _dense(case, seed)
        out, low = _factor_storage(a, n, case["uplo"])
        del a
        x = None
        if b is not None:
            wide = b.to(low.dtype)
            # storage (columns, rows): side L solves A X = B with X = wide^T, side R X A = B, A Hermitian
            rhs = wide.t() if case.get("side", "L") == "L" else wide
            y = torch.linalg.solve_triangular(low, rhs, upper=False)
            y = torch.linalg.solve_triangular(low.mH, y, upper=True)
            x = (y.t() if case.get("side", "L") == "L" else y).contiguous()
        if kind == "posv":
            return {"factor": out, "x": x, "info": None}
        if kind == "potrf":
            return {"factor": out, "info": None}
        return {"x": x} if kind == "potrs" else {"x": x, "info": None}
    if kind == "vbatched":
        sizes, a, b = _batch_inputs(case, seed)
        a, b, nrhs = a.cpu().double().numpy(), b.cpu().double().numpy(), case["nrhs"]
        logdet, at, bt = np.empty(len(sizes)), 0, 0
        for i, n in enumerate(sizes.tolist()):
            m = a[at:at + n * n].reshape(n, n)  # m[j, i] = A(i, j)
            low = np.linalg.cholesky(np.triu(m).T + np.triu(m, 1))
            y = b[bt:bt + n * nrhs].reshape(nrhs, n)
            y[:] = np.linalg.solve(low.T, np.linalg.solve(low, y.T)).T
            m[:] = np.triu(low.T) + np.tril(m, -1)
            logdet[i] = 2.0 * np.log(np.diagonal(low)).sum()
            at, bt = at + n * n, bt + n * nrhs
        return {"factors": a, "x": b, "logdet": logdet, "info": None}
    if kind == "gp":
        k, y = _gp_inputs(case, seed)
        loss, dk, dy = torch.empty(len(k), dtype=k.dtype, device=DEVICE), torch.empty_like(k), torch.empty_like(y)
        for b in range(len(k)):
            low = torch.linalg.cholesky(k[b])
            alpha = torch.cholesky_solve(y[b][:, None], low)
            loss[b] = 0.5 * (y[b] @ alpha[:, 0]) + low.diagonal().log().sum()
            dk[b] = 0.5 * (torch.cholesky_inverse(low) - alpha @ alpha.t())
            dy[b] = alpha[:, 0]
        return {"loss": loss, "dk": dk, "dy": dy}
    a, b, w = _grad_inputs(case, seed)
    inv = torch.linalg.inv(a)
    inv = 0.5 * (inv + inv.t())
    x, db = inv @ b, inv @ w
    outer = db @ x.t()
    return {"loss": (w * x).sum() + torch.linalg.slogdet(a)[1], "x": x, "da": inv - 0.5 * (outer + outer.t()),
            "db": db}
