"""Factorizations and solves at the edges of their blocks: orders around the
64-row blocks and the largest one-panel orders (4096; complex128 3840), the same matrix by narrow
panels, complex elements, and the 128-row solve sweeps over orders, right-hand
sides, triangles and sides.

Checked against the problem itself, in float64 on the GPU, row by row of the factor
and column by column of the solution, so that a lost row, block or column shows
whatever the order: max over rows of |A - L L^H| and over columns of |B - A X| / |X|
in infinity norms within 0.05 n eps |A| (n >= 64), the suite's bound.  A
backward-stable factorization or solve of a well-conditioned system (every spectrum
lies in [0.5, 4.6]) is off by a few eps there."""
import numpy as np
import pytest

import libddla_amd as dd

pytestmark = pytest.mark.gpu

TORCH = {np.float64: "float64", np.float32: "float32", np.complex128: "complex128", np.complex64: "complex64"}


def system(n, dtype, seed):
    """Hermitian positive definite A in float64 / complex128 (rounded to dtype) on the GPU."""
    import torch

    gen = torch.Generator(device="cuda").manual_seed(seed)
    wide = torch.complex128 if np.dtype(dtype).kind == "c" else torch.float64
    g = torch.randn(n, n, dtype=wide, device="cuda", generator=gen)
    a = torch.mm(g, g.mH.contiguous()) / n
    a = (0.5 * (a + a.mH)).contiguous()
    a.diagonal().add_(0.5)
    return a.to(getattr(torch, TORCH[dtype])).to(wide), gen


def factor(handle, a, dtype, uplo):
    import torch

    s = a.t().to(getattr(torch, TORCH[dtype])).clone(memory_format=torch.contiguous_format)  # column-major storage
    torch.cuda.synchronize()
    A = dd.DistributedMatrix.from_torch(handle, s, a.shape[0], a.shape[0])
    assert dd.ppotrf(A, uplo)[1] == 0
    return A, s


def residual(a, s, uplo):
    """max over rows of |A - L L^H| / |A| in infinity norms."""
    import torch

    m = s.t().to(a.dtype)
    low = m.tril() if uplo == "L" else m.triu().mH
    r = (a - torch.mm(low, low.mH.contiguous())).abs().sum(1).max()
    return (r / a.abs().sum(1).max()).item()


def column_error(a, x, b):
    """max over columns of |b - a x| / (|a| |x|) in infinity norms, float64 / complex128 on the GPU."""
    import torch

    r = (b - torch.mm(a, x)).abs().amax(0)
    return (r / (a.abs().sum(1).max() * x.abs().amax(0))).max().item()


def bound(n, dtype):
    return 0.05 * max(n, 64) * np.finfo(dtype).eps


@pytest.mark.parametrize("dtype,n", [(np.float64, n) for n in (65, 128, 191, 1000, 4032, 4096, 4160)] +
                         [(np.float32, n) for n in (129, 1500, 4095, 4097)] +
                         [(np.complex128, n) for n in (1, 63, 65, 200, 1025, 3840, 3841)] +
                         [(np.complex64, n) for n in (64, 130, 1500, 4161)])
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_factor_units(handle, dtype, n, uplo):
    print(f"case units n={n} {np.dtype(dtype).name} {uplo}", flush=True)
    a, _ = system(n, dtype, n)
    tol = bound(n, dtype)
    A, s = factor(handle, a, dtype, uplo)
    assert residual(a, s, uplo) <= tol
    if n > 192:  # several panels with rows below them, updates between them
        previous = dd.lib.ddla_c_set_panel_width(192)
        try:
            _, s2 = factor(handle, a, dtype, uplo)
        finally:
            dd.lib.ddla_c_set_panel_width(previous)
        assert residual(a, s2, uplo) <= tol


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (129, 17), (447, 3), (448, 1), (513, 16), (639, 33), (640, 15), (641, 17),
                                    (767, 64), (1000, 255)])
@pytest.mark.parametrize("uplo,side", [("L", "L"), ("U", "L"), ("L", "R")])
def test_solve_sweeps(handle, dtype, n, nrhs, uplo, side):
    import torch

    print(f"case sweeps n={n} nrhs={nrhs} {np.dtype(dtype).name} {uplo} {side}", flush=True)
    a, gen = system(n, dtype, 7 * n + nrhs)
    A, _ = factor(handle, a, dtype, uplo)
    rows, cols = (n, nrhs) if side == "L" else (nrhs, n)
    pad = 5  # rows of B's parent that stay as they are
    full = torch.randn(cols, rows + pad, dtype=a.dtype, device="cuda", generator=gen)
    b = full.to(getattr(torch, TORCH[dtype])).clone()
    keep = b.clone()
    torch.cuda.synchronize()
    B = dd.DistributedMatrix.from_torch(handle, b, rows, cols)
    dd.ppotrs(A, B, uplo, side)
    x, b0 = b[:, :rows].t().to(a.dtype).contiguous(), keep[:, :rows].t().to(a.dtype).contiguous()
    if side == "R":  # X A = B  is  A X^H = B^H
        x, b0 = x.mH.contiguous(), b0.mH.contiguous()
    assert column_error(a, x, b0) <= bound(n, dtype)
    assert torch.equal(b[:, rows:], keep[:, rows:])


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n,nrhs", [(3, 1048577), (129, 6416), (129, 11008), (700, 3000)])
@pytest.mark.parametrize("uplo,side", [("L", "L"), ("U", "L"), ("L", "R"), ("U", "R")])
def test_complex_solves_with_many_columns(handle, dtype, n, nrhs, uplo, side):
    """On both sides of the change from sweeps to products, and more columns than one launch's grid
    takes in its second dimension.  Column by column, within the suite's 0.05 n eps (n >= 64)."""
    import torch

    print(f"case many columns n={n} nrhs={nrhs} {np.dtype(dtype).name} {uplo} {side}", flush=True)
    a, gen = system(n, dtype, 5 * n)
    A, _ = factor(handle, a, dtype, uplo)
    rows, cols = (n, nrhs) if side == "L" else (nrhs, n)
    b0 = torch.randn(cols, rows, dtype=a.dtype, device="cuda", generator=gen).to(getattr(torch, TORCH[dtype]))
    b = b0.clone()
    torch.cuda.synchronize()
    B = dd.DistributedMatrix.from_torch(handle, b, rows, cols)
    dd.ppotrs(A, B, uplo, side)
    x, c = b.t().to(a.dtype).contiguous(), b0.t().to(a.dtype).contiguous()
    if side == "R":  # X A = C  is  A X^H = C^H
        x, c = x.mH.contiguous(), c.mH.contiguous()
    assert column_error(a, x, c) <= bound(n, dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,nrhs,uplo", [(512, 1500, "L"), (800, 4700, "L"), (640, 816, "L"), (640, 817, "L"), (1024, 513, "L"),
                                         (640, 64, "U"), (700, 63, "U"), (768, 1, "U"), (895, 2, "U"), (896, 2, "U"),
                                         (1024, 512, "U"), (1024, 528, "U")])
def test_solve_routes(handle, dtype, n, nrhs, uplo):
    """Both sides of each line between the 64-row and the 128-row sweeps; column by column."""
    import torch

    print(f"case routes n={n} nrhs={nrhs} {np.dtype(dtype).name} {uplo}", flush=True)
    a, gen = system(n, dtype, 3 * n + nrhs)
    A, _ = factor(handle, a, dtype, uplo)
    b0 = torch.randn(nrhs, n, dtype=a.dtype, device="cuda", generator=gen).to(getattr(torch, TORCH[dtype]))
    b = b0.clone()
    torch.cuda.synchronize()
    dd.ppotrs(A, dd.DistributedMatrix.from_torch(handle, b, n, nrhs), uplo)
    x, c = b.t().to(a.dtype).contiguous(), b0.t().to(a.dtype).contiguous()
    assert column_error(a, x, c) <= bound(n, dtype)


@pytest.mark.parametrize("dtype,jitter", [(np.float64, 1e-6), (np.float32, 1e-3)])
@pytest.mark.parametrize("n", [700, 1000])
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_solves_with_ill_conditioned_blocks(handle, dtype, jitter, n, uplo):
    """A smooth kernel matrix with pairs of points 64 rows apart that nearly coincide: condition about n /
    jitter, in its 128 x 128 diagonal blocks too, which the solve inverts.  Backward stable all the same."""
    import torch

    print(f"case ill-conditioned n={n} {np.dtype(dtype).name} {uplo}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.rand(n, 3, dtype=torch.float64, device="cuda", generator=gen)
    i = torch.arange(0, n - 64, device="cuda")
    i = i[i % 128 < 64]
    x[i + 64] = x[i] + 1e-7
    d2 = (x[:, None] - x[None]).square().sum(-1)
    a = torch.exp(-d2 / (2 * 0.2 ** 2))
    a.diagonal().add_(jitter)
    a = a.to(getattr(torch, TORCH[dtype])).double()
    A, s = factor(handle, a, dtype, uplo)
    assert residual(a, s, uplo) <= bound(n, dtype)
    for nrhs in (1, 70):
        b0 = torch.randn(nrhs, n, dtype=a.dtype, device="cuda", generator=gen).to(getattr(torch, TORCH[dtype]))
        b = b0.clone()
        torch.cuda.synchronize()
        dd.ppotrs(A, dd.DistributedMatrix.from_torch(handle, b, n, nrhs), uplo)
        assert column_error(a, b.t().double().contiguous(), b0.t().double().contiguous()) <= bound(n, dtype)
