"""The 64 x 64 diagonal block's factorization (four columns a step, 16-column
strips): orders at the edges of steps, strips and blocks, and a failed pivot in
each place of a step, against the oracle; blocks with pivots down to rounding.

Tolerance of the first: backward-stable Cholesky of order n has |L - L_ref| <= c n eps
cond(A) |L|; the matrices have cond(A) < 10 (spectrum in [0.5, 4.6]), so 4 n eps
cond covers both factors."""
import numpy as np
import pytest

import libddla_amd as dd
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [3, 4, 5, 15, 16, 17, 32, 33, 47, 49, 63, 64, 65, 127])
def test_factor_and_failed_pivots(handle, dtype, n):
    print(f"case diag block n={n} {np.dtype(dtype).name}", flush=True)
    a = orc.spd_matrix(n, seed=7, delta=0.5).astype(dtype)
    ref, info = orc.potrf("L", a)
    assert info == 0
    tol = 4 * n * np.finfo(dtype).eps * 10
    poisoned = np.where(np.tril(np.ones((n, n), bool)), a, np.nan).astype(dtype)
    A = dd.DistributedMatrix.from_global_matrix(handle, poisoned)
    assert dd.ppotrf(A, "L")[1] == 0
    got = np.tril(A.to_global_matrix())
    assert np.linalg.norm(got - np.tril(ref)) <= tol * np.linalg.norm(np.tril(ref))
    # a pivot that is not positive (or is NaN) in column p: its 1-based index, the columns before it intact
    for p, value in ((0, -1.0), (n // 2, np.nan), (n - 2, 0.0), (n - 1, -2.0)):
        bad = poisoned.copy()
        bad[p, p] = value if p else -1.0
        A = dd.DistributedMatrix.from_global_matrix(handle, bad)
        assert dd.ppotrf(A, "L")[1] == p + 1
        got = A.to_global_matrix()[:p, :p]
        want = np.tril(ref)[:p, :p]
        assert np.linalg.norm(np.tril(got) - want) <= tol * max(1.0, np.linalg.norm(want))


def nearly_singular(dtype, n, rank, shift, rng):
    """G G^H of n x rank normals, its diagonal raised by `shift` eps of itself: pivots from eps^2 up."""
    g = rng.standard_normal((n, rank))
    if np.dtype(dtype).kind == "c":
        g = g + 1j * rng.standard_normal((n, rank))
    a = g @ g.conj().T
    a[np.arange(n), np.arange(n)] *= 1 + shift * np.finfo(dtype).eps
    return a.astype(dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
def test_nearly_singular_blocks(handle, dtype):
    """Within a block the columns are found by substitution, so that the factorization
    is backward stable element by element however small a pivot is: |A - L L^H|(i, j)
    <= c eps sqrt(a_ii a_jj), c = n + 1 for real products summed in any order (Higham,
    Accuracy and Stability, th. 10.3), two more per element for the reciprocal square
    root and its multiplication, doubled for complex products.  And a factor that is
    reported complete has positive pivots on its diagonal."""
    print(f"case nearly singular {np.dtype(dtype).name}", flush=True)
    rng = np.random.RandomState(11)
    wide = np.clongdouble if np.dtype(dtype).kind == "c" else np.longdouble
    complete = 0
    for trial in range(600):
        n = rng.randint(2, 20 if trial < 500 else 65)  # small ones: a pivot is tiny beside a large one more often
        a = nearly_singular(dtype, n, rng.randint(1, n + 1), rng.choice([0, 0.5, 1, 2, 8, 100, 1e4]), rng)
        A = dd.DistributedMatrix.from_global_matrix(handle, a)
        if dd.ppotrf(A, "L")[1] != 0:
            continue
        complete += 1
        low = np.tril(A.to_global_matrix()).astype(wide)
        assert (np.diagonal(low).real > 0).all(), trial
        diag = np.sqrt(np.diagonal(a).real.astype(np.longdouble))
        off = np.abs(np.tril(a.astype(wide) - low @ low.conj().T)) / np.outer(diag, diag)
        assert off.max() <= 2 * (n + 3) * np.finfo(dtype).eps, (trial, n, float(off.max()))
    assert complete >= 200


@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.complex128, np.complex64])
def test_failed_row_keeps_its_finished_columns(handle, dtype):
    """A NaN or infinite pivot in row p leaves L(p, 0 .. p - 1), which does not depend on it, as it is."""
    print(f"case failed row {np.dtype(dtype).name}", flush=True)
    rng = np.random.RandomState(12)
    n = 64
    a = nearly_singular(dtype, n, n, 0, rng) / n + np.eye(n, dtype=dtype)
    ref = np.linalg.cholesky(a.astype(np.complex128 if np.dtype(dtype).kind == "c" else np.float64))
    tol = 10 * n * np.finfo(dtype).eps  # |A^-1| < 1 and |A| < 6: an element's error is below 10 n eps
    for p in (1, 2, 3, 6, 17, 34, 47, 63):
        for value in (np.nan, np.inf):
            bad = a.copy()
            bad[p, p] = value
            A = dd.DistributedMatrix.from_global_matrix(handle, bad)
            info = dd.ppotrf(A, "L")[1]
            if np.isnan(value):
                assert info == p + 1
            assert np.abs(A.to_global_matrix()[p, :p] - ref[p, :p]).max() <= tol, (p, value)


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_complex_block_rounds_once_a_step(handle, dtype):
    """Order 64, well conditioned: the mean relative error of the factor.  Elements round
    at the scale of the trailing matrix (about half of A's) once per four columns: 16
    roundings of independent sign and rms u / sqrt(3) make 16^(1/2) / (2 sqrt(3)) = 1.2 u,
    the strip products' and the last operations' own roundings less than that again.
    Rounding at each of the 128 real terms would make 3.3 u; allowed are 2 u = eps."""
    print(f"case complex block rounding {np.dtype(dtype).name}", flush=True)
    rng = np.random.RandomState(13)
    n, errors = 64, []
    for _ in range(12):
        a = nearly_singular(dtype, n, n, 0, rng) / n + np.eye(n, dtype=dtype)
        a = ((a + a.conj().T) / 2).astype(dtype)
        # column by column in extended precision
        wide = a.astype(np.clongdouble)
        ref = np.zeros_like(wide)
        for j in range(n):
            ref[j, j] = np.sqrt((wide[j, j] - (ref[j, :j] * ref[j, :j].conj()).sum()).real)
            ref[j + 1:, j] = (wide[j + 1:, j] - ref[j + 1:, :j] @ ref[j, :j].conj()) / ref[j, j]
        A = dd.DistributedMatrix.from_global_matrix(handle, a)
        assert dd.ppotrf(A, "L")[1] == 0
        low = np.tril(A.to_global_matrix())
        errors.append(float(np.sqrt((np.abs(low - ref) ** 2).sum() / (np.abs(ref) ** 2).sum())))
    assert np.mean(errors) <= np.finfo(dtype).eps, np.mean(errors) / np.finfo(dtype).eps
