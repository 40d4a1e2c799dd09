"""The 64 x 64 diagonal block's factorization (four columns a step, 16-column
strips): orders at the edges of steps, strips and blocks, and a failed pivot in
each place of a step, against the oracle.

Tolerance: backward-stable Cholesky of order n has |L - L_ref| <= c n eps
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
