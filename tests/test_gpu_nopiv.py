"""FP32 factorisations without interchanges (nopiv.hip): the diagonal block, the
panel's rows and the diagonal-block inverses at ragged sizes."""
import numpy as np
import pytest

from emfa_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ctx():
    c = hip.Context(0)
    c.lu_params(256, 0, 2)
    yield c
    c.close()


def _lu(A):
    """LU without interchanges in complex128"""
    A = A.copy()
    for k in range(A.shape[0] - 1):
        A[k + 1:, k] /= A[k, k]
        A[k + 1:, k + 1:] -= np.outer(A[k + 1:, k], A[k, k + 1:])
    return A


def _matrix(n, seed):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)) + 3 * np.sqrt(n) * np.eye(n)
    return A.astype(np.complex64).astype(np.complex128)


# one block and less, the 4- and 8-column seams inside it, panels of 64, a
# ragged last panel, more than one outer block of 256
@pytest.mark.parametrize("n", [1, 2, 5, 8, 17, 33, 63, 64, 65, 100, 128, 191, 257, 300, 515])
def test_factor_and_solve_match_complex128(ctx, n):
    A = _matrix(n, n)
    Z = hip.Mat.from_numpy(ctx, A, hip.F32)
    lu = hip.LU(ctx, Z, hip.F32)
    assert lu.pivoting() == (0, 0) and np.array_equal(lu.pivots(), np.arange(n))
    ref = _lu(A)
    # diagonally dominant: |L| |U| <= 2 |A| row-wise and n FP32 operations per entry
    tol = 8 * np.sqrt(n) * 2.0 ** -23 * np.abs(ref).max() + 1e-6
    assert np.abs(lu.factor().numpy() - ref).max() <= tol
    for m in (1, 70):
        B = _matrix(max(n, m), 7)[:n, :m]
        X = hip.Mat.from_numpy(ctx, B, hip.F32)
        lu.solve(X)
        want = np.linalg.solve(A, B)
        assert np.linalg.norm(X.numpy() - want) <= 32 * np.sqrt(n) * 2.0 ** -23 * np.linalg.norm(want)
        X.close()
    lu.close()
    Z.close()


@pytest.mark.parametrize("n,at", [(64, 0), (64, 63), (130, 70), (200, 199), (65, 64)])
def test_zero_pivot_and_growth_fall_back_to_interchanges(ctx, n, at):
    # the leading minor of order at + 1 vanishes: column `at` has a zero pivot
    A = np.eye(n, dtype=np.complex128) * 2
    A[at, at] = 0
    if at + 1 < n:
        A[at, at + 1] = A[at + 1, at] = 1
    Z = hip.Mat.from_numpy(ctx, A, hip.F32)
    lu = hip.LU(ctx, Z, hip.F32)
    assert lu.pivoting() == (1, 1)
    assert lu.singular == (at + 1 == n)
    lu.close()
    Z.close()
