"""FP32 factorisations without interchanges (nopiv.hip): the diagonal block, the
panel's rows and the diagonal-block inverses at ragged sizes, and factors with
multipliers well above one."""
import numpy as np
import pytest
from scipy.linalg import solve_triangular

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


def _lu32(A):
    """LU without interchanges in complex64, 64 columns at a time: U's rows by
    substitution, the rows below through U^-1 of the panel"""
    A = A.astype(np.complex64)
    n = A.shape[0]
    for j in range(0, n, 64):
        e = min(n, j + 64)
        for k in range(j, e):
            A[k + 1:e, k] /= A[k, k]
            A[k + 1:e, k + 1:e] -= np.outer(A[k + 1:e, k], A[k, k + 1:e])
        if e < n:
            A[e:, j:e] = A[e:, j:e] @ solve_triangular(A[j:e, j:e], np.eye(e - j, dtype=np.complex64))
            A[j:e, e:] = solve_triangular(A[j:e, j:e], A[j:e, e:], lower=True, unit_diagonal=True)
            A[e:, e:] -= A[e:, j:e] @ A[j:e, e:]
    return A.astype(np.complex128)


def _solution_error(F, B, want):
    X = solve_triangular(F, solve_triangular(F, B, lower=True, unit_diagonal=True))
    return np.linalg.norm(X - want) / np.linalg.norm(want)


# one diagonal block with multipliers below one, where every rounding counts alike
@pytest.mark.parametrize("n", [20, 32, 64])
def test_diagonal_block_rounds_once_per_product(ctx, n):
    logs = []
    for seed in range(16):
        rng = np.random.default_rng(seed + n)
        A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)) + 2 * np.sqrt(n) * np.eye(n)
        A = A.astype(np.complex64).astype(np.complex128)
        Z = hip.Mat.from_numpy(ctx, A, hip.F32)
        lu = hip.LU(ctx, Z, hip.F32)
        ref = _lu(A)
        logs.append(np.log(np.linalg.norm(lu.factor().numpy() - ref) / np.linalg.norm(_lu32(A) - ref)))
        lu.close()
        Z.close()
    # the same roundings as complex64's; a second one per product at the size of
    # the entry makes this sqrt(2)
    assert np.mean(logs) <= np.log(1.2)


# Small shifts leave multipliers of 10 to 100.  One outer block with U rows
# beside it, a ragged second 256-block of an outer block, several outer blocks;
# FP32 and bf16-split updates.
@pytest.mark.parametrize("n,nb,split,shift", [(300, 256, 0, 1.0), (400, 300, 0, 1.0), (790, 320, 1, 1.0),
                                              (1100, 256, 0, 1.0), (1100, 256, 0, 0.5), (1100, 512, 0, 1.0)])
def test_large_multipliers_cost_no_more_than_substitution(n, nb, split, shift):
    ctx = hip.Context(0)
    ctx.lu_params(nb, 0, 2)
    ctx.lu_update_mode(split)
    logs = []
    for seed in range(12):
        rng = np.random.default_rng(7 * seed + n)
        A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)) + shift * np.sqrt(n) * np.eye(n)
        A = A.astype(np.complex64).astype(np.complex128)
        B = rng.standard_normal((n, 3)) + 1j * rng.standard_normal((n, 3))
        Z = hip.Mat.from_numpy(ctx, A, hip.F32)
        lu = hip.LU(ctx, Z, hip.F32)
        if lu.pivoting() == (0, 0):
            F, want = lu.factor().numpy(), np.linalg.solve(A, B)
            assert np.abs(np.tril(F, -1)).max() <= 100
            if not split:
                logs.append(np.log(_solution_error(F, B, want) / _solution_error(_lu32(A), B, want)))
            dB, X = hip.Mat.from_numpy(ctx, B), hip.Mat(ctx, n, 3)
            rep, ok = hip.refine(ctx, Z, lu, dB, X, 1e-10, 30)
            assert ok and np.linalg.norm(X.numpy() - want) <= 1e-10 * np.linalg.cond(A) * np.linalg.norm(want)
            for x in (dB, X):
                x.close()
        lu.close()
        Z.close()
        if len(logs) == 8:
            break
    if not split:
        assert len(logs) >= 4
        # The mean ratio of the two errors: at most sqrt(2) from the matrix cores'
        # two roundings per complex step, and three deviations of a mean of
        # single ratios that spread by a factor of e^0.6
        assert np.mean(logs) <= 0.5 * np.log(2) + 3 * 0.6 / np.sqrt(len(logs))
    ctx.close()


# runs of one and two multipliers of 5 to 90: inverses of L hold their products
@pytest.mark.parametrize("n,t,run", [(300, 90, 1), (515, 10, 2), (1100, 90, 1)])
def test_runs_of_large_multipliers_refine(ctx, n, t, run):
    rng = np.random.default_rng(n + t)
    L = np.eye(n, dtype=np.complex128) + np.tril(rng.standard_normal((n, n)), -1) / n
    for k in range(n - 1):
        if k % (run + 1) != run:
            L[k + 1, k] = rng.uniform(5, t) * np.exp(2j * np.pi * rng.random())
    U = np.triu(rng.standard_normal((n, n)), 1) / np.sqrt(n) + np.diag(1 + rng.random(n))
    A = (L @ U).astype(np.complex64).astype(np.complex128)
    B = rng.standard_normal((n, 2)) + 1j * rng.standard_normal((n, 2))
    Z = hip.Mat.from_numpy(ctx, A, hip.F32)
    lu = hip.LU(ctx, Z, hip.F32)
    assert lu.pivoting() == (0, 0)
    want = np.linalg.solve(A, B)
    mine, plain = _solution_error(lu.factor().numpy(), B, want), _solution_error(_lu32(A), B, want)
    assert mine <= 4 * plain
    dB, X = hip.Mat.from_numpy(ctx, B), hip.Mat(ctx, n, 2)
    # FP64 rounds the residual at 2^-53 |A| |X|, far above 1e-12 |B| for some of these
    floor = 8 * 2.0 ** -53 * np.linalg.norm(A) * np.linalg.norm(want) / np.linalg.norm(B, axis=0).min()
    rep, ok = hip.refine(ctx, Z, lu, dB, X, max(1e-12, floor), 6)
    assert ok
    for x in (lu, Z, dB, X):
        x.close()


@pytest.mark.parametrize("n,nb", [(700, 300), (1100, 448)])
def test_ragged_outer_blocks_in_a_graph_match_eager_launches(n, nb):
    ctxs = [hip.Context(0) for _ in range(2)]
    for c in ctxs:
        c.lu_params(nb, 0, 2)
        c.lu_update_mode(1)
    ctxs[0].graphs(True)
    for seed in range(4):
        A = _matrix(n, seed)
        F = []
        for c in ctxs:
            Z = hip.Mat.from_numpy(c, A, hip.F32)
            lu = hip.LU(c, Z, hip.F32)
            assert lu.pivoting() == (0, 0)
            F.append(lu.factor().numpy())
            lu.close()
            Z.close()
        assert np.array_equal(F[0], F[1])
    assert ctxs[0].graph_stats() == (1, 4)
    L, U = np.tril(F[0], -1) + np.eye(n), np.triu(F[0])
    tol = (6 * 2.0 ** -18 + 4 * n ** 0.5 * 2.0 ** -23) * (np.abs(L) @ np.abs(U))
    assert (np.abs(L @ U - A) <= tol).all()
    for c in ctxs:
        c.close()


# U rows in strips of 8, 16 and 32 columns: the CUs to fill decide, an entry's
# sums do not depend on it; ragged blocks of rows and ragged last strips
@pytest.mark.parametrize("n,nb", [(301, 64), (523, 100), (700, 300), (777, 512)])
def test_strips_of_every_width_give_the_same_factor(n, nb):
    A = _matrix(n, nb)
    F = []
    for share in (0, (n - nb) // 12, 2):  # one round of 8, of 16, none
        c = hip.Context(0)
        c.lu_params(nb, 0, 2)
        if share:
            c.set_cu_share(share)
        Z = hip.Mat.from_numpy(c, A, hip.F32)
        lu = hip.LU(c, Z, hip.F32)
        assert lu.pivoting() == (0, 0)
        F.append(lu.factor().numpy())
        lu.close()
        Z.close()
        c.close()
    ref = _lu(A)
    tol = 8 * np.sqrt(n) * 2.0 ** -23 * np.abs(ref).max() + 1e-6
    assert np.abs(F[0] - ref).max() <= tol
    assert np.array_equal(F[0], F[1]) and np.array_equal(F[0], F[2])
