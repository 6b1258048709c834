"""Few-column products (skinny.hip) at the edges of their tiles: the
refinement residual and the steps of a triangular solve."""
import numpy as np
import pytest

from emfa_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


def _cplx(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


# rows and K around the 16-row tile and the 16 / 64 / 128 / 256 chunks of K,
# columns around the 8..64-column tiles and the 128-column limit
@pytest.mark.parametrize("prec", [hip.F32, hip.F64])
@pytest.mark.parametrize("n,m", [(1, 1), (15, 8), (16, 9), (17, 64), (65, 65), (127, 2), (129, 33), (255, 7), (257, 128),
                                 (1031, 17)])
def test_residual_product_edges(ctx, prec, n, m):
    rng = np.random.default_rng(31 * n + m)
    A = _cplx(rng, n, n)
    if prec == hip.F32:
        A = A.astype(np.complex64).astype(np.complex128)
    X, C = _cplx(rng, n, m), _cplx(rng, n, m)
    dA, dX, dC = hip.Mat.from_numpy(ctx, A, prec), hip.Mat.from_numpy(ctx, X), hip.Mat.from_numpy(ctx, C)
    for negate, accumulate in ((True, True), (False, False)):
        dC.upload(C)
        hip.gemm_residual(ctx, dA, dX, dC, negate, accumulate)
        ref = (C if accumulate else 0) + (-1 if negate else 1) * (A @ X)
        # FP64 sums of 2n products per part, in any order, on both sides
        bound = 4 * (2 * n + 4) * 2.0 ** -53 * (np.abs(A) @ np.abs(X) + np.abs(C))
        assert (np.abs(dC.numpy() - ref) <= bound).all()
    for x in (dA, dX, dC):
        x.close()


@pytest.mark.parametrize("prec", [hip.F32, hip.F64])
@pytest.mark.parametrize("n,m", [(1, 1), (17, 3), (255, 64), (257, 65), (511, 8), (513, 181), (1281, 256)])
def test_solve_steps_match_the_expanded_gemm_and_columns_stand_alone(ctx, monkeypatch, prec, n, m):
    rng = np.random.default_rng(17 * n + m)
    A = _cplx(rng, n, n) + 4 * np.sqrt(n) * np.eye(n)
    B = _cplx(rng, n, m)
    dA, dB = hip.Mat.from_numpy(ctx, A, prec), hip.Mat.from_numpy(ctx, B, prec)
    lu = hip.LU(ctx, dA, prec)
    lu.solve(dB)
    got = dB.numpy()
    # a column's bits do not depend on the block it is solved in
    j = m // 2
    one = hip.Mat.from_numpy(ctx, B[:, j], prec)
    lu.solve(one)
    assert np.array_equal(one.numpy()[:, 0], got[:, j])
    monkeypatch.setenv("EMFA_SKINNY_MAX", "0")
    dB.upload(B)
    lu.solve(dB)
    # kappa <= 4 here; backward error of the factor and two substitutions over n terms
    tol = 4 * 8 * np.sqrt(n) * (2.0 ** -24 if prec == hip.F32 else 2.0 ** -53) + 1e-15
    assert np.linalg.norm(got - dB.numpy()) <= tol * np.linalg.norm(got)
    ref = np.linalg.solve(dA.numpy(), B)
    assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)
    for x in (lu, dA, dB, one):
        x.close()


def _tiles(m, mt, slices):
    """(row tiles, column tiles) of a workgroup by the launcher's rule, for
    products of mt rows in all"""
    wgs = lambda rt, ct: -(-mt // (16 * rt)) * -(-m // (8 * ct)) * slices  # noqa: E731
    ct = 1
    while ct < 4 and 8 * ct < m:
        ct *= 2
    while ct > 1 and wgs(1, ct) < 256:
        ct //= 2
    return 2 if ct >= 2 and wgs(2, ct) >= 512 else 1, ct


def _slices(n, m, cus):
    wgs = -(-n // 16) * -(-m // 64)
    s = min(32, max(1, -(-16 * cus // wgs)))
    kc = -(-(-(-n // s)) // 128) * 128
    return -(-n // kc)


# two row tiles with two and four column tiles, rows, K and columns ragged
@pytest.mark.parametrize("prec", [hip.F32, hip.F64])
@pytest.mark.parametrize("n,m,tiles", [(2077, 13, (2, 2)), (2063, 16, (2, 2)), (2077, 33, (2, 4)), (2049, 97, (2, 4)),
                                       (4113, 64, (2, 4))])
def test_residual_with_two_row_tiles(ctx, prec, n, m, tiles):
    if ctx.cu_count() == 256:
        assert _tiles(m, n, _slices(n, m, 256)) == tiles
    rng = np.random.default_rng(31 * n + m)
    A = _cplx(rng, n, n)
    if prec == hip.F32:
        A = A.astype(np.complex64).astype(np.complex128)
    X, C = _cplx(rng, n, m), _cplx(rng, n, m)
    dA, dX, dC = hip.Mat.from_numpy(ctx, A, prec), hip.Mat.from_numpy(ctx, X), hip.Mat.from_numpy(ctx, C)
    hip.gemm_residual(ctx, dA, dX, dC)
    got, ref = dC.numpy(), C - A @ X
    bound = 4 * (2 * n + 4) * 2.0 ** -53 * (np.abs(A) @ np.abs(X) + np.abs(C))
    assert (np.abs(got - ref) <= bound).all()
    if m <= 64:  # the same slices, whatever the block: the same bits
        j = m // 2
        d1, c1 = hip.Mat.from_numpy(ctx, X[:, j:j + 1].copy()), hip.Mat.from_numpy(ctx, C[:, j:j + 1].copy())
        hip.gemm_residual(ctx, dA, d1, c1)
        assert np.array_equal(c1.numpy()[:, 0], got[:, j])
        for x in (d1, c1):
            x.close()
    for x in (dA, dX, dC):
        x.close()


@pytest.mark.parametrize("prec", [hip.F32, hip.F64])
def test_solve_steps_with_two_row_tiles(ctx, monkeypatch, prec):
    n, m = 4501, 130
    if ctx.cu_count() == 256:
        assert _tiles(m, n - 256, 1) == (2, 4)
    rng = np.random.default_rng(n)
    A = _cplx(rng, n, n)
    A[np.arange(n), np.arange(n)] += 4 * np.sqrt(n)
    B = _cplx(rng, n, m)
    dA, dB = hip.Mat.from_numpy(ctx, A, prec), hip.Mat.from_numpy(ctx, B, prec)
    lu = hip.LU(ctx, dA, prec)
    lu.solve(dB)
    got = dB.numpy()
    one = hip.Mat.from_numpy(ctx, B[:, 77], prec)
    lu.solve(one)
    assert np.array_equal(one.numpy()[:, 0], got[:, 77])
    monkeypatch.setenv("EMFA_SKINNY_MAX", "0")
    dB.upload(B)
    lu.solve(dB)
    tol = 4 * 8 * np.sqrt(n) * (2.0 ** -24 if prec == hip.F32 else 2.0 ** -53) + 1e-15
    assert np.linalg.norm(got - dB.numpy()) <= tol * np.linalg.norm(got)
    # kappa <= 4
    assert np.linalg.norm(A @ got - B) <= 4 * tol * np.linalg.norm(B)
    for x in (lu, dA, dB, one):
        x.close()
