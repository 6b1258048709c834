"""BiCGSTAB with several right-hand sides at once, and the row-sharing
matrix-vector product under it, at the sizes where their rules change."""
import numpy as np
import pytest

from emfa_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


def _system(n, m, seed):
    # a dominant diagonal with entries of different size, so that columns end
    # after different numbers of steps
    rng = np.random.default_rng(seed)
    Z = rng.standard_normal((n, n)).astype(np.float32) + 1j * rng.standard_normal((n, n)).astype(np.float32)
    Z = Z.astype(np.complex64) / np.float32(4 * np.sqrt(n))
    Z[np.arange(n), np.arange(n)] += np.exp(1j * rng.uniform(0, 1, n)).astype(np.complex64)
    B = rng.standard_normal((n, m)) + 1j * rng.standard_normal((n, m))
    B[:, 0] = 0
    B[0, 0] = 1
    return Z, B


# one row per wave and two, with remainders of rows; 5 columns run as a group of
# four and one alone
@pytest.mark.parametrize("prec", [hip.F32, hip.F64])
@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("n,m", [(1, 2), (63, 5), (257, 3), (3073, 2), (6147, 4)])
def test_columns_of_a_group_are_solved_as_if_alone(ctx, prec, variant, n, m):
    Z, B = _system(n, m, n + m)
    if m > 2:
        B[:, 2] = 0  # done before the first step
    dZ, dB, X = hip.Mat.from_numpy(ctx, Z, prec), hip.Mat.from_numpy(ctx, B), hip.Mat(ctx, n, m)
    rep, ok = hip.bicgstab(ctx, dZ, dB, X, tol=1e-9, max_iter=60, variant=variant)
    assert ok and rep.relres < 2e-9
    got, steps, most = X.numpy(), 0, 0
    for j in range(m):
        d1, x1 = hip.Mat.from_numpy(ctx, B[:, j:j + 1].copy()), hip.Mat(ctx, n, 1)
        r1, ok1 = hip.bicgstab(ctx, dZ, d1, x1, tol=1e-9, max_iter=60, variant=variant)
        assert ok1 and np.array_equal(x1.numpy()[:, 0], got[:, j])
        steps, most = steps + r1.iterations, max(most, r1.max_steps)
    assert (rep.iterations, rep.max_steps) == (steps, most)
    # FP64 sums over n elements on both sides, against the solver's own 2e-9
    res = np.linalg.norm(B - Z.astype(np.complex128) @ got, axis=0)
    assert (res <= 2.1e-9 * np.linalg.norm(B, axis=0)).all()


def _rows_per_wave(n, nc, prec, cus):
    """The rule under test: fewest rows whose matrix bytes match the vectors'"""
    fit, r = n // ((12 if nc == 1 else 7) * cus), 1
    while r < 4 and 2 * r <= fit and r * (8 if prec == hip.F32 else 16) < 16 * nc:
        r *= 2
    return r


# Four rows per wave with remainders of one to three rows; two for the columns
# alone in FP32; FP64 matrices around the last cache's size, where one vector
# alone loads less ahead than a group does
@pytest.mark.parametrize("prec,n,m,rows,alone", [(hip.F32, 7169, 2, 4, 2), (hip.F32, 7170, 3, 4, 2), (hip.F32, 7171, 4, 4, 2),
                                                 (hip.F64, 7170, 3, 4, 1), (hip.F64, 7171, 4, 4, 1), (hip.F64, 4097, 2, 2, 1)])
def test_rows_shared_by_a_wave_keep_a_columns_bits(ctx, prec, n, m, rows, alone):
    cus = ctx.cu_count()
    if cus == 256:
        assert (_rows_per_wave(n, m, prec, cus), _rows_per_wave(n, 1, prec, cus)) == (rows, alone)
    Z, B = _system(n, m, n + m)
    dZ, dB, X = hip.Mat.from_numpy(ctx, Z, prec), hip.Mat.from_numpy(ctx, B), hip.Mat(ctx, n, m)
    rep, ok = hip.bicgstab(ctx, dZ, dB, X, tol=1e-6, max_iter=60)
    assert ok
    got = X.numpy()
    for j in range(m):
        d1, x1 = hip.Mat.from_numpy(ctx, B[:, j:j + 1].copy()), hip.Mat(ctx, n, 1)
        hip.bicgstab(ctx, dZ, d1, x1, tol=1e-6, max_iter=60)
        assert np.array_equal(x1.numpy()[:, 0], got[:, j])
        for x in (d1, x1):
            x.close()
    # the last rows, whose waves have fewer of them
    res = (B - Z.astype(np.complex128) @ got)[-8:]
    assert np.linalg.norm(res) <= 2e-6 * np.linalg.norm(B)
    for x in (dZ, dB, X):
        x.close()
