"""The three-term bf16 trailing update at ragged sizes: both tile sizes, K
padded to whole stages, single matrices and the growth of the error."""
import numpy as np
import pytest

from emfa_amd import hip

pytestmark = pytest.mark.gpu


# outer blocks whose 2 nb reals are and are not whole stages of 32, trailing
# blocks from one row to more than 1.5 large tiles per CU (5300 unknowns)
@pytest.mark.parametrize("n,nb", [(65, 64), (130, 64), (321, 40), (515, 256), (700, 24), (1153, 256), (5300, 512)])
def test_factors_multiply_back(n, nb):
    ctx = hip.Context(0)
    ctx.lu_params(nb, 0, 2)
    ctx.lu_update_mode(1)
    rng = np.random.default_rng(n)
    A = (rng.standard_normal((n, n), np.float32) + 1j * rng.standard_normal((n, n), np.float32)).astype(np.complex64)
    A[np.arange(n), np.arange(n)] += np.float32(3 * n ** 0.5)
    Z = hip.Mat.from_numpy(ctx, A, hip.F32)
    lu = hip.LU(ctx, Z, hip.F32)
    assert lu.pivoting() == (0, 0)
    F = lu.factor().numpy().astype(np.complex128)
    L, U = np.tril(F, -1) + np.eye(n), np.triu(F)
    cols = np.unique(np.r_[np.arange(0, n, -(-n // 150)), np.arange(max(0, n - 70), n)])
    err = np.abs(L @ U[:, cols] - A[:, cols])
    # hi + lo keeps x to 2^-18 |x|, lo lo is dropped (2^-18), and a part of a
    # complex product has two real ones: 6 2^-18 |L||U|; and FP32 sums
    tol = (6 * 2.0 ** -18 + 4 * n ** 0.5 * 2.0 ** -23) * (np.abs(L) @ np.abs(U[:, cols]))
    assert (err <= tol).all()
    lu.close()
    Z.close()
    ctx.close()
