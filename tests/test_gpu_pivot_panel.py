"""Panels with interchanges (packet exchange): the pivots of LAPACK's rule at
the edges of workgroups' rows, panels and the packets' 12-bit epoch."""
import numpy as np
import pytest
import scipy.linalg

from emfa_amd import hip

pytestmark = pytest.mark.gpu


# one row; one workgroup and a row more (48); three workgroups; a ragged panel;
# more columns than the 4096 epochs of a packet
@pytest.mark.parametrize("prec,n", [(p, n) for p in (hip.F64, hip.F32) for n in (1, 2, 47, 48, 49, 65, 97, 145, 333)] +
                         [(hip.F64, 4133)])
def test_pivots_and_factors_match_lapack(prec, n):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    if prec == hip.F32:
        A = A.astype(np.complex64).astype(np.complex128)
    ctx = hip.Context(0)
    ctx.lu_params(256, 0, 1)
    Z = hip.Mat.from_numpy(ctx, A, prec)
    lu = hip.LU(ctx, Z, prec)
    ref, piv = scipy.linalg.lu_factor(A)
    assert np.array_equal(lu.pivots(), piv)
    L, U = np.tril(ref, -1) + np.eye(n), np.triu(ref)
    F = lu.factor().numpy().astype(np.complex128)
    # each side's L U differs from the permuted A by at most a small multiple of
    # n u |L| |U| (complex products and sums of up to n terms)
    u = 2.0 ** (-24 if prec == hip.F32 else -53)
    bound = 8 * n * u * (np.abs(L) @ np.abs(U))
    got = (np.tril(F, -1) + np.eye(n)) @ np.triu(F)
    assert (np.abs(got - L @ U) <= bound).all()
    lu.close()
    Z.close()
    ctx.close()
