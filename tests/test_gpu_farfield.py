"""Excitation columns and far field at the edges of their launches: columns per
thread, triangle slices, direction blocks, against the FP64 oracle."""
import numpy as np
import pytest

from emfa_amd import hip
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.Context(0)
    yield c
    c.close()


def _mesh(ctx, mesh, size):
    xyz, tri = hip.plate(size, 0.9) if mesh == "plate" else hip.icosphere(size, 0.5, 0.55, 0.4)
    rwg, _ = hip.rwg_build(tri)
    return hip.Mesh(ctx, xyz, tri, rwg), xyz, tri, rwg


# 70 columns of 7680 unknowns take four columns per thread (a ragged last group),
# the others one: the line is at 2048 values per CU
@pytest.mark.parametrize("kind", [hip.EFIE, hip.CFIE])
@pytest.mark.parametrize("mesh,size,m", [("plate", 1, 1), ("plate", 7, 5), ("ico", 2, 64), ("ico", 3, 181),
                                         ("ico", 4, 70)])
def test_excitation_matches_oracle(ctx, kind, mesh, size, m):
    M, xyz, tri, rwg = _mesh(ctx, mesh, size)
    assert (M.n * m >= 2048 * ctx.cu_count()) == (M.n * m == 7680 * 70) or ctx.cu_count() != 256
    k, inc = hip.wavenumber(4e8), hip.inc_table([(3.0 + 170.0 * j / m, 20.0, 35.0) for j in range(m)])
    ref = O.rhs(xyz, tri, rwg, kind, k, 0.3, inc)
    for prec, tol in ((hip.F64, 1e-13), (hip.F32, 2e-7)):
        B = hip.Mat(ctx, M.n, m, prec)
        hip.rhs_fill(ctx, M, B, kind, k, 0.3, inc)
        assert np.abs(B.numpy() - ref).max() <= tol * np.abs(ref).max()
        if kind == hip.EFIE:  # the magnetic field is not read
            bad = inc.copy()
            bad[:, 6:9] = np.nan
            hip.rhs_fill(ctx, M, B, kind, k, 0.3, bad)
            assert np.abs(B.numpy() - ref).max() <= tol * np.abs(ref).max()
        B.close()
    M.close()


@pytest.mark.parametrize("prec", [hip.F32, hip.F64])
@pytest.mark.parametrize("mesh,size,ndir,ncol", [("plate", 1, 1, 1), ("ico", 1, 65, 2), ("plate", 12, 64, 64),
                                                 ("ico", 3, 181, 3), ("ico", 4, 7, 1)])
def test_far_field_matches_oracle(ctx, mesh, size, ndir, ncol, prec):
    M, xyz, tri, rwg = _mesh(ctx, mesh, size)
    rng = np.random.default_rng(ndir)
    X = (rng.standard_normal((M.n, ncol)) + 1j * rng.standard_normal((M.n, ncol))).astype(np.complex64)
    dirs = rng.standard_normal((ndir, 3))
    dirs /= np.linalg.norm(dirs, axis=1)[:, None]
    cols = rng.integers(0, ncol, ndir).astype(np.int32)
    dX = hip.Mat.from_numpy(ctx, X.astype(np.complex128), prec)
    k = hip.wavenumber(4e8)
    for c in (cols, None):
        got = hip.rcs(ctx, M, k, dX, dirs, c)
        use = cols if c is not None else np.zeros(ndir, dtype=np.int32)
        ref = O.rcs(xyz, tri, rwg, k, X.astype(np.complex128), dirs, use)
        assert np.abs(got - ref).max() <= 1e-9
    dX.close()
    M.close()
