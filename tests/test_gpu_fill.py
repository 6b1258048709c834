"""Impedance fill at its seams: chunks of test triangles, the 64-triangle and
4-half-function tiles, both rules, both precisions, with and without a surface
impedance, against the FP64 oracle."""
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


# plates: 2, 18, 64 and 162 triangles (open edges); spheres 80 and 320.  A
# scratch of 0 MB takes chunks of four triangles, so rows span chunks.
@pytest.mark.parametrize("quad", [3, 7])
@pytest.mark.parametrize("kind,mesh,size", [(hip.EFIE, "plate", 1), (hip.EFIE, "plate", 3), (hip.EFIE, "ico", 1),
                                            (hip.CFIE, "ico", 1), (hip.CFIE, "ico", 2), (hip.EFIE, "plate", 9)])
@pytest.mark.parametrize("scratch_mb", [None, "0"])
def test_fill_matches_oracle(ctx, monkeypatch, kind, mesh, size, quad, scratch_mb):
    if scratch_mb is not None:
        monkeypatch.setenv("EMFA_FILL_SCRATCH_MB", scratch_mb)
    xyz, tri = hip.plate(size, 0.7) if mesh == "plate" else hip.icosphere(size, 0.5, 0.45, 0.6)
    rwg, _ = hip.rwg_build(tri)
    k = hip.wavenumber(2.5e8)
    sigma = (20.0 + 5.0j) if kind == hip.EFIE and mesh == "plate" else 0j
    M = hip.Mesh(ctx, xyz, tri, rwg)
    if kind == hip.EFIE:
        ref = O.fill_efie(xyz, tri, rwg, k, quad, sigma=sigma)
    else:
        ref = O.fill_cfie(xyz, tri, rwg, k, 0.4, quad)
    for prec, tol in ((hip.F64, 1e-12), (hip.F32, 2e-5)):  # 64 and 2^-24 x the near entries' cancellation
        Z = hip.Mat(ctx, M.n, M.n, prec)
        Z.upload(np.full((M.n, M.n), np.nan + 1j * np.nan))  # every entry is written
        hip.fill(ctx, M, Z, kind, k, quad, alpha=0.4, sigma=sigma)
        assert np.abs(Z.numpy() - ref).max() <= tol * np.abs(ref).max()
        Z.close()
    M.close()


@pytest.mark.parametrize("kr", [0.01, 3.0, 400.0])
def test_phase_reduction_follows_the_wave_number(ctx, kr):
    # two far triangle pairs: Z tends to a plane phase; k R up to 400 radians
    xyz, tri = hip.plate(2, 1.0)
    xyz2 = np.concatenate([xyz, xyz + np.array([10.0, 3.0, 1.0])])
    tri2 = np.concatenate([tri, tri + len(xyz)]).astype(np.int32)
    rwg, _ = hip.rwg_build(tri2)
    k = kr / np.linalg.norm([10.0, 3.0, 1.0])
    M = hip.Mesh(ctx, xyz2, tri2, rwg)
    ref = O.fill_efie(xyz2, tri2, rwg, k, 7)
    for prec, tol in ((hip.F64, 1e-12), (hip.F32, 2e-5 + kr * 2.0 ** -24)):
        Z = hip.Mat(ctx, M.n, M.n, prec)
        hip.fill(ctx, M, Z, hip.EFIE, k, 7)
        assert np.abs(Z.numpy() - ref).max() <= tol * np.abs(ref).max()
        Z.close()
    M.close()
