"""Coefficient fit on the GPU against the FP64 oracle.

Reference: ThinShells::cpCoefficients (ThinShells.cpp:511-617).  It assembles
A_ij = B_j(v_i) and runs Eigen's LeastSquaresConjugateGradient from x = 0.
The GPU operator is matrix-free.  The solver is mixed precision: binary32
matvec, binary64 dots and binary64 refinement.
"""
import numpy as np
import pytest

from helpers import fitted

pytestmark = pytest.mark.gpu


def _gpu(ctx, F):
    from its_amd import _capi
    c = F.case
    return _capi.Octree(ctx, c.tris, c.origin, c.width, c.R)


@pytest.mark.parametrize("name,R", [("icosphere", 64), ("bunny", 32), ("torus", 32), ("single", 8), ("corner", 16)])
def test_collocation_products_match_assembled_matrix(ctx, name, R):
    F = fitted(name, R)
    g = _gpu(ctx, F)
    rng = np.random.default_rng(0)
    x = rng.standard_normal(g.num_verts)
    y_ref, yt_ref = F.A.mul(x), F.A.tmul(x)
    y, yt = g.mul(x), g.mul(x, transpose=True)
    scale = np.abs(y_ref).max()
    assert np.abs(y - y_ref).max() <= 1e-12 * max(scale, 1)
    assert np.abs(yt - yt_ref).max() <= 1e-12 * max(np.abs(yt_ref).max(), 1)


@pytest.mark.parametrize("name,R", [("icosphere", 64), ("bunny", 64), ("torus", 32)])
def test_lscg_cold_matches_oracle(ctx, name, R):
    F = fitted(name, R)
    c = F.case
    print(f"[lscg] {c} n={F.A.n}", flush=True)
    g = _gpu(ctx, F)
    lam, st = g.lscg(F.b, tol=1e-6)
    print(st, "oracle", F.st)
    assert st["converged"] and st["normal_rel"] < 1e-6
    # binary64 check of the returned coefficients with the assembled matrix
    r = F.b - F.A.mul(lam)
    g_rel = np.linalg.norm(F.A.tmul(r)) / np.linalg.norm(F.A.tmul(F.b))
    assert g_rel < 1e-6
    # distance to the tightly converged minimum-norm solution, as for the
    # oracle's own 1e-6 iterate
    ref_err = np.abs(F.lam - F.lam_tight).max()
    err = np.abs(lam - F.lam_tight).max()
    print("lambda max err gpu", err, "oracle@1e-6", ref_err, "|lambda|max", np.abs(F.lam_tight).max())
    assert err <= max(10 * ref_err, 1e-6)
    # f at vertices (the fit targets) within 1e-5 of the oracle fit
    assert np.abs(F.A.mul(lam) - F.A.mul(F.lam)).max() <= 1e-5


def test_lscg_warm_start_from_solution(ctx):
    F = fitted("icosphere", 64)
    g = _gpu(ctx, F)
    lam, st = g.lscg(F.b, x0=F.lam_tight, tol=1e-6)
    assert st["iterations"] == 0 and st["converged"]
    np.testing.assert_allclose(lam, F.lam_tight, rtol=0, atol=0)


def test_lscg_zero_rhs(ctx):
    F = fitted("single", 8)
    g = _gpu(ctx, F)
    lam, st = g.lscg(np.zeros(g.num_verts), tol=1e-6)
    assert np.all(lam == 0)


@pytest.mark.parametrize("name,R", [("icosphere", 64), ("bunny", 32), ("torus", 32), ("single", 8), ("corner", 16)])
def test_assembled_nnz_matches_oracle(ctx, name, R):
    """The library's count of the reference matrix's non-zeros (for the
    assembled-matrix byte count of an iteration) equals the oracle's
    assembled CSR (ThinShells.cpp:556-605)."""
    F = fitted(name, R)
    g = _gpu(ctx, F)
    st = g.lscg_structure()
    assert st["n"] == F.A.n and st["nnz"] == F.A.nnz
    assert st["bytes_assembled_per_iteration"] == 16.0 * F.A.nnz + 72.0 * F.A.n
    # the operator's lists: 2 parents per odd lattice coordinate below the root
    # level; a 16-byte word of parent columns per vertex, nine 4-byte columns
    # per vertex with children
    key, level = g.vert_lattice()
    odd = (key & 1).sum(1)[level < g.depth - 1]
    assert st["parent_entries"] == (1 << odd).sum()
    assert st["bytes_matrix_free_per_iteration"] == (
        (16 + 73) * F.A.n + (36 + 8) * (level > 0).sum() + 8 * (1 << odd).sum())
