"""V-cycles whose levels are smoothed from assembled rows, from tiled moments
or both, with one to three smoothing steps (with one, the first Chebyshev step
is worked out inside the residual): the solution against the oracle's where
the mesh is small, and the momentum residual |f - K u - G p| / |f| (evaluated
point by point) where it is not.  Meshes: even and odd, unequal axes, one that
does not coarsen (eight smoothing steps in place of a coarse solve)."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


def _sinker(gale, dim, res, ppc=6):
    lo, hi = (0.0,) * dim, (1.0,) * dim
    coord = gale.layout_random(dim, res, lo, hi, ppc, 13)
    mat = gale.shape_layout(dim, coord, [gale.everywhere(0), gale.sphere(1, (0.5, 0.55, 0.5), 0.3)])
    mask, vals = gale.free_slip(dim, res)
    return dict(dim=dim, res=res, lo=lo, hi=hi, materials=[gale.material(density=1.0),
                                                           gale.material(eta0=50.0, density=1.2)], bc_mask=mask,
                bc_value=vals, gravity=1.0, ghat=(0.0, -1.0, 0.0), eta_clamp=(0.0, 0.0), eta0_particle=None), coord, mat


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("nu,nuc", [(1, 1), (2, 1), (3, 2)])
@pytest.mark.parametrize("dim,res,dense_max", [
    (2, (24, 40), 300),     # 24x40 assembled, 12x20 assembled, 6x10 dense
    (2, (31, 26), 300),     # does not coarsen and too large for the bound: smoothing only
    (3, (8, 12, 10), 600),  # assembled, 4x6x5 dense
    (3, (9, 7, 8), 600),    # smoothing only
])
def test_small_levels_match_oracle(gale, oracle, monkeypatch, dim, res, dense_max, nu, nuc, prec):
    monkeypatch.setenv("GALE_MG_DENSE_MAX", str(dense_max))
    kw, coord, mat = _sinker(gale, dim, res)
    pb = gale.Problem(coord=coord, material_index=mat, **kw)
    s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(
        tolerance=1e-10, inner_rtol_override=1e-12, precision=prec, maxIterations=20000, mg_smooth=nu,
        mg_smooth_coarse=nuc))
    u, p, rep = s.Solve()
    assert rep.inner_iterations > 2 * rep.uzawa_iterations  # the V-cycle ran, not the direct solve
    o = oracle.Problem(coord=coord, material=mat, **kw)
    st, ou, op, _ = o.uzawa(oracle.uzawa_params(tolerance=1e-10, inner_rtol_override=1e-13))
    assert st == 0 and rel(u, ou) < 1e-8 and rel(p - p.mean(), op - op.mean()) < 1e-8


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dim,res", [(2, (520, 512)), (3, (36, 32, 34)), (3, (40, 36, 32))])
def test_large_levels_momentum_residual(gale, dim, res, prec):
    kw, coord, mat = _sinker(gale, dim, res, ppc=4)
    pb = gale.Problem(coord=coord, material_index=mat, **kw)
    for nu in (1, 2):
        s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(tolerance=1e-3, inner_rtol_override=1e-9, precision=prec,
                                                              maxIterations=200, mg_smooth=nu))
        u, p, rep = s.Solve()
        # the velocity is a sum of inner solves, each to 1e-9 of its right-hand side
        assert rep.status == 0 and rep.momentum_residual < 1e-7
        s.close()
