"""The dense solve that reads half of the symmetric inverse (inverses of 96 MB
and more): directly on meshes whose free dofs end inside, at and just short of
a 64-row block, against the oracle; and in FP32 as the coarsest level of a
V-cycle, where a wrong solve costs inner iterations."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


def problem(gale, dim, res):
    lo, hi = (0.0,) * dim, (1.0,) * dim
    coord = gale.layout_random(dim, res, lo, hi, 6, 13)
    mats = [gale.material(eta0=1.0, density=1.0), gale.material(eta0=1e2, density=1.1)]
    mat = gale.shape_layout(dim, coord, [gale.everywhere(0), gale.sphere(1, (0.5, 0.55, 0.5), 0.3)])
    mask, vals = gale.free_slip(dim, res)
    kw = dict(dim=dim, res=res, lo=lo, hi=hi, materials=mats, bc_mask=mask, bc_value=vals, gravity=1.0,
              ghat=(0.0, -1.0, 0.0), eta_clamp=(0.0, 0.0), eta0_particle=None)
    return coord, mat, mask, kw


@pytest.mark.parametrize("nx,ny,nfree", [(42, 43, 3610), (25, 73, 3648), (50, 60, 5998)])
def test_direct(gale, oracle, nx, ny, nfree):
    coord, mat, mask, kw = problem(gale, 2, (nx, ny))
    assert int((mask == 0).sum()) == nfree and 8 * nfree ** 2 >= 96 << 20
    pb = gale.Problem(coord=coord, material_index=mat, **kw)
    s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(tolerance=1e-9, inner_rtol_override=1e-12,
                                                          maxIterations=20000))
    u, p, rep = s.Solve()
    assert rep.inner_iterations <= 3 * (rep.uzawa_iterations + 2)
    o = oracle.Problem(coord=coord, material=mat, **kw)
    st, ou, op, _ = o.uzawa(oracle.uzawa_params(tolerance=1e-9, inner_rtol_override=1e-12))
    # both stop at 1e-9 of the right-hand side
    assert st == 0 and rel(u, ou) < 1e-7 and rel(p - p.mean(), op - op.mean()) < 1e-7


def test_coarsest_level(gale):
    """24^3: the 12^3 level (5577 free dofs, 124 MB in FP32) is the dense one.
    FP32 V-cycles precondition as well as FP64 ones, so an inner solve needs
    no more iterations (one a solve for rounding)."""
    coord, mat, _, kw = problem(gale, 3, (24, 24, 24))
    out = []
    for prec in (0, 1):
        pb = gale.Problem(coord=coord, material_index=mat, **kw)
        s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(tolerance=1e-7, inner_rtol_override=1e-9, precision=prec))
        u, p, rep = s.Solve()
        out.append((u, rep.inner_iterations, rep.uzawa_iterations))
    (u0, i0, n0), (u1, i1, n1) = out
    assert abs(n0 - n1) <= 1 and i1 <= i0 + n1 + 20
    assert rel(u1, u0) < 1e-6
