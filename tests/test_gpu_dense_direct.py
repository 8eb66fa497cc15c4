"""Meshes small enough for the dense inverse are solved directly: the inverse
(64-row symmetric sweep on the device) at free-dof counts below, at and above
multiples of its block, in 2D and 3D.  With an accurate inverse the inner CG
needs at most three iterations per solve (one product, one correction of its
rounding, one to confirm), and the solution is the oracle's to the solver
tolerance of the other parity tests."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

# free dofs with free-slip walls: 2 (nx ny - 1) in 2D
MESHES = [(2, 3, 5, 1, 28), (2, 4, 8, 1, 62), (2, 3, 11, 1, 64), (2, 5, 7, 1, 68), (2, 5, 13, 1, 128),
          (2, 6, 11, 1, 130), (2, 16, 24, 1, 766), (2, 33, 31, 1, 2044), (3, 3, 4, 5, None), (3, 7, 6, 5, None)]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dim,nx,ny,nz,nfree", MESHES)
def test_direct_inner_solve(gale, oracle, dim, nx, ny, nz, nfree, prec):
    res = (nx, ny, nz)[:dim]
    lo, hi = (0.0,) * dim, (1.0,) * dim
    coord = gale.layout_random(dim, res, lo, hi, 6, 13)
    mats = [gale.material(eta0=1.0, density=1.0), gale.material(eta0=1e3, density=1.1)]
    mat = gale.shape_layout(dim, coord, [gale.everywhere(0), gale.sphere(1, (0.5, 0.55, 0.5), 0.3)])
    mask, vals = gale.free_slip(dim, res)
    if nfree is not None:
        assert int((mask == 0).sum()) == nfree
    kw = dict(dim=dim, res=res, lo=lo, hi=hi, materials=mats, bc_mask=mask, bc_value=vals, gravity=1.0,
              ghat=(0.0, -1.0, 0.0), eta_clamp=(0.0, 0.0), eta0_particle=None)
    pb = gale.Problem(coord=coord, material_index=mat, **kw)
    s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(tolerance=1e-10, inner_rtol_override=1e-12, precision=prec,
                                                          maxIterations=20000))
    u, p, rep = s.Solve()
    assert rep.inner_iterations <= 3 * (rep.uzawa_iterations + 2)
    o = oracle.Problem(coord=coord, material=mat, **kw)
    st, ou, op, _ = o.uzawa(oracle.uzawa_params(tolerance=1e-10, inner_rtol_override=1e-13))
    assert st == 0 and rel(u, ou) < 1e-8 and rel(p - p.mean(), op - op.mean()) < 1e-8
    # solving again (the inverse is formed anew in the same buffers) changes nothing
    s.set_pressure(None)
    s.setup()
    u2, p2, _ = s.Solve()
    assert np.array_equal(u, u2) and np.array_equal(p, p2)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dim,nx,ny,nz", [(2, 16, 24, 1), (2, 33, 31, 1), (3, 7, 6, 5)])
def test_direct_at_contrast_1e6(gale, oracle, dim, nx, ny, nz, prec):
    """A million in viscosity, the range of the sinker batches: still at most
    three inner iterations a solve.  Both sides stop at 1e-8; a residual of a
    contrast C is worth up to sqrt(C) times as much error: 1e-5 each."""
    res = (nx, ny, nz)[:dim]
    lo, hi = (0.0,) * dim, (1.0,) * dim
    coord = gale.layout_random(dim, res, lo, hi, 6, 13)
    mats = [gale.material(eta0=1.0, density=1.0), gale.material(eta0=1e6, density=1.1)]
    mat = gale.shape_layout(dim, coord, [gale.everywhere(0), gale.sphere(1, (0.5, 0.55, 0.5), 0.3)])
    mask, vals = gale.free_slip(dim, res)
    kw = dict(dim=dim, res=res, lo=lo, hi=hi, materials=mats, bc_mask=mask, bc_value=vals, gravity=1.0,
              ghat=(0.0, -1.0, 0.0), eta_clamp=(0.0, 0.0), eta0_particle=None)
    pb = gale.Problem(coord=coord, material_index=mat, **kw)
    s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(tolerance=1e-8, inner_rtol_override=1e-10, precision=prec,
                                                          maxIterations=20000))
    u, p, rep = s.Solve()
    assert rep.inner_iterations <= 3 * (rep.uzawa_iterations + 2)
    o = oracle.Problem(coord=coord, material=mat, **kw)
    st, ou, op, _ = o.uzawa(oracle.uzawa_params(tolerance=1e-8, inner_rtol_override=1e-12))
    assert st == 0 and rel(u, ou) < 2e-5 and rel(p - p.mean(), op - op.mean()) < 2e-5


def test_refused_when_singular(gale):
    """An operator without any stiffness (everything yields to zero viscosity)
    has zero pivots on every level: the setup reports it."""
    coord = gale.layout_random(2, (6, 5), (0.0, 0.0), (1.0, 1.0), 6, 13)
    mask, vals = gale.free_slip(2, (6, 5))
    pb = gale.Problem(2, (6, 5), (0.0, 0.0), (1.0, 1.0), coord, np.zeros(len(coord), np.int32),
                      [gale.material(density=1.0, yield_type=2, cohesion=0.0)], bc_mask=mask, bc_value=vals)
    s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params())
    s.setup()  # nothing yields without a previous velocity
    with pytest.raises(gale.GaleError) as e:
        s.setup(np.random.default_rng(3).standard_normal(pb.N * 2), np.zeros(pb.E), yield_on=True)
    assert e.value.status == gale.E_NAN
