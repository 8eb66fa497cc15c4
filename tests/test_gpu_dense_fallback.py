"""The dense inverse when its operator has no stiffness somewhere: materials
that yield to zero viscosity leave zero pivots, which are certain to fail.
Around a node that the next coarser level does not have, only the finest level
fails and the setup falls back to that coarser one; everywhere, every level
fails and the setup reports it.  Either way the next setup starts afresh: the
solver then gives the bits of one that never saw the bad field."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


def _problem(gale, dim, everywhere):
    res = (16, 12, 8)[:dim] if dim == 2 else (8, 6, 8)
    lo, hi = (0.0,) * dim, (1.0,) * dim
    coord = gale.layout_random(dim, res, lo, hi, 6, 13)
    # the elements around node (5, 3) or (5, 3, 3): one element of the coarser level
    a = [4 / res[0], 2 / res[1], 2 / res[-1]][:dim]
    b = [6 / res[0], 4 / res[1], 4 / res[-1]][:dim]
    mat = gale.shape_layout(dim, coord, [gale.everywhere(0), gale.box(1, a + [0.0] * (3 - dim), b + [1.0] * (3 - dim))])
    zero = dict(yield_type=2, cohesion=0.0, min_viscosity=0.0)
    mats = [gale.material(eta0=2.0, density=1.0, **(zero if everywhere else {})),
            gale.material(eta0=1.0, density=1.2, **zero)]
    mask, vals = gale.free_slip(dim, res)
    pb = gale.Problem(dim, res, lo, hi, coord, mat, mats, bc_mask=mask, bc_value=vals)
    u = np.random.default_rng(3).standard_normal(pb.N * dim)
    return pb, u, np.zeros(pb.E)


def _solver(gale, pb, prec):
    return gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(tolerance=1e-8, inner_rtol_override=1e-11,
                                                             precision=prec, maxIterations=5000))


def _solve(s):
    s.set_pressure(None)
    s.setup()
    return s.Solve()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dim", [2, 3])
def test_falls_back_to_the_coarser_level_and_returns(gale, dim, prec):
    import torch
    pb, u, p = _problem(gale, dim, False)
    uf, pf, rf = _solve(_solver(gale, pb, prec))
    assert rf.inner_iterations <= 3 * (rf.uzawa_iterations + 2)  # the direct solve
    s = _solver(gale, pb, prec)
    for _ in range(2):
        s.setup(u, p, yield_on=True)  # the coarser level's inverse exists
        v = torch.randn(pb.N * dim, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
        ym, yp = torch.empty_like(v), torch.empty_like(v)
        s.apply_K_moments(v, ym)
        s.apply_K(v, yp)
        s.sync()
        assert rel(ym.cpu().numpy(), yp.cpu().numpy()) < 1e-12  # sums of 64-bit products in another order
        us, ps, rs = _solve(s)
        assert rs.inner_iterations == rf.inner_iterations
        assert np.array_equal(us, uf) and np.array_equal(ps, pf)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dim", [2, 3])
def test_failed_setup_leaves_no_trace(gale, dim, prec):
    import torch
    pb, u, p = _problem(gale, dim, True)
    uf, pf, rf = _solve(_solver(gale, pb, prec))
    for solved_before in (False, True):
        s = _solver(gale, pb, prec)
        if solved_before:
            _solve(s)
        with pytest.raises(gale.GaleError) as e:
            s.setup(u, p, yield_on=True)
        assert e.value.status == gale.E_NAN
        # both forms of the operator are of the same field: the failed setup's,
        # without any stiffness, or, where none had succeeded before, that of a
        # setup of their own, in which nothing yields
        v = torch.randn(pb.N * dim, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
        ym, yp = torch.empty_like(v), torch.empty_like(v)
        s.apply_K_moments(v, ym)
        s.apply_K(v, yp)
        s.sync()
        ym, yp = ym.cpu().numpy(), yp.cpu().numpy()
        if solved_before:
            assert not ym.any() and not yp.any()
            assert s.Solve(raise_on_error=False)[2].status == gale.E_NAN
        else:
            assert yp.any() and rel(ym, yp) < 1e-12
        us, ps, rs = _solve(s)
        assert rs.inner_iterations == rf.inner_iterations
        assert np.array_equal(us, uf) and np.array_equal(ps, pf)
