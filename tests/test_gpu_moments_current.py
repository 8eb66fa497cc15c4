"""The moment form of K is that of the solver's last setup also where the
inner solves do not use the multigrid levels (Jacobi): after a setup that
yields, after one that does not, and again."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,res", [(2, (12, 9)), (3, (8, 6, 10))])
def test_moment_apply_follows_each_setup(gale, dim, res):
    import torch
    lo, hi = (0.0,) * dim, (1.0,) * dim
    coord = gale.layout_random(dim, res, lo, hi, 6, 13)
    mask, vals = gale.free_slip(dim, res)
    pb = gale.Problem(dim, res, lo, hi, coord, np.zeros(len(coord), np.int32),
                      [gale.material(eta0=10.0, density=1.0, yield_type=2, cohesion=0.1, min_viscosity=0.01)],
                      bc_mask=mask, bc_value=vals)
    s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(inner_preconditioner=gale.INNER_JACOBI))
    u, p = np.random.default_rng(3).standard_normal(pb.N * dim), np.zeros(pb.E)
    v = torch.randn(pb.N * dim, dtype=torch.float64, device="cuda", generator=torch.Generator("cuda").manual_seed(1))
    norms = []
    for yields in (True, False, True):
        s.setup(u, p, yield_on=True) if yields else s.setup()
        ym, yp = torch.empty_like(v), torch.empty_like(v)
        s.apply_K_moments(v, ym)
        s.apply_K(v, yp)
        s.sync()
        assert rel(ym.cpu().numpy(), yp.cpu().numpy()) < 1e-12  # sums of 64-bit products in another order
        norms.append(float(yp.norm()))
    assert norms[0] < 0.5 * norms[1] and norms[2] == norms[0]
