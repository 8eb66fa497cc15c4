"""The parts of a multigrid setup do not depend on one another's scratch: the
operator, the smoothing bounds and the inverse of a second setup in the same
buffers, after solves and applies have used them, give the first one's bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dim,res", [(2, (64, 80)), (3, (16, 20, 16)), (3, (9, 21, 17))])
def test_setup_repeats(gale, dim, res, prec):
    lo, hi = (0.0,) * dim, (1.0,) * dim
    coord = gale.layout_random(dim, res, lo, hi, 5, 13)
    mat = gale.shape_layout(dim, coord, [gale.everywhere(0), gale.sphere(1, (0.5, 0.55, 0.5), 0.3)])
    mask, vals = gale.free_slip(dim, res)
    pb = gale.Problem(dim, res, lo, hi, coord, mat, [gale.material(density=1.0), gale.material(eta0=50.0, density=1.2)],
                      bc_mask=mask, bc_value=vals)
    s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(tolerance=1e-6, precision=prec, maxIterations=5000))
    out = []
    for _ in range(2):
        s.set_pressure(None)
        s.setup()
        u, p, rep = s.Solve()
        out.append((u, p, rep.inner_iterations))
    assert out[0][2] == out[1][2] and np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
