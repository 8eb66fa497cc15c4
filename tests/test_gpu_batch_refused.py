"""Batched solves of meshes that do not coarsen: up to 2000 free dofs their
inverse is the V-cycle's only level and is rounded to FP32, so contrast costs
inner iterations; the solutions are still the single-problem solver's.  From
2001 to 6000 free dofs such a batch is refused, beyond that it is smoothed."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


def _problem(gale, nx, ny, contrast=1.0):
    coord = gale.layout_random(2, (nx, ny), (0.0, 0.0), (1.0, 1.0), 6, 101)
    mat = gale.shape_layout(2, coord, [gale.everywhere(0), gale.sphere(1, (0.45, 0.6, 0.0), 0.2)])
    mask, vals = gale.free_slip(2, (nx, ny))
    return mask, dict(dim=2, res=(nx, ny), lo=(0.0, 0.0), hi=(1.0, 1.0), coord=coord, material_index=mat,
                      materials=[gale.material(density=1.0), gale.material(eta0=contrast, density=1.1)], bc_mask=mask,
                      bc_value=vals)


@pytest.mark.parametrize("nx,ny,nfree,accepted", [
    (7, 143, 2000, True), (3, 334, 2002, False), (31, 33, 2044, False), (45, 45, 4048, False), (43, 69, 5932, False),
    (19, 158, 6002, True),
    (46, 62, 5702, True),   # coarsens to 23 x 31, 1424 free dofs
    (62, 66, 8182, False),  # coarsens to 31 x 33, 2044 free dofs
])
def test_which_meshes_are_accepted(gale, nx, ny, nfree, accepted):
    mask, kw = _problem(gale, nx, ny)
    assert int((mask == 0).sum()) == nfree
    if accepted:
        gale.BatchSolver([kw]).close()
    else:
        with pytest.raises(gale.GaleError) as e:
            gale.BatchSolver([kw])
        assert e.value.status == gale.E_INVALID


@pytest.mark.parametrize("relax", [0.0, 0.03])
@pytest.mark.parametrize("contrast", [1e5, 1e6])
def test_contrast_without_a_smoothed_level(gale, contrast, relax):
    meshes = [(5, 7), (13, 40), (31, 31)]
    kws = [_problem(gale, nx, ny, contrast)[1] for nx, ny in meshes]
    bs = gale.BatchSolver(kws)
    # rounding the inverse to FP32 leaves inner solves of at most about 30
    # iterations at 1e6 (FP64: one or two); 200 tells a preconditioner that
    # has stopped working
    st, res, _ = bs.solve(gale.batch_params(tolerance=1e-8, maxIterations=20000, max_inner=200, inner_relax_max=relax))
    assert st == 0 and all(r["status"] == 0 and r["rel_residual"] <= 1e-8 for r in res)
    for i, kw in enumerate(kws):
        u, p = bs.solution(i)
        s = gale.Stokes_SLE_UzawaSolver(gale.Problem(**kw), gale.uzawa_params(tolerance=1e-8, maxIterations=20000,
                                                                              inner_rtol_override=1e-12))
        us, ps, _ = s.Solve()
        assert rel(u, us) < 1e-4 and rel(p - p.mean(), ps - ps.mean()) < 1e-4, (meshes[i], rel(u, us))
