"""Batched solves of meshes that take each branch of the in-workgroup V-cycle:
a dense coarsest solve with its columns split over spare threads, one with
more rows than threads, one on the mesh itself (it does not coarsen), and a
coarsest level too large for it (Chebyshev smoothing only); every instance
against the single-problem solver (which solves these meshes directly) at the
batched parity tests' tolerance."""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

MESHES = [(5, 7), (2, 2), (16, 16), (24, 24), (22, 26), (34, 34), (13, 40), (63, 61)]


def _problem(gale, nx, ny, i):
    coord = gale.layout_random(2, (nx, ny), (0.0, 0.0), (1.0, 1.0), 6, 100 + i)
    mat = gale.shape_layout(2, coord, [gale.everywhere(0), gale.sphere(1, (0.45, 0.6, 0.0), 0.2)])
    mask, vals = gale.free_slip(2, (nx, ny))
    return dict(dim=2, res=(nx, ny), lo=(0.0, 0.0), hi=(1.0, 1.0), coord=coord, material_index=mat,
                materials=[gale.material(density=1.0), gale.material(eta0=100.0, density=1.1)], bc_mask=mask,
                bc_value=vals)


@pytest.mark.parametrize("relax", [0.0, 0.03])
@pytest.mark.parametrize("block,tx", [(256, 16), (512, 32), (1024, 64)])
def test_batch_branches(gale, block, tx, relax):
    kws = [_problem(gale, nx, ny, i) for i, (nx, ny) in enumerate(MESHES)]
    bs = gale.BatchSolver(kws)
    bs.set_tile(block, tx)
    prm = gale.batch_params(tolerance=1e-10, inner_rtol_factor=1e-3, maxIterations=20000, inner_relax_max=relax)
    bs.solve(prm)
    for i, kw in enumerate(kws):
        u, p = bs.solution(i)
        pb = gale.Problem(**kw)
        s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(tolerance=1e-10, inner_rtol_override=1e-13,
                                                              inner_max_iterations=200000, maxIterations=20000))
        us, ps, _ = s.Solve()
        assert rel(u, us) < 1e-7, (MESHES[i], rel(u, us))
        assert rel(p - p.mean(), ps - ps.mean()) < 1e-6, (MESHES[i], rel(p - p.mean(), ps - ps.mean()))


def test_autotune_times_each_block_size_once(gale):
    """The two widths of a block size are one kernel: one time for both, and
    the fastest block size at its first width."""
    bs = gale.BatchSolver([_problem(gale, nx, ny, i) for i, (nx, ny) in enumerate([(16, 16), (24, 24)])])
    best, ms = bs.autotune(gale.batch_params(tolerance=1e-6))
    t = [ms[c] for c in gale.TILE_CANDIDATES]
    assert t[0] == t[1] and t[2] == t[3] and t[4] == t[5] and min(t) > 0
    assert best == gale.TILE_CANDIDATES[t.index(min(t))]
