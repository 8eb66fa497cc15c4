"""What the dense inverse of a small mesh takes on the device: 8 bytes an entry
where the mesh is solved directly (in FP64 in both precisions), and 4 more only
where an FP32 V-cycle has it as its coarsest level."""
import gc

import pytest

pytestmark = pytest.mark.gpu


def _bytes_of_setup(gale, res, prec):
    import torch
    dim = len(res)
    lo, hi = (0.0,) * dim, (1.0,) * dim
    coord = gale.layout_random(dim, res, lo, hi, 4, 13)
    mask, vals = gale.free_slip(dim, res)
    pb = gale.Problem(dim, res, lo, hi, coord, [0] * len(coord), [gale.material(density=1.0)], bc_mask=mask,
                      bc_value=vals)
    s = gale.Stokes_SLE_UzawaSolver(pb, gale.uzawa_params(precision=prec))
    s.sync()
    gc.collect()  # no solver of another test is freed in between
    before = torch.cuda.mem_get_info()[0]
    s.setup()
    s.sync()
    used = before - torch.cuda.mem_get_info()[0]
    s.close()
    pb.close()
    return used


@pytest.mark.parametrize("res,prec,entry", [((50, 60), 0, 8), ((50, 60), 1, 8), ((24, 24, 24), 0, 8),
                                            ((24, 24, 24), 1, 12)])
def test_bytes_per_entry(gale, res, prec, entry):
    ld = 6016 if len(res) == 2 else 5632  # 5998 and 5577 free dofs, rows padded to 64
    _bytes_of_setup(gale, res, prec)  # code objects and the first allocations
    used = _bytes_of_setup(gale, res, prec)
    # the levels and the 24^3 level's assembled rows (30 MB) beside it, far less than 4 bytes an entry
    assert entry * ld * ld <= used < entry * ld * ld + (96 << 20)
