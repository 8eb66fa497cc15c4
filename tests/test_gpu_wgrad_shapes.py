"""Weight and bias gradients on grids where the padded channel-major layout
has edges: one sample and several, unequal axes, a bottom level of one voxel,
row lengths that are and are not multiples of the 32-voxel step.  Biases keep
every ReLU active, so no mask can flip: device and oracle differ by the BF16
roundings of the intermediate gradients that land on the other side of a tie
(2^-9 relative, few of them), and a wrong index is an O(1) difference in its
layer; the bounds are those of the affine-regime backward test."""
import numpy as np
import pytest

from conftest import rel
from oracle import lpc_net as N

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,nx,ny,nz", [(1, 16, 16, 16), (3, 16, 32, 16), (2, 48, 16, 32), (5, 16, 16, 16)])
def test_backward_matches_oracle(gale, B, nx, ny, nz):
    import torch
    net = gale.LearnedPreconditioner(seed=5)
    P = net.get_params()
    sl = N.layer_slices()[0]
    for l, (a, b) in enumerate(sl):
        P[a] *= 0.02
        P[b] = 5.0 if l < N.NL - 1 else 0.05
    net.set_params(P)
    rng = np.random.default_rng(100 * B + nx + ny + nz)
    x = rng.standard_normal((B, nz, ny, nx, 2)).astype(np.float32)
    gout = rng.standard_normal((B, nz, ny, nx)).astype(np.float32)
    d_in, d_go = torch.from_numpy(x).cuda(), torch.from_numpy(gout).cuda()
    g = net.backward(d_in, d_go)
    assert np.array_equal(g, net.backward(d_in, d_go))  # fixed summation order
    _, cache = N.forward(P, x, mimic=True)
    gref = N.backward(P, cache, gout.astype(np.float64))
    assert rel(g, gref) < 2e-3, rel(g, gref)
    for l, (a, b) in enumerate(sl):
        assert rel(g[a], gref[a]) < 1e-2, (l, "W", rel(g[a], gref[a]))
        assert rel(g[b], gref[b]) < 1e-2, (l, "b", rel(g[b], gref[b]))
