"""A grid whose network buffers do not fit on the device is refused each time it
is asked for (no kernel runs on the buffers that did fit), gives back what it
had taken, and leaves the network usable."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_refused_each_time(gale):
    import torch
    net = gale.LearnedPreconditioner()
    net.set_params(np.load(os.path.join(os.path.dirname(gale.__file__), "lpc_weights.npy"), allow_pickle=False))
    inp = torch.randn((1, 16, 16, 16, 2), dtype=torch.float32, device="cuda",
                      generator=torch.Generator("cuda").manual_seed(1))
    ref, out = torch.empty((1, 16, 16, 16), device="cuda"), torch.empty((1, 16, 16, 16), device="cuda")
    net.forward(inp, ref)
    free = torch.cuda.mem_get_info()[0]
    n = 2160  # the input takes 81 GB, the first layer's output 322 GB: more than the device has
    assert 32 * n ** 3 > torch.cuda.mem_get_info()[1]
    for _ in range(3):
        st = gale.lib().gs_lpc_forward(net._h, n, n, n, 1, inp.data_ptr(), out.data_ptr())
        assert st == gale.E_HIP
        assert torch.cuda.mem_get_info()[0] >= free
    net.forward(inp, out)
    assert torch.equal(out, ref)
