"""Several threads read the particles of one problem at once (the library is
called without the interpreter lock): each gets what a single reader gets, for
every combination of outputs and both kinds of weights."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,res,weights", [(2, (60, 40), "voronoi"), (3, (16, 12, 20), "constant")])
def test_concurrent_read_back(gale, dim, res, weights):
    lo, hi = (0.0,) * dim, (1.0,) * dim
    coord = gale.layout_random(dim, res, lo, hi, 20, 5)
    coord = coord[np.random.default_rng(2).permutation(len(coord))]
    pb = gale.Problem(dim, res, lo, hi, coord, np.zeros(len(coord), np.int32), [gale.material()])
    if weights == "voronoi":
        pb.set_weights(gale.WEIGHTS_DVC)
    ref = pb.particles()
    assert np.array_equal(ref[0], coord)
    wrong = []

    def read(t):
        for k in range(30):
            want = (t + k) % 15 + 1  # which of the four outputs
            out = [np.full_like(r, 77) if (want >> i) & 1 else None for i, r in enumerate(ref)]
            st = gale.lib().gs_problem_particles(pb._h, *[None if o is None else o.ctypes.data_as(ctypes.c_void_p)
                                                          for o in out])
            if st != 0 or any(o is not None and not np.array_equal(o, r) for o, r in zip(out, ref)):
                wrong.append((t, k, want, st))

    threads = [threading.Thread(target=read, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
