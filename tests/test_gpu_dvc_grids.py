"""Voronoi weights on sub-grids around the bound between the two ways of
dealing sub-cells to lanes (256 sub-cells), from one sub-cell up, with more
particles than lanes and many in the same sub-cell: integer work, so equal to
the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,res", [(2, (1, 1)), (2, (1, 5)), (2, (8, 8)), (2, (16, 16)), (2, (15, 17)), (2, (29, 9)),
                                     (2, (17, 16)), (3, (1, 1, 1)), (3, (4, 8, 8)), (3, (6, 6, 7)), (3, (6, 6, 8))])
def test_grids_bit_exact(gale, oracle, dim, res):
    rng = np.random.default_rng(sum(res))
    counts = rng.integers(1, 40, size=40)
    counts[:4] = (1, 64, 65, 150)
    off = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    xi = rng.uniform(-1.0, 1.0, (off[-1], dim))
    xi[off[4]:off[8]] *= 0.05  # crowded around the centre: shared seeds
    xi[off[9]:off[10]] = xi[off[9]]  # every particle of a cell at one point
    cent, w = gale.dvc_cells(dim, res, off, xi)
    for e in range(len(counts)):
        sl = slice(off[e], off[e + 1])
        oc, ow = oracle.dvc_cell(dim, res, xi[sl])
        assert np.array_equal(cent[sl], oc) and np.array_equal(w[sl], ow), e
