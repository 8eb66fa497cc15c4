"""A captured relaxed solve holds the addresses of its direction rings.  When
another window has replaced them in between (an eager solve, the autotuner),
the next graph solve captures anew instead of replaying with the freed rings:
every replay gives the eager solve's bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("other", ["solve", "autotune"])
def test_graph_survives_another_window(gale, other):
    from gale_amd import configs
    cfgs = configs.sinker_batch(count=6, seed=81, ppc=8, res_range=(16, 32))
    bs = gale.BatchSolver([c.problem_kwargs() for c in cfgs])

    def prm(window, graph):
        return gale.batch_params(tolerance=1e-6, inner_relax_max=0.03, flexible_window=window, use_graph=graph)

    def solutions():
        return [bs.solution(i) for i in range(len(cfgs))]

    bs.solve(prm(8, False))
    ref = solutions()
    shape = (512, 32)
    for window in (4, 16, 4):
        bs.set_tile(*shape)
        for _ in range(2):  # capture, replay
            st, res, _ = bs.solve(prm(8, True))
            assert st == 0 and all(r["status"] == 0 for r in res)
            for (u, p), (ur, pr) in zip(solutions(), ref):
                assert np.array_equal(u, ur) and np.array_equal(p, pr)
        if other == "solve":
            bs.solve(prm(window, False))
        else:
            bs.autotune(prm(window, False))
