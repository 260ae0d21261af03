"""Lock-step cycles replayed in pieces of a few steps: restart lengths below, at
and above a piece and not a multiple of it, with bodies that stop in different
pieces (a small next to a large one, one body whose warm start is already good
enough), against launch-by-launch cycles, bit for bit: the pieces that run after
every body has stopped change nothing.  Norms of bodies of fewer and more rows
than one workgroup takes at a time come with the sizes."""
import numpy as np
import pytest

from timfilsimmod_amd import geometry as G
from timfilsimmod_amd.solver import PRECOND_BLOCKS, SOLVE_FP64, SOLVE_MIXED, EnsembleBeat

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [SOLVE_FP64, SOLVE_MIXED])
@pytest.mark.parametrize("restart", [3, 5, 6, 12, 47])
@pytest.mark.parametrize("sizes", [[(1, 0, 4.0), (9, 900, 14.0)], [(30, 1100, 16.0), (2, 40, 5.0), (4, 0, 8.0)]])
def test_pieces_equal_launch_by_launch(sizes, restart, mode):
    print(f"case bodies={sizes} restart={restart} mode={mode}", flush=True)
    bodies = [G.make_body(nf, 10, nb, r, force_seed=10 + i, perturb_seed=20 + i, centre=(60.0 * i, 0.0, 0.0))
              for i, (nf, nb, r) in enumerate(sizes)]
    out = {}
    for graphs in (True, False):
        ens = EnsembleBeat(bodies, graphs=graphs, mode=mode, restart=restart, tol=1e-8, inner_tol=1e-3,
                           max_refinements=30, max_cycles=200, precond=PRECOND_BLOCKS)
        try:
            for _ in range(2):
                assert ens.step()["converged"] == 1
            out[graphs] = ens.state(), ens.body_stats()
        finally:
            ens.close()
    (sg, bg), (se, be) = out[True], out[False]
    assert bg["graph_cycles"] > 0 and be["eager_cycles"] > 0
    assert np.array_equal(bg["iterations"], be["iterations"])
    for key in ("phase", "angle", "x_segs", "solution"):
        assert np.array_equal(sg[key], se[key]), key
