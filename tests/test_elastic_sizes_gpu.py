"""The launches that an elastic step's iterations are made of, at the sizes where
they change: filaments of up to 64 segments (update, robot arm and forces in
one launch) and longer ones, residuals of up to 1,024 rows (flags set by the
residual's own workgroup) and longer ones, one filament of two segments.  Each
step is taken with the Broyden step in two launches and, with a loop allowed
one iteration more than the engine holds, with the end of an iteration and the
update one after the other: the same iterations in exact arithmetic.

Tolerance: both converge to residuals below tol, and the first iterates differ
by rounding only; the iterations contract, so the states agree to tol times the
segment length (positions) with a factor 10 for the inverse Jacobian."""
import numpy as np
import pytest
import torch
from scipy.spatial.transform import Rotation

from timfilsimmod_amd import _lib as L
from timfilsimmod_amd import filament as FM
from timfilsimmod_amd import geometry as G
from timfilsimmod_amd.broyden import BroydenSolver
from timfilsimmod_amd.solver import BLOB_DIRECT, SOLVE_FP64, ElasticVelocities

pytestmark = pytest.mark.gpu

MAX_ITER, TOL, DL = 200, 1e-6, 2.2


def dev(a):
    return torch.tensor(np.asarray(a, dtype=np.float64), device="cuda")


def run(nfil, nseg, nb, radius, graphs, loop_iters):
    body = G.make_body(nfil, nseg, nb, radius)
    kb = 18.0 if nseg > 2 else 180.0     # soft enough for J0 to lead the way
    efm = 20.0 * kb / (DL * DL * nseg * nseg)
    q0 = np.array([np.roll(Rotation.align_vectors([n], [[1.0, 0.0, 0.0]])[0].as_quat(), 1) for n in body.fil_normal])
    pert = np.random.default_rng(0).standard_normal((nfil, 6)) * 0.1 * efm
    ts = torch.cuda.Stream()
    handles = []
    with torch.cuda.stream(ts):
        try:
            kw = dict(memory=L.MEMORY_DEVICE, stream=ts.cuda_stream)
            model = FM.FilamentModel(1, nfil, nseg, dl=DL, kb=kb, kt=kb, dt=0.01, end_force=efm, **kw)
            handles.append(model)
            model.set_state(dev(body.fil_base.reshape(-1)), dev(np.repeat(q0[:, None, :], nseg, axis=1).reshape(-1)))
            model.set_perturbation(nseg // 2, nseg - 1, dev(pert.reshape(-1)))
            ev = ElasticVelocities(1, nfil * nseg, nb, mode=SOLVE_FP64, restart=30, max_cycles=200, tol=1e-10, **kw)
            handles.append(ev)
            ev.set_preconditioner(BLOB_DIRECT)
            eng = BroydenSolver(model.block_sizes(), max_iter=MAX_ITER, **kw)
            handles.append(eng)
            f_blobs = dev(np.zeros(3 * nb))
            keep = [dev(body.x_blobs), dev(np.zeros(3)), dev(np.zeros(6))]
            step = FM.ElasticStep(model, ev, eng, *keep, f_blobs, tol=TOL, max_iter=loop_iters)
            handles.append(step)
            step.set_graphs(graphs)
            st = step.step(0)
            torch.cuda.synchronize()
            return st, model.read(FM.X), f_blobs.cpu().numpy()
        finally:
            for h in reversed(handles):
                h.close()


@pytest.mark.parametrize("nfil,nseg,nb,radius", [(1, 2, 20, 4.0), (3, 63, 60, 6.0), (2, 64, 60, 6.0), (2, 65, 60, 6.0),
                                                 (31, 33, 70, 20.0), (32, 32, 70, 20.0)])
def test_step_in_two_launches_equals_the_parts(nfil, nseg, nb, radius):
    print(f"case {nfil} x {nseg} segments + {nb} blobs", flush=True)
    plain, x_p, f_p = run(nfil, nseg, nb, radius, True, MAX_ITER + 1)
    for graphs in (True, False):
        st, x, f = run(nfil, nseg, nb, radius, graphs, MAX_ITER)
        print(f"  graphs {graphs}: iterations {st['broyden_iterations']} ({plain['broyden_iterations']}), positions differ by "
              f"{np.abs(x - x_p).max():.1e}", flush=True)
        assert st["converged"] == plain["converged"] == 1
        assert abs(st["broyden_iterations"] - plain["broyden_iterations"]) <= 1
        assert np.abs(x - x_p).max() <= 10.0 * TOL * DL
        assert np.linalg.norm(f - f_p) <= 1e-3 * np.linalg.norm(f_p)
