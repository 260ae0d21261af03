"""The flow evaluator's launch forms against the FP64 oracle: targets shared by
a workgroup's waves or two per lane, sources undivided or divided between
workgroups (partial last chunks and batches, a chunk boundary inside either
class, one point, one source), every block size and mode, and captured
evaluations.

Tolerances: FP64 sums of n terms in another order differ from the oracle's by
at most ~n eps times the terms' sum, in norm well under 1e-13 at these sizes;
1e-12 is the evaluator's FP64 bar.  FP32 tiles carry ~6e-8 per operation over
~30 operations, partly averaged out: 2e-6 bounds it at sizes down to one source."""
import numpy as np
import pytest

from oracle import oracle as O
from timfilsimmod_amd import _lib as L
from timfilsimmod_amd.flow import RPY, STOKESLET_ROTLET, FlowFieldEvaluator

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def make(ns, nb, nt, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-20, 20, 3 * ns), rng.standard_normal(6 * ns), rng.uniform(-20, 20, 3 * nb),
            rng.standard_normal(3 * nb), np.zeros(3), rng.uniform(-25, 25, 3 * nt))


@pytest.mark.parametrize("ns,nb,nt", [(1, 0, 1), (0, 1, 63), (1, 1, 64), (127, 1, 65), (129, 300, 130), (640, 1000, 1000),
                                      (300, 4000, 2049), (2500, 37, 10007)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("mode,block", [("stokeslet", 256), ("stokeslet", 64), ("rpy", 128)])
def test_shared_targets_match_oracle(ns, nb, nt, precision, mode, block):
    print(f"case ns={ns} nb={nb} nt={nt} {precision} {mode} block={block}", flush=True)
    xs, fs, xb, fb, xc, pts = make(ns, nb, nt, 5)
    if nb == 0:                      # no blobs: the half-space images
        xs.reshape(-1, 3)[:, 2] = np.abs(xs.reshape(-1, 3)[:, 2]) + 2.0
        pts.reshape(-1, 3)[:, 2] = np.abs(pts.reshape(-1, 3)[:, 2])
    remove = mode == "stokeslet" and nb > 0
    ev = FlowFieldEvaluator(1, ns, nb, mode=STOKESLET_ROTLET if mode == "stokeslet" else RPY, precision=precision,
                            remove_net_force=remove)
    try:
        ev.set_block(block)
        ev.set_sources(xs, fs, xb, fb, xc)
        got = ev.velocities(pts)
        again = ev.velocities(pts)
        assert ev.last_kernel_ms() > 0.0
    finally:
        ev.close()
    ref = (O.flow_velocities(pts, xs, fs, xb, fb, xc, num_bodies=1, remove_net_force=remove) if mode == "stokeslet" else
           O.flow_rpy(pts, xs, fs, xb, fb))
    assert np.array_equal(got, again)
    assert rel(got, ref) <= (1e-12 if precision == "fp64" else 2e-6)


@pytest.mark.parametrize("nt", [700003, 540001])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_divided_sources_of_own_targets_match_oracle(nt, precision):
    """Enough points for two targets per lane; 4,600 sources in several chunks,
    one with a boundary between the classes inside it."""
    print(f"case nt={nt} {precision}", flush=True)
    xs, fs, xb, fb, xc, pts = make(1000, 3600, nt, 6)
    ev = FlowFieldEvaluator(1, 1000, 3600, precision=precision)
    try:
        ev.set_sources(xs, fs, xb, fb, xc)
        got = ev.velocities(pts)
        small = ev.velocities(pts[:3 * 500])         # a smaller call after a larger one
    finally:
        ev.close()
    pick = np.concatenate([np.arange(0, nt, 97), np.arange(nt - 600, nt)])
    ref = O.flow_velocities(np.ascontiguousarray(pts.reshape(-1, 3)[pick].reshape(-1)), xs, fs, xb, fb, xc)
    tol = 1e-12 if precision == "fp64" else 1e-6
    assert rel(got.reshape(-1, 3)[pick].reshape(-1), ref) <= tol
    assert rel(small, got[:1500]) <= tol


def test_captured_evaluation_replays():
    """A captured evaluation holds no buffer that a later, larger call replaces."""
    import torch
    xs, fs, xb, fb, xc, pts = make(640, 1000, 5000, 7)
    dev = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")
    stream = torch.cuda.Stream()
    ev = FlowFieldEvaluator(1, 640, 1000, memory=L.MEMORY_DEVICE, stream=stream.cuda_stream)
    src = [dev(a) for a in (xs, fs, xb, fb, xc)]
    x, v = dev(pts), torch.zeros(15000, dtype=torch.float64, device="cuda")
    big = dev(make(1, 1, 40000, 8)[5])
    vbig = torch.zeros_like(big)
    torch.cuda.synchronize()
    try:
        ev.set_sources(*src)
        ev.velocities(x[:300], torch.empty_like(x[:300]))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ev.velocities(x, v)
        ref = O.flow_velocities(pts, xs, fs, xb, fb, xc)
        for _ in range(3):
            ev.velocities(big, vbig)
            v.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert rel(v.cpu().numpy(), ref) <= 1e-12
    finally:
        ev.close()
