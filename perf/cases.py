"""The work that a user of this framework has it do, as measured cases.

Seven kinds of call, all through the package's public entry points:

* ``mobility``  the drop-in back-end class: host arrays in, one full mobility evaluation, host arrays
  out, at positions that moved since the last call (an elastic model's velocity evaluation);
* ``matvec``    one block product at new positions with everything resident on the GPU, for one body
  or for independent bodies of uneven size, 6- or 3-component segments, FP64 or FP32 tiles;
* ``wall``      the same above a no-slip wall (filaments on a plane, no blobs);
* ``beat``      a prescribed-beat run taken up from a saved state for a few timesteps (each one
  saddle-point GMRES solve), mixed precision or FP64;
* ``ensemble``  the same for independent bodies of uneven size solved in lock-step;
* ``flow``      flow-field velocities at a plane of points or at scattered tracers;
* ``elastic``   one implicit timestep of the Cosserat filament model, Broyden to 1e-8.

Sizes are those of the package's own configurations: the small body (16 filaments x 20 segments,
2,000 blobs), the production body (640 x 20, 9,000 blobs), the flow-source body (1,280 x 20, 9,000
blobs), the uneven ensemble, and odd sizes between them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from timfilsimmod_amd import _lib as L
from timfilsimmod_amd import filament as FM
from timfilsimmod_amd import geometry as G
from timfilsimmod_amd import solver as S
from timfilsimmod_amd.broyden import BroydenSolver
from timfilsimmod_amd.flow import RPY, STOKESLET_ROTLET, FlowFieldEvaluator
from timfilsimmod_amd.mobility import RpyHandle, RpyMobilitySolver

PRECISION = {"fp64": L.PRECISION_FP64, "fp32": L.PRECISION_FP32_ACC64}
AREA_PER_BLOB = 4.0 * math.pi * 50.0**2 / 9000.0    # the production body's, as in geometry.ensemble_sizes


def listed():
    return [
        # one velocity evaluation of a small elastic body through the drop-in class: the smallest call
        {"name": "mobility_small_fp64", "kind": "mobility", "num_fil": 16, "num_seg": 20, "num_blobs": 2000,
         "precision": "fp64"},
        # an ordinary body of odd size in the faster precision
        {"name": "matvec_odd_fp32", "kind": "matvec", "bodies": 1, "num_fil": 107, "num_seg": 23,
         "num_blobs": 3333, "seg_dof": 6, "precision": "fp32"},
        # the benchmark's 6-component product of the production body, both precisions
        {"name": "matvec_body_fp64", "kind": "matvec", "bodies": 1, "num_fil": 640, "num_seg": 20,
         "num_blobs": 9000, "seg_dof": 6, "precision": "fp64"},
        {"name": "matvec_body_fp32", "kind": "matvec", "bodies": 1, "num_fil": 640, "num_seg": 20,
         "num_blobs": 9000, "seg_dof": 6, "precision": "fp32"},
        # many independent bodies of uneven size in one product
        {"name": "matvec_bodies_fp32", "kind": "matvec", "bodies": 12, "num_fil": 1000, "num_seg": 20,
         "num_blobs": 9000, "seg_dof": 6, "precision": "fp32"},
        # a carpet of filaments above a no-slip wall
        {"name": "wall_carpet_fp64", "kind": "wall", "num_fil": 256, "num_seg": 20, "seg_dof": 6,
         "precision": "fp64"},
        # the headline timestep, both precisions
        {"name": "beat_body_mixed", "kind": "beat", "num_fil": 640, "num_seg": 20, "num_blobs": 9000,
         "mode": "mixed", "steps": 4},
        {"name": "beat_body_fp64", "kind": "beat", "num_fil": 640, "num_seg": 20, "num_blobs": 9000,
         "mode": "fp64", "steps": 4},
        # uneven bodies beating side by side
        {"name": "ensemble_mixed", "kind": "ensemble", "bodies": 6, "num_fil": 400, "num_seg": 20,
         "num_blobs": 5000, "mode": "mixed", "steps": 3},
        # the flow field of a large body at a plane of points, for a picture
        {"name": "flow_plane_fp32", "kind": "flow", "num_fil": 1280, "num_seg": 20, "num_blobs": 9000,
         "points": "plane", "num_points": 1000000, "mode": "stokeslet", "precision": "fp32"},
        # an odd number of tracers advected around a small body
        {"name": "flow_tracers_fp64", "kind": "flow", "num_fil": 16, "num_seg": 20, "num_blobs": 2000,
         "points": "scattered", "num_points": 10007, "mode": "stokeslet", "precision": "fp64"},
        # one implicit step of the elastic model on a body held still
        {"name": "elastic_small", "kind": "elastic", "num_fil": 16, "num_seg": 20, "num_blobs": 2000},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    kind = rng.choice(["mobility", "matvec", "matvec", "bodies", "wall", "beat", "ensemble", "flow", "flow", "elastic"])
    prec = rng.choice(["fp64", "fp32"])
    if kind == "mobility":
        return {"kind": kind, "num_fil": log(4, 200), "num_seg": rng.randint(8, 30), "num_blobs": log(200, 4000),
                "precision": prec}
    if kind == "matvec":
        return {"kind": kind, "bodies": 1, "num_fil": log(8, 600), "num_seg": rng.randint(10, 21),
                "num_blobs": log(200, 9000), "seg_dof": rng.choice([6, 6, 3]), "precision": prec}
    if kind == "bodies":
        return {"kind": "matvec", "bodies": rng.randint(2, 11), "num_fil": log(40, 500), "num_seg": rng.randint(10, 21),
                "num_blobs": log(800, 6000), "seg_dof": rng.choice([6, 6, 3]), "precision": prec}
    if kind == "wall":
        return {"kind": kind, "num_fil": log(5, 250), "num_seg": rng.randint(6, 20), "seg_dof": rng.choice([6, 3]),
                "precision": prec}
    if kind == "beat":
        return {"kind": kind, "num_fil": log(20, 500), "num_seg": rng.randint(10, 20), "num_blobs": log(500, 8000),
                "mode": rng.choice(["mixed", "fp64"]), "steps": rng.randint(2, 4)}
    if kind == "ensemble":
        return {"kind": kind, "bodies": rng.randint(2, 5), "num_fil": log(40, 300), "num_seg": rng.randint(12, 20),
                "num_blobs": log(600, 4000), "mode": rng.choice(["mixed", "mixed", "fp64"]), "steps": 2}
    if kind == "flow":
        return {"kind": kind, "num_fil": log(8, 900), "num_seg": rng.randint(10, 21), "num_blobs": log(300, 9000),
                "points": rng.choice(["plane", "scattered"]), "num_points": log(1000, 300000),
                "mode": rng.choice(["stokeslet", "stokeslet", "rpy"]), "precision": prec}
    return {"kind": "elastic", "num_fil": rng.randint(4, 16), "num_seg": rng.randint(14, 20), "num_blobs": log(300, 2000)}


# ---------------------------------------------------------------- inputs

def _body(num_fil, num_seg, num_blobs, seed, centre=(0.0, 0.0, 0.0)):
    radius = math.sqrt(max(num_blobs, 200) * AREA_PER_BLOB / (4.0 * math.pi))
    return G.make_body(num_fil, num_seg, num_blobs, radius, force_seed=2 * seed + 11, perturb_seed=2 * seed + 12,
                       centre=centre)


def _bodies(case, seed):
    """One body of the case's size, or `bodies` of them with filament and blob counts uniform between
    a tenth (segments) and a quarter (blobs) of it and all of it, well apart."""
    if case.get("bodies", 1) == 1:
        return [_body(case["num_fil"], case["num_seg"], case["num_blobs"], seed)]
    sizes = np.random.default_rng([7, case["bodies"], case["num_fil"], case["num_blobs"]])
    out = []
    for b in range(case["bodies"]):
        nf = int(sizes.integers(max(2, case["num_fil"] // 10), case["num_fil"] + 1))
        nb = int(sizes.integers(max(100, case["num_blobs"] // 4), case["num_blobs"] + 1))
        out.append(_body(nf, case["num_seg"], nb, 100 * seed + b, centre=(400.0 * (b % 4), 400.0 * (b // 4), 0.0)))
    return out


def _dev(a):
    return torch.tensor(np.asarray(a, dtype=np.float64), device="cuda")


def _carpet(case, seed):
    """Filaments standing on a jittered grid above the wall z = 0: x_segs, f_segs."""
    rng = np.random.default_rng([31, seed])
    nf, ns = case["num_fil"], case["num_seg"]
    side = int(math.ceil(math.sqrt(nf)))
    base = np.stack([np.arange(nf) % side, np.arange(nf) // side], axis=1) * 8.0 + rng.uniform(-1.5, 1.5, (nf, 2))
    lean = rng.normal(0.0, 0.25, (nf, 2))
    z = 1.6 + 2.2 * np.arange(ns)
    x = np.empty((nf, ns, 3))
    x[..., :2] = base[:, None, :] + lean[:, None, :] * (z[None, :, None] - 1.6)
    x[..., 2] = z
    x += rng.normal(0.0, 0.05, x.shape)
    return x.reshape(-1), rng.standard_normal(6 * nf * ns)


def _points(case, seed):
    """A square grid on the plane z = 0 through the body, or scattered tracers outside its surface."""
    n = case["num_points"]
    radius = math.sqrt(max(case["num_blobs"], 200) * AREA_PER_BLOB / (4.0 * math.pi))
    half = radius + 1.2 * 2.2 * (case["num_seg"] - 1)
    rng = np.random.default_rng([53, seed])
    if case["points"] == "plane":
        side = int(math.ceil(math.sqrt(n)))
        t = np.linspace(-half, half, side)
        pts = np.zeros((side * side, 3))
        pts[:, 0], pts[:, 1] = np.tile(t, side), np.repeat(t, side)
        pts[:, 2] = 0.05 * rng.uniform(-1.0, 1.0)      # the plane's height differs from one picture to the next
        return pts[:n].reshape(-1)
    u = rng.standard_normal((n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    return (u * rng.uniform(radius + 1.5, half, (n, 1))).reshape(-1)


def _elastic(case, seed):
    """The elastic step of bench.py's elastic leg: a body held still, blob forces from the dense inverse."""
    from scipy.spatial.transform import Rotation
    nfil, nseg, nb = case["num_fil"], case["num_seg"], case["num_blobs"]
    body = _body(nfil, nseg, nb, seed)
    dl, kb = 2.2, 1800.0
    end = 220.0 * kb / (dl * dl * nseg * nseg)
    ex = np.array([1.0, 0.0, 0.0])
    q0 = np.array([np.roll(Rotation.align_vectors([n], [ex])[0].as_quat(), 1) for n in body.fil_normal])
    qs = np.repeat(q0[:, None, :], nseg, axis=1)
    kick = np.random.default_rng([71, seed]).standard_normal((nfil, 6)) * 0.1 * end
    stream = _stream()
    model = FM.FilamentModel(1, nfil, nseg, dl=dl, kb=kb, kt=kb, dt=0.1, end_force=end, memory=L.MEMORY_DEVICE,
                             stream=stream)
    vel = S.ElasticVelocities(1, nfil * nseg, nb, mode=S.SOLVE_FP64, restart=30, max_cycles=200, tol=1e-10,
                              memory=L.MEMORY_DEVICE, stream=stream)
    vel.set_preconditioner(S.BLOB_DIRECT)
    engine = BroydenSolver(model.block_sizes(), memory=L.MEMORY_DEVICE, stream=stream)
    f_blobs = _dev(np.zeros(3 * nb))
    keep = [_dev(body.x_blobs), _dev(np.zeros(3)), _dev(np.zeros(6)), _dev(body.fil_base.reshape(-1)),
            _dev(qs.reshape(-1)), _dev(kick.reshape(-1))]
    torch.cuda.synchronize()
    model.set_state(keep[3], keep[4])
    model.set_perturbation(min(4, nseg - 2), min(12, nseg - 1), keep[5])
    step = FM.ElasticStep(model, vel, engine, keep[0], keep[1], keep[2], f_blobs, tol=1e-8, max_iter=400)
    step.step(0)
    step.step(1)
    return {"step": step, "model": model, "f_blobs": f_blobs, "saved": step.backup(), "keep": [keep, vel, engine]}


_STREAM = []


def _stream():
    """The program's working stream (a HIP stream at the default priority)."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0].cuda_stream


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mobility":
        body = _body(case["num_fil"], case["num_seg"], case["num_blobs"], seed)
        m = RpyMobilitySolver(body.num_segs, body.num_blobs, seg_dof=6, precision=case["precision"], bs_accumulate=True)
        m.initialise()
        for dst, src in ((m.x_segs_host, body.x_segs), (m.f_segs_host, body.f_segs), (m.x_blobs_host, body.x_blobs),
                         (m.f_blobs_host, body.f_blobs)):
            dst[:] = src
        return {"kind": kind, "mobility": m}
    if kind == "matvec":
        bodies = _bodies(case, seed)
        ns, nb = sum(b.num_segs for b in bodies), sum(b.num_blobs for b in bodies)
        h = RpyHandle(ns, nb, seg_dof=case["seg_dof"], precision=PRECISION[case["precision"]], bs_accumulate=True,
                      memory=L.MEMORY_DEVICE, stream=_stream())
        if len(bodies) > 1:
            h.set_bodies([b.num_segs for b in bodies], [b.num_blobs for b in bodies])
        cat = {k: _dev(np.concatenate([getattr(b, k) for b in bodies])) for k in ("x_segs", "x_blobs", "f_segs", "f_blobs")}
        v = (torch.zeros(6 * ns, dtype=torch.float64, device="cuda"), torch.zeros(3 * nb, dtype=torch.float64, device="cuda"))
        return {"kind": kind, "handle": h, **cat, "v": v}
    if kind == "wall":
        x, f = _carpet(case, seed)
        ns = x.size // 3
        h = RpyHandle(ns, 0, seg_dof=case["seg_dof"], precision=PRECISION[case["precision"]], bs_accumulate=True,
                      memory=L.MEMORY_DEVICE, stream=_stream())
        h.set_domain(L.DOMAIN_HALF_SPACE)
        return {"kind": kind, "handle": h, "x_segs": _dev(x), "f_segs": _dev(f),
                "v": torch.zeros(6 * ns, dtype=torch.float64, device="cuda")}
    if kind in ("beat", "ensemble"):
        bodies = _bodies(case, seed) if kind == "ensemble" else [_body(case["num_fil"], case["num_seg"], case["num_blobs"], seed)]
        kw = dict(mode=S.SOLVE_MIXED if case["mode"] == "mixed" else S.SOLVE_FP64, tol=1e-8, restart=50, inner_tol=1e-6,
                  max_cycles=40, max_refinements=20, stream=_stream(), warm_start=2, precond=S.PRECOND_BLOCKS)
        setups = [S.beat_setup(b, phase_seed=1000 * seed + 3 + i) for i, b in enumerate(bodies)]
        sim = S.EnsembleBeat(bodies, setups=setups, **kw) if kind == "ensemble" else S.BeatSimulation(bodies[0], setup=setups[0], **kw)
        sim.step()
        sim.step()
        return {"kind": kind, "sim": sim, "saved": sim.state(), "steps": case["steps"]}
    if kind == "flow":
        body = _body(case["num_fil"], case["num_seg"], case["num_blobs"], seed)
        ev = FlowFieldEvaluator(1, body.num_segs, body.num_blobs, mode=RPY if case["mode"] == "rpy" else STOKESLET_ROTLET,
                                precision=case["precision"], memory=L.MEMORY_DEVICE, stream=_stream())
        src = [_dev(a) for a in (body.x_segs, body.f_segs, body.x_blobs, body.f_blobs, body.centre)]
        pts = _dev(_points(case, seed))
        return {"kind": kind, "flow": ev, "sources": src, "points": pts, "out": torch.empty_like(pts)}
    return {"kind": kind, **_elastic(case, seed)}


# ---------------------------------------------------------------- one pass

def run(state):
    kind = state["kind"]
    if kind == "mobility":
        m = state["mobility"]
        m.copy_segment_positions_to_device()
        m.copy_blob_positions_to_device()
        m.copy_segment_forces_to_device()
        m.copy_blob_forces_to_device()
        m.evaluate_full_mobility()
        m.wait_for_device()
        return {"v_segs": m.v_segs_host, "v_blobs": m.v_blobs_host}
    if kind == "matvec":
        h, (vs, vb) = state["handle"], state["v"]
        h.upload(L.SEG_POSITIONS, state["x_segs"])
        h.upload(L.BLOB_POSITIONS, state["x_blobs"])
        h.apply(L.BLOCK_ALL, state["f_segs"], state["f_blobs"], vs, vb)
        return {"v_segs": vs, "v_blobs": vb}
    if kind == "wall":
        h = state["handle"]
        h.upload(L.SEG_POSITIONS, state["x_segs"])
        h.apply(L.BLOCK_SS, state["f_segs"], None, state["v"], None)
        return {"v_segs": state["v"]}
    if kind in ("beat", "ensemble"):
        # a run taken up from its saved state: the first step solves again at the saved phases, from the
        # saved solution, the others advance the beat
        sim, saved = state["sim"], state["saved"]
        sim.restore(saved["phase"], saved["angle"], saved["solution"])
        for _ in range(state["steps"]):
            sim.step()
        return sim.state()
    if kind == "flow":
        ev = state["flow"]
        ev.set_sources(*state["sources"])
        return ev.velocities(state["points"], state["out"])
    step = state["step"]
    step.restore(state["saved"])
    step.step(2)
    return {"state": step.backup(), "f_blobs": state["f_blobs"], "x_segs": state["model"].read(FM.X)}


# ---------------------------------------------------------------- what a pass cannot do without

# Operations per pair, + - x = 1, fused multiply-add = 2, square root and division = 1: the far-field forms.
TT, SS6, SB6, BS6 = 36, 88, 52, 52
WALL_TT, WALL_SS6 = 150, 320
GMRES_STEPS = 40       # iterations that a production body's timestep takes


def _pairs_flops(ns, nb, seg_dof):
    if seg_dof == 6:
        return float(SS6) * ns * ns + float(SB6 + BS6) * ns * nb + float(TT) * nb * nb
    return float(TT) * (ns + nb) ** 2


def work(case):
    kind = case["kind"]
    if kind in ("mobility", "matvec", "beat", "ensemble"):
        dof = 3 if kind in ("beat", "ensemble") else case.get("seg_dof", 6)
        if kind in ("matvec", "ensemble") and case["bodies"] > 1:
            sizes = [(b.num_segs, b.num_blobs) for b in _bodies(case, 0)]
        else:
            sizes = [(case["num_fil"] * case["num_seg"], case["num_blobs"])]
        flops = sum(_pairs_flops(ns, nb, dof) for ns, nb in sizes)
        per_seg = 15 if dof == 6 else 9
        moved = sum(8.0 * (per_seg * ns + 9 * nb) for ns, nb in sizes)
        if kind in ("beat", "ensemble"):
            solves = case["steps"] - 1
            return {"bytes": 2.0 * moved * case["steps"], "flops": flops * GMRES_STEPS * solves}
        return {"bytes": moved, "flops": flops}
    if kind == "wall":
        ns = case["num_fil"] * case["num_seg"]
        six = case["seg_dof"] == 6
        return {"bytes": 8.0 * (15 if six else 9) * ns, "flops": float(WALL_SS6 if six else WALL_TT) * ns * ns}
    if kind == "flow":
        ns, nb, nt = case["num_fil"] * case["num_seg"], case["num_blobs"], case["num_points"]
        per = (44.0 * ns + 28.0 * nb) if case["mode"] == "stokeslet" else (float(BS6) * ns + float(TT) * nb)
        return {"bytes": 8.0 * (9 * ns + 6 * nb + 6 * nt), "flops": per * nt}
    ns, nb, iters = case["num_fil"] * case["num_seg"], case["num_blobs"], 55
    inverse = (3.0 * nb) * (3.0 * nb + 1.0) / 2.0     # the blob mobility's, symmetric
    pairs = float(SS6) * ns * ns + float(SB6 + BS6) * ns * nb
    return {"bytes": 8.0 * inverse, "flops": iters * (pairs + 4.0 * inverse)}


def tolerance(case):
    kind = case["kind"]
    if kind == "elastic":
        # Broyden stops at 1e-8: against the same step stopped at 1e-10, blob forces 1.2e-4 (largest 2.4e-3)
        return {"rel": 5e-4, "max": 1e-2}
    if kind in ("beat", "ensemble"):
        # GMRES stops at 1e-8: against the same steps solved to 1e-12, solutions 8e-5 (largest 7e-3)
        return {"rel": 3e-4, "max": 3e-2}
    # direct sums against exact(): FP64 up to 8e-16 (1.5e-15 above the wall), FP32 tiles up to 2.4e-7
    # (3.8e-7 above the wall, 6.5e-7 for the flow field, which has no self terms)
    if case["precision"] == "fp64":
        return {"rel": 6e-15 if kind == "wall" else 3.2e-15}
    return {"rel": {"wall": 1.6e-6, "flow": 2.6e-6}.get(kind, 1e-6)}


# ---------------------------------------------------------------- the same results in 64-bit torch

PI = math.pi


def _cross(a, b):
    return (a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0])


def _rpy_rows(xt, xs, fs, six_out, six_in):
    """Velocities (and angular velocities) of spheres of radius 1 at xt from forces (and torques) fs on
    spheres of radius 1 at xs, viscosity 1: Rotne-Prager-Yamakawa with the overlap forms."""
    d = [xt[:, None, k] - xs[None, :, k] for k in range(3)]
    r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
    r = r2.sqrt()
    far = r > 2.0
    ri = torch.where(r2 > 0, 1.0 / torch.where(r2 > 0, r, torch.ones_like(r)), torch.zeros_like(r))
    e = [c * ri for c in d]
    f = [fs[None, :, k] for k in range(3)]
    c8 = 1.0 / (8.0 * PI)
    A = torch.where(far, c8 * ri * (1.0 + (2.0 / 3.0) * ri * ri), (1.0 - 9.0 / 32.0 * r) / (6.0 * PI))
    B = torch.where(far, c8 * ri * (1.0 - 2.0 * ri * ri), (3.0 / 32.0) * r / (6.0 * PI))
    ef = B * (e[0] * f[0] + e[1] * f[1] + e[2] * f[2])
    out = [(A * f[k] + ef * e[k]).sum(1) for k in range(3)]
    if six_in or six_out:
        C = torch.where(far, c8 * ri * ri, (8.0 * r - 3.0 * r2) / (128.0 * PI))
    if six_in:
        t = [fs[None, :, 3 + k] for k in range(3)]
        for k, c in enumerate(_cross(t, e)):
            out[k] += (C * c).sum(1)
    if six_out:
        w = [(C * c).sum(1) for c in _cross(f, e)]
        if six_in:
            Ar = torch.where(far, -0.5 * c8 * ri**3, (5.0 * r2 * r - 54.0 * r + 64.0) / (512.0 * PI))
            Br = torch.where(far, 1.5 * c8 * ri**3, 3.0 * r * (6.0 - r2) / (512.0 * PI))
            et = Br * (e[0] * t[0] + e[1] * t[1] + e[2] * t[2])
            for k in range(3):
                w[k] += (Ar * t[k] + et * e[k]).sum(1)
        out += w
    return torch.stack(out, dim=1)


def _wall_rows(xt, xs, fs, first, six):
    """The same above a no-slip wall at z = 0 (Swan & Brady 2007; spheres of radius 1, viscosity 1; no
    overlap form); row i is particle first + i of the sources."""
    d = [xt[:, None, k] - xs[None, :, k] for k in range(3)]
    f = [fs[None, :, k] for k in range(3)]
    t = [fs[None, :, 3 + k] for k in range(3)] if six else None
    k6, k8 = 1.0 / (6.0 * PI), 1.0 / (8.0 * PI)
    n = xt.shape[0]
    rows = torch.arange(n, device=xt.device)
    same = torch.zeros((n, xs.shape[0]), dtype=torch.bool, device=xt.device)
    same[rows, first + rows] = True
    r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
    q = 1.0 / torch.where(same, torch.ones_like(r2), r2).sqrt()
    u = [c * q for c in d]
    v = [None] * 3
    uf = u[0] * f[0] + u[1] * f[1] + u[2] * f[2]
    ca, cb, cc = k8 * q, 1.0 + (2.0 / 3.0) * q * q, (1.0 - 2.0 * q * q) * uf
    for k in range(3):
        v[k] = ca * (cb * f[k] + cc * u[k])
    w = [0.0, 0.0, 0.0]
    if six:
        c2 = ca * q
        ut = u[0] * t[0] + u[1] * t[1] + u[2] * t[2]
        tx, fx = _cross(t, u), _cross(f, u)
        for k in range(3):
            v[k] = v[k] + c2 * tx[k]
            w[k] = c2 * fx[k] + 0.5 * c2 * q * (3.0 * ut * u[k] - t[k])
    # image of the source at the mirrored height: separation (dx, dy, zi + zj)
    zi, zj = xt[:, None, 2], xs[None, :, 2]
    rz = zi + zj
    p = 1.0 / (d[0] * d[0] + d[1] * d[1] + rz * rz).sqrt()
    p2, p3, p4, p5 = p**2, p**3, p**4, p**5
    ex, ey, ez = d[0] * p, d[1] * p, rz * p
    z2, h = ez * ez, zj / rz
    ef = ex * f[0] + ey * f[1] + ez * f[2]
    g0 = -(0.75 * p * (1.0 + 2.0 * h * (1.0 - h) * z2) + 0.5 * (p3 * (1.0 - 3.0 * z2) - p5 * (1.0 - 5.0 * z2)))
    g1 = (-(0.75 * p * (1.0 - 6.0 * h * (1.0 - h) * z2) - 1.5 * p3 * (1.0 - 5.0 * z2) + 2.5 * p5 * (1.0 - 7.0 * z2)) * ef
          + ez * f[2] * (1.5 * h * p * (1.0 - 6.0 * (1.0 - h) * z2) - 3.0 * p3 * (1.0 - 5.0 * z2) + 5.0 * p5 * (2.0 - 7.0 * z2)))
    g3 = (1.5 * h * p - 5.0 * p5) * ef
    g4 = -((3.0 * h * h * p + 3.0 * p3) * z2 + (2.0 - 15.0 * z2) * p5) * f[2]
    v[0] = v[0] + k6 * (g0 * f[0] + g1 * ex)
    v[1] = v[1] + k6 * (g0 * f[1] + g1 * ey)
    v[2] = v[2] + k6 * (g0 * f[2] + (g1 + g3) * ez + g4)
    if six:
        a0 = 0.75 * p2
        a1 = f[2] * (9.0 * h * z2 * p2 + (1.5 - 15.0 * z2) * p4) - ez * ef * (4.5 * h * p2 - 7.5 * p4)
        a3 = -1.5 * ez * (h * p2 - p4)
        w[0] = w[0] - k6 * (a0 * (f[1] * ez - f[2] * ey) - a1 * ey + a3 * f[1])
        w[1] = w[1] - k6 * (a0 * (f[2] * ex - f[0] * ez) + a1 * ex - a3 * f[0])
        w[2] = w[2] - k6 * a0 * (f[0] * ey - f[1] * ex)
        et = ex * t[0] + ey * t[1] + ez * t[2]
        b0, b1, b2 = p3 * (0.375 - 2.25 * z2), -1.125 * p3 * et, 2.25 * ez * p3 * et
        b3 = 2.25 * p3 * (ex * t[1] - ey * t[0])
        w[0] = w[0] + k6 * (b0 * t[0] + b1 * ex - b3 * ey)
        w[1] = w[1] + k6 * (b0 * t[1] + b1 * ey + b3 * ex)
        w[2] = w[2] + k6 * (b0 * t[2] + b1 * ez + b2)
        hh, bx, by = 1.0 - h, -ex, -ey
        ext = bx * t[1] - by * t[0]
        c1 = (9.0 * hh * z2 * p2 + (1.5 - 15.0 * z2) * p4) * ext
        c2_ = -ez * (4.5 * hh * p2 - 7.5 * p4) * ext
        c3 = -1.5 * ez * (hh * p2 - p4)
        v[0] = v[0] - k6 * (a0 * (t[2] * by - t[1] * ez) + c2_ * bx - c3 * t[1])
        v[1] = v[1] - k6 * (a0 * (t[0] * ez - t[2] * bx) + c2_ * by + c3 * t[0])
        v[2] = v[2] - k6 * (a0 * (t[1] * bx - t[0] * by) + c2_ * ez + c1)
    out = [torch.where(same, torch.zeros_like(r2), c).sum(1) for c in v + (w if six else [])]
    # the particle's own mobility
    own = fs[first:first + n]
    g1_ = 1.0 / xt[:, 2]
    g3_, g4_, g5_ = g1_**3, g1_**4, g1_**5
    par = k6 - (9.0 * g1_ - 2.0 * g3_ + g5_) * (k6 / 16.0)
    perp = k6 - (9.0 * g1_ - 4.0 * g3_ + g5_) * (k6 / 8.0)
    out[0], out[1], out[2] = out[0] + par * own[:, 0], out[1] + par * own[:, 1], out[2] + perp * own[:, 2]
    if six:
        cpl = g4_ * (k6 * 3.0 / 32.0)
        out[0], out[1] = out[0] + cpl * own[:, 4], out[1] - cpl * own[:, 3]
        rpar, rperp = k8 - g3_ * (k6 * 15.0 / 64.0), k8 - g3_ * (k6 * 3.0 / 32.0)
        out[3] = out[3] - cpl * own[:, 1] + rpar * own[:, 3]
        out[4] = out[4] + cpl * own[:, 0] + rpar * own[:, 4]
        out[5] = out[5] + rperp * own[:, 5]
    return torch.stack(out, dim=1)


def _flow_rows(xt, xs, fs, rpy):
    """Velocities at points from Stokeslets (and rotlets), or from spheres of radius 1 on point tracers."""
    d = [xt[:, None, k] - xs[None, :, k] for k in range(3)]
    f = [fs[None, :, k] for k in range(3)]
    r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
    ri = r2.rsqrt()
    df = d[0] * f[0] + d[1] * f[1] + d[2] * f[2]
    c8 = 1.0 / (8.0 * PI)
    rot = None
    if not rpy:
        A, B, rot = c8 * ri, c8 * ri**3 * df, c8 * ri**3
    else:
        r = r2 * ri
        out_ = r > 1.0
        A = torch.where(out_, c8 * ri * (1.0 + ri * ri / 3.0), torch.full_like(r, 1.0 / (6.0 * PI)))
        B = torch.where(out_, c8 * ri**3 * (1.0 - ri * ri) * df, torch.zeros_like(r))
        rot = torch.where(out_, c8 * ri**3, torch.full_like(r, c8))
    out = [(A * f[k] + B * d[k]).sum(1) for k in range(3)]
    if fs.shape[1] == 6:
        for k, c in enumerate(_cross([fs[None, :, 3 + k] for k in range(3)], d)):
            out[k] = out[k] + (rot * c).sum(1)
    return torch.stack(out, dim=1)


def _by_rows(n_rows, n_cols, rows):
    """rows(lo, hi) over blocks of targets that keep each temporary under 128 MB."""
    step = max(1, min(n_rows, (1 << 24) // max(1, n_cols)))
    return torch.cat([rows(lo, min(n_rows, lo + step)) for lo in range(0, n_rows, step)]) if n_rows else torch.zeros((0, 3))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mobility", "matvec"):
        bodies = _bodies({**case, "bodies": case.get("bodies", 1)}, seed)
        six = case.get("seg_dof", 6) == 6
        vs, vb = [], []
        for b in bodies:
            xs, xb = _dev(b.x_segs).view(-1, 3), _dev(b.x_blobs).view(-1, 3)
            fs, fb = _dev(b.f_segs).view(-1, 6), _dev(b.f_blobs).view(-1, 3)
            if not six:
                fs = fs[:, :3].contiguous()
            n = len(xs) + len(xb)
            s = _by_rows(len(xs), n, lambda lo, hi: _rpy_rows(xs[lo:hi], xs, fs, six, six) + _rpy_rows(xs[lo:hi], xb, fb, six, False))
            vs.append(s if six else torch.cat([s, torch.zeros_like(s)], dim=1))
            vb.append(_by_rows(len(xb), n, lambda lo, hi: _rpy_rows(xb[lo:hi], xb, fb, False, False) + _rpy_rows(xb[lo:hi], xs, fs, False, six)))
        vs, vb = torch.cat(vs).reshape(-1), torch.cat(vb).reshape(-1)
        return {"v_segs": vs, "v_blobs": vb}
    if kind == "wall":
        x, f = (_dev(a) for a in _carpet(case, seed))
        six = case["seg_dof"] == 6
        x, f = x.view(-1, 3), f.view(-1, 6)
        v = _by_rows(len(x), len(x), lambda lo, hi: _wall_rows(x[lo:hi], x, f, lo, six))
        return {"v_segs": (v if six else torch.cat([v, torch.zeros_like(v)], dim=1)).reshape(-1)}
    if kind == "flow":
        b = _body(case["num_fil"], case["num_seg"], case["num_blobs"], seed)
        xs, fs = _dev(b.x_segs).view(-1, 3), _dev(b.f_segs).view(-1, 6)
        xb, fb = _dev(b.x_blobs).view(-1, 3), _dev(b.f_blobs).view(-1, 3)
        p = _dev(_points(case, seed)).view(-1, 3)
        rpy = case["mode"] == "rpy"
        return _by_rows(len(p), len(xs) + len(xb), lambda lo, hi: _flow_rows(p[lo:hi], xs, fs, rpy) + _flow_rows(p[lo:hi], xb, fb, rpy)).reshape(-1)
    # beat, ensemble: iterative solves of tens of thousands of unknowns, over several steps; elastic: an
    # implicit step of a nonlinear model.  A 64-bit restatement of either takes minutes.
    return None
