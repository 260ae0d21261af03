"""New positions: the fixed-point frame of FP32 tiles and the overlapping-pair
lists against the FP64 oracle, from one particle on: particles by the hundred
in one place (lists sorted from LDS and by rank, or made in order, capacities
grown), thousands of them, coincident ones and cells with more particles than a walk visits, independent bodies in the same place and bodies without particles, positions that are refused and the ones after
them, lists rebuilt while an earlier capacity is in use.

Tolerances: the matvec's bars, 1e-12 (FP64 sums of n terms in another order)
and 1e-6 (FP32 tiles)."""
import numpy as np
import pytest

from oracle import oracle as O
from timfilsimmod_amd import _lib as L
from timfilsimmod_amd.mobility import RpyHandle

pytestmark = pytest.mark.gpu

P32, P64 = L.PRECISION_FP32_ACC64, L.PRECISION_FP64
TOLS = {P32: 1e-6, P64: 1e-12}


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def cloud(ns, nb, cluster, seed, centre=(0.0, 0.0, 0.0)):
    """ns + nb particles at about one per 8 cubic radii, the first `cluster` of
    the segments and of the blobs within one radius of the centre."""
    rng = np.random.default_rng(seed)
    box = (ns + nb) ** (1 / 3) + 2.0
    c = np.asarray(centre)
    xs, xb = rng.uniform(-box, box, (ns, 3)) + c, rng.uniform(-box, box, (nb, 3)) + c
    for x in (xs, xb):
        m = min(cluster, len(x))
        x[:m] = rng.uniform(-0.55, 0.55, (m, 3)) + c
    return xs.ravel(), xb.ravel(), rng.normal(size=6 * ns), rng.normal(size=3 * nb)


def evaluate(h, ns, nb, xs, xb, fs, fb):
    for what, a in ((L.SEG_POSITIONS, xs), (L.BLOB_POSITIONS, xb), (L.SEG_FORCES, fs), (L.BLOB_FORCES, fb)):
        if a.size:
            h.upload(what, a)
    h.evaluate()
    vs, vb = np.zeros(6 * ns), np.zeros(3 * nb)
    if ns:
        h.download(L.SEG_VELOCITIES, vs)
    if nb:
        h.download(L.BLOB_VELOCITIES, vb)
    h.sync()
    return np.concatenate([vs, vb])


def oracle_all(xs, xb, fs, fb):
    return np.concatenate(O.full_mobility(xs, xb, fs, fb, seg_dof=6, bs_accumulate=True, a_seg=1.0, a_blob=1.2))


def handle(ns, nb, precision):
    return RpyHandle(ns, nb, seg_dof=6, precision=precision, bs_accumulate=True, seg_radius=1.0, blob_radius=1.2)


@pytest.mark.parametrize("precision", [P32, P64])
@pytest.mark.parametrize("ns,nb,cluster", [(1, 0, 0), (0, 3, 2), (16, 1, 9), (130, 71, 20), (340, 300, 170),
                                           (340, 301, 170), (700, 500, 170), (511, 1, 30),
                                           (6100, 45, 30), (3300, 3100, 60), (4000, 2600, 170)])
def test_sizes_and_clusters(ns, nb, cluster, precision):
    print(f"case ns={ns} nb={nb} cluster={cluster} precision={precision}", flush=True)
    h = handle(ns, nb, precision)
    try:
        for k, m in enumerate((0, cluster, 3)):      # grown capacities stay for the lists after them
            case = cloud(ns, nb, m, 7 * ns + nb + k)
            err = rel(evaluate(h, ns, nb, *case), oracle_all(*case))
            print(f"  cluster {m}: rel err {err:.2e}", flush=True)
            assert err <= TOLS[precision]
    finally:
        h.close()


@pytest.mark.parametrize("precision", [P32, P64])
@pytest.mark.parametrize("sizes", [[(40, 30), (0, 0), (1, 0), (0, 129), (300, 200)],
                                   [(2000, 900), (0, 0), (1300, 1700), (40, 900)], [(3, 2)] * 300])
def test_bodies_in_one_place(sizes, precision):
    print(f"case bodies={len(sizes)} precision={precision}", flush=True)
    cases = [cloud(ns, nb, 5, 11 + b, (0.3 * b, 0.0, 0.0)) for b, (ns, nb) in enumerate(sizes)]
    ns, nb = sum(s for s, _ in sizes), sum(b for _, b in sizes)
    h = handle(ns, nb, precision)
    try:
        h.set_bodies([s for s, _ in sizes], [b for _, b in sizes])
        got = evaluate(h, ns, nb, *(np.concatenate([c[k] for c in cases]) for k in range(4)))
        parts = [oracle_all(*c) if c[0].size + c[1].size else np.zeros(0) for c in cases]
        want = np.concatenate([p[:6 * s] for p, (s, _) in zip(parts, sizes)] +
                              [p[6 * s:] for p, (s, _) in zip(parts, sizes)])
        err = rel(got, want)
        print(f"  rel err {err:.2e}", flush=True)
        assert err <= TOLS[precision]
    finally:
        h.close()


@pytest.mark.parametrize("ns,nb", [(200, 100), (5000, 1500)])
def test_refused_positions_and_the_ones_after_them(ns, nb):
    print(f"case ns={ns} nb={nb}", flush=True)
    xs, xb, fs, fb = cloud(ns, nb, 4, 5)
    h = handle(ns, nb, P32)
    try:
        want = oracle_all(xs, xb, fs, fb)
        assert rel(evaluate(h, ns, nb, xs, xb, fs, fb), want) <= TOLS[P32]
        for value, where in ((np.nan, 0), (np.inf, 3 * ns - 1), (-1.1e4, 4), (1e308, 7)):
            bad = xs.copy()
            bad[where] = value
            with pytest.raises(Exception) as err:
                evaluate(h, ns, nb, bad, xb, fs, fb)
            assert ("finite" if not np.isfinite(value) else "1024") in str(err.value)
            assert rel(evaluate(h, ns, nb, xs, xb, fs, fb), want) <= TOLS[P32]
    finally:
        h.close()
    # the frame far from the origin: the centre goes, the step stays
    far = xs + 1e5
    h = handle(ns, nb, P32)
    try:
        assert rel(evaluate(h, ns, nb, far, xb + 1e5, fs, fb), oracle_all(far, xb + 1e5, fs, fb)) <= TOLS[P32]
    finally:
        h.close()


@pytest.mark.parametrize("device", [False, True])
@pytest.mark.parametrize("ns,nb", [(200, 100), (5000, 1500)])
def test_profile_counts_no_refused_evaluation(ns, nb, device):
    print(f"case ns={ns} nb={nb} device={device}", flush=True)
    import torch

    put = (lambda a: torch.tensor(a, device="cuda")) if device else (lambda a: a)
    xs, xb, fs, fb = (put(a) for a in cloud(ns, nb, 4, 5))
    bad = put(np.full(3 * ns, np.nan))
    torch.cuda.synchronize()
    h = RpyHandle(ns, nb, seg_dof=6, precision=P32, bs_accumulate=True, seg_radius=1.0, blob_radius=1.2,
                  memory=L.MEMORY_DEVICE if device else L.MEMORY_HOST)
    try:
        for what, a in ((L.SEG_POSITIONS, xs), (L.BLOB_POSITIONS, xb), (L.SEG_FORCES, fs), (L.BLOB_FORCES, fb)):
            h.upload(what, a)
        h.profile(True)
        h.evaluate()
        ms, launches = h.profile_read()[P32]
        assert launches == 1 and ms > 0
        for _ in range(2):
            h.upload(L.SEG_POSITIONS, bad)
            with pytest.raises(Exception, match="finite"):
                h.evaluate()
            assert h.profile_read()[P32] == (0.0, 0)
        h.upload(L.SEG_POSITIONS, xs)
        for _ in range(3):
            h.evaluate()
        again, launches = h.profile_read()[P32]
        assert launches == 3 and 0 < again < 30 * ms + 1.0
    finally:
        h.close()


@pytest.mark.parametrize("radius", [1e-9, 3e-7, 1.0, 4e5])
def test_one_particle_of_any_radius(radius):
    """Force and torque on a particle by itself, whose extent gives the
    fixed-point scale no bound: neither the staged torques (times the scale's
    square) nor the third power of 1/r may leave a float's range."""
    print(f"case radius={radius}", flush=True)
    fs = np.array([0.3, -0.7, 0.2, 1.0, 0.4, -0.5])
    got = {}
    for precision in (P32, P64):
        h = RpyHandle(1, 0, seg_dof=6, precision=precision, bs_accumulate=True, seg_radius=radius, blob_radius=radius)
        try:
            got[precision] = evaluate(h, 1, 0, np.array([radius, 0.0, 0.0]), np.zeros(0), fs, np.zeros(0))
        finally:
            h.close()
    exact = np.concatenate([fs[:3] / (6 * np.pi * radius), fs[3:] / (8 * np.pi * radius**3)])
    for precision, v in got.items():
        for part in (slice(0, 3), slice(3, 6)):
            assert rel(v[part], exact[part]) <= TOLS[precision]


def test_radii_too_small_for_the_scale_are_refused():
    h = RpyHandle(1, 0, seg_dof=6, precision=P32, bs_accumulate=True, seg_radius=1e-13, blob_radius=1e-13)
    try:
        with pytest.raises(Exception, match="1024"):
            evaluate(h, 1, 0, np.zeros(3), np.zeros(0), np.ones(6), np.zeros(0))
    finally:
        h.close()


def seconds(run):
    import time

    t0 = time.perf_counter()
    out = run()
    return out, time.perf_counter() - t0


# a list of one entry per particle of the body, beside a second body as crowded
@pytest.mark.parametrize("precision", [P32, P64])
@pytest.mark.parametrize("ns,nb,spread", [(1500, 1500, 0.5), (700, 1, 1e-3), (2500, 3600, 0.3)])
def test_thousands_in_one_place(ns, nb, spread, precision):
    """Every particle overlaps every other: the lists' cost stays a pass over the
    body for each target (milliseconds for all; their lengths squared, moved one
    by one, would be seconds)."""
    print(f"case ns={ns} nb={nb} spread={spread} precision={precision}", flush=True)
    rng = np.random.default_rng(ns)
    xs, xb = spread * rng.uniform(-1, 1, 3 * ns), spread * rng.uniform(-1, 1, 3 * nb)
    fs, fb = rng.normal(size=6 * ns), rng.normal(size=3 * nb)
    h = handle(ns, nb, precision)
    try:
        evaluate(h, ns, nb, xs, xb, fs, fb)                       # grows the lists
        got, took = seconds(lambda: evaluate(h, ns, nb, xs, xb, fs, fb))
        want = oracle_all(xs, xb, fs, fb)
        print(f"  rel err {rel(got, want):.2e}, {took * 1e3:.1f} ms", flush=True)
        assert rel(got, want) <= TOLS[precision]
        assert took < 0.25
        assert np.array_equal(evaluate(h, ns, nb, xs, xb, fs, fb), got)
    finally:
        h.close()


@pytest.mark.parametrize("precision", [P32, P64])
@pytest.mark.parametrize("bodies", [1, 2])
def test_small_particles_crowd_a_cell(bodies, precision):
    """Cells take their side from the larger radius: thousands of small blobs in
    each, nearly none of which overlap."""
    print(f"case bodies={bodies} precision={precision}", flush=True)
    rng = np.random.default_rng(3)
    ns, nb, kw = 20, 4000, dict(a_seg=1.0, a_blob=0.02)
    parts = [(rng.uniform(-3, 3, 3 * ns), rng.uniform(-2, 2, 3 * nb), rng.normal(size=6 * ns), rng.normal(size=3 * nb))
             for _ in range(bodies)]
    h = RpyHandle(ns * bodies, nb * bodies, seg_dof=6, precision=precision, bs_accumulate=True, seg_radius=1.0,
                  blob_radius=0.02)
    try:
        if bodies > 1:
            h.set_bodies([ns] * bodies, [nb] * bodies)
        got = evaluate(h, ns * bodies, nb * bodies, *(np.concatenate([p[k] for p in parts]) for k in range(4)))
        each = [O.full_mobility(*p, seg_dof=6, bs_accumulate=True, **kw) for p in parts]
        want = np.concatenate([e[0] for e in each] + [e[1] for e in each])
        print(f"  rel err {rel(got, want):.2e}", flush=True)
        assert rel(got, want) <= TOLS[precision]
    finally:
        h.close()


def test_positions_that_are_not_finite_in_fp64():
    """FP64 does not look at the positions: an evaluation of such ones ends as
    soon as any other and says so in its velocities."""
    ns, nb = 3000, 1000
    xs, xb, fs, fb = cloud(ns, nb, 4, 5)
    h = handle(ns, nb, P64)
    try:
        want = evaluate(h, ns, nb, xs, xb, fs, fb)
        evaluate(h, ns, nb, np.full(3 * ns, np.nan), xb, fs, fb)  # grows the lists
        got, took = seconds(lambda: evaluate(h, ns, nb, np.full(3 * ns, np.nan), xb, fs, fb))
        print(f"case ns={ns} nb={nb}: {took * 1e3:.1f} ms", flush=True)
        assert np.all(np.isnan(got.reshape(-1, 3)[:2 * ns:2])) and took < 0.25
        assert np.array_equal(evaluate(h, ns, nb, xs, xb, fs, fb), want)
    finally:
        h.close()


@pytest.mark.parametrize("precision", [P32, P64])
@pytest.mark.parametrize("num_bodies", [1024, 1025, 70_000])
def test_more_bodies_than_a_grid_has_rows(num_bodies, precision):
    """Bodies of one segment each, all in one place: each its own mobility only;
    then most of them empty (FP64: the small problem's one launch)."""
    print(f"case bodies={num_bodies} precision={precision}", flush=True)
    rng = np.random.default_rng(num_bodies)
    a = 1.0
    for ns in (num_bodies, 300):
        xs, fs = rng.uniform(-5, 5, 3 * ns), rng.normal(size=6 * ns)
        h = handle(ns, 0, precision)
        try:
            h.set_bodies([1] * ns + [0] * (num_bodies - ns), [0] * num_bodies)
            for _ in range(2):
                got = evaluate(h, ns, 0, xs, np.zeros(0), fs, np.zeros(0)).reshape(ns, 6)
                f = fs.reshape(ns, 6)
                assert rel(got[:, :3], f[:, :3] / (6 * np.pi * a)) <= TOLS[precision]
                assert rel(got[:, 3:], f[:, 3:] / (8 * np.pi * a**3)) <= TOLS[precision]
                xs = xs[::-1].copy()
        finally:
            h.close()
        if num_bodies < 2000:
            break
