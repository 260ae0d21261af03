"""The symmetric pair kernel where a handle takes it by its size (no shape set):
6-component segments (each unordered pair once, with the rotational couplings)
and mid-size bodies, against the FP64 oracle, over sizes that leave the last
tile and the last panel partly empty, one class only, overlapping pairs,
unequal radii, both BS write rules, and independent bodies whose panels
straddle bodies; what such a handle reports, block subsets, chosen shapes, the
autotuner and captured evaluations next to larger ones.

Tolerances: the matvec's bars, 1e-12 (FP64 sums of n terms in another order,
~n eps at worst, the 1/r of one Newton step 4e-15) and 1e-6 (FP32 tiles, ~30
roundings of 6e-8 per pair, averaged over the pairs)."""
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


def cloud(ns, nb, seed):
    rng = np.random.default_rng(seed)
    box = 1.1 * (ns + nb) ** (1 / 3) + 2.0      # dense enough for overlapping pairs
    return (rng.uniform(-box, box, 3 * ns), rng.uniform(-box, box, 3 * nb), rng.normal(size=6 * ns),
            rng.normal(size=3 * nb))


def load(h, xs, xb, fs, fb):
    for what, a in ((L.SEG_POSITIONS, xs), (L.BLOB_POSITIONS, xb), (L.SEG_FORCES, fs), (L.BLOB_FORCES, fb)):
        if a.size:
            h.upload(what, a)


def read(h, ns, nb):
    vs, vb = np.zeros(6 * ns), np.zeros(3 * nb)
    if ns:
        h.download(L.SEG_VELOCITIES, vs)
    if nb:
        h.download(L.BLOB_VELOCITIES, vb)
    h.sync()
    return np.concatenate([vs, vb])


# one particle per lane from ~4,100 particles on, two per lane from ~11,500 on
@pytest.mark.parametrize("precision", [P32, P64])
@pytest.mark.parametrize("seg_dof,ns,nb,bs_acc", [(6, 2050, 2130, True), (6, 4225, 0, False), (6, 0, 4100, True),
                                                  (6, 4097, 65, False), (3, 2111, 2111, True), (6, 7001, 5190, True),
                                                  (6, 11600, 1, False), (6, 129, 11777, True), (3, 5000, 3000, False)])
def test_default_handles_match_oracle(seg_dof, ns, nb, bs_acc, precision):
    print(f"case dof={seg_dof} ns={ns} nb={nb} bs_accumulate={bs_acc} precision={precision}", flush=True)
    xs, xb, fs, fb = cloud(ns, nb, ns + 3 * nb)
    rs, rb = O.full_mobility(xs, xb, fs, fb, seg_dof=seg_dof, bs_accumulate=bs_acc, a_seg=1.0, a_blob=1.3)
    h = RpyHandle(ns, nb, seg_dof=seg_dof, precision=precision, bs_accumulate=bs_acc, seg_radius=1.0, blob_radius=1.3)
    try:
        load(h, xs, xb, fs, fb)
        h.evaluate()
        got = read(h, ns, nb)
        err = rel(got, np.concatenate([rs, rb]))
        print(f"  rel err {err:.2e}", flush=True)
        assert err <= TOLS[precision]
        if ns:                                   # the rotations alone
            w = got[:6 * ns].reshape(ns, 6)[:, 3:]
            if seg_dof == 6:
                assert rel(w, rs.reshape(ns, 6)[:, 3:]) <= TOLS[precision]
            else:
                assert not np.any(w)
        h.evaluate()
        assert np.array_equal(read(h, ns, nb), got)
    finally:
        h.close()


BODIES = [(3, 40), (1, 0), (290, 2900), (0, 70), (30, 400), (250, 3100), (2, 33), (300, 2500), (45, 900)]


@pytest.mark.parametrize("precision", [P32, P64])
@pytest.mark.parametrize("seg_dof,bodies", [(6, BODIES), (6, BODIES[:5]), (3, BODIES[:6])])
def test_independent_bodies_match_per_body_oracle(seg_dof, bodies, precision):
    from timfilsimmod_amd.ensemble import make_ensemble

    sizes = [(f, b, max(4.0, 50.0 * np.sqrt(b / 9000.0))) for f, b in bodies]
    e = make_ensemble(sizes=sizes, num_seg=10)
    print(f"case {len(e.bodies)} bodies dof={seg_dof} precision={precision}", flush=True)
    per = [O.full_mobility(b.x_segs, b.x_blobs, b.f_segs, b.f_blobs, seg_dof=seg_dof, bs_accumulate=True)
           for b in e.bodies]
    ref = np.concatenate([p[0] for p in per] + [p[1] for p in per])
    h = RpyHandle(e.num_segs, e.num_blobs, seg_dof=seg_dof, precision=precision, bs_accumulate=True)
    try:
        h.set_bodies(e.segs_per_body, e.blobs_per_body)
        load(h, e.x_segs, e.x_blobs, e.f_segs, e.f_blobs)
        h.body_timing(True)
        h.evaluate()
        got = read(h, e.num_segs, e.num_blobs)
        assert rel(got, ref) <= TOLS[precision]
        ms = h.body_times(len(e.bodies))
        assert np.all(np.isfinite(ms)) and np.all(ms >= 0) and ms.max() > 0
    finally:
        h.close()


def test_reported_shapes_subsets_and_chosen_shapes():
    ns, nb = 2500, 2300
    xs, xb, fs, fb = cloud(ns, nb, 4)
    h = RpyHandle(ns, nb, seg_dof=6, precision=P64, bs_accumulate=True)
    plain = RpyHandle(ns, nb, seg_dof=6, precision=P64, bs_accumulate=True)
    try:
        shape = plain.tile_shape(P64)
        assert shape == h.tile_shape(P64) and not h.symmetric(P64)
        load(h, xs, xb, fs, fb)
        load(plain, xs, xb, fs, fb)
        s = shape
        (plain.set_split_shape if s["split"] else plain.set_tile_shape)(P64, s["block"], s["per_thread"], s["chunk"])
        h.evaluate()
        plain.evaluate()
        a, b = read(h, ns, nb), read(plain, ns, nb)
        assert rel(a, b) <= 1e-12 and not np.array_equal(a, b)   # another order of the same sums
        # block subsets take the reported shape, bit for bit
        for blocks in (L.BLOCK_SS | L.BLOCK_SB, L.BLOCK_BB | L.BLOCK_BS, L.BLOCK_SS):
            h.evaluate(blocks)
            plain.evaluate(blocks)
            part = slice(0, 6 * ns) if blocks & L.BLOCK_SS else slice(6 * ns, None)
            assert np.array_equal(read(h, ns, nb)[part], read(plain, ns, nb)[part])
        h.autotune(P64, reps=1)
        assert not h.symmetric(P64)
        h.evaluate()
        assert rel(read(h, ns, nb), b) <= 1e-12
        h.set_tile_shape(P64, 256, 1, 256)
        h.set_persistent(P64, 2)
        h.evaluate()
        assert rel(read(h, ns, nb), b) <= 1e-12
    finally:
        h.close()
        plain.close()


def test_graph_of_a_subset_survives_a_larger_evaluation():
    """A captured evaluation of one block replays rightly after an evaluation of
    all of them needed a larger buffer of partial sums."""
    ns, nb = 2300, 2200
    xs, xb, fs, fb = cloud(ns, nb, 8)
    h = RpyHandle(ns, nb, seg_dof=6, precision=P64, bs_accumulate=True)
    try:
        load(h, xs, xb, fs, fb)
        h.evaluate(L.BLOCK_SS)
        ss = read(h, ns, nb)[:6 * ns]
        g = h.graph(L.BLOCK_SS)
        for _ in range(3):
            h.evaluate()
            full = read(h, ns, nb)[:6 * ns]
            assert not np.array_equal(full, ss)
            g.launch()
            assert np.array_equal(read(h, ns, nb)[:6 * ns], ss)
        g.close()
    finally:
        h.close()


def test_large_ensembles_take_the_form_within_the_buffer_limit():
    """Sixty-four uneven bodies: a tile's slots are one per run of source tiles, so
    the form's buffer stays inside the 4 GiB it may take (beside it, lists and
    positions of ~200 bytes per particle); so with one body of 170,000 particles,
    and not with one of 400,000."""
    import torch

    from timfilsimmod_amd.ensemble import make_ensemble

    e = make_ensemble(64)
    for seg_dof in (3, 6):
        kw = dict(seg_dof=seg_dof, precision=P32, bs_accumulate=True)
        h, plain = (RpyHandle(e.num_segs, e.num_blobs, **kw) for _ in range(2))
        try:
            for x in (h, plain):
                x.set_bodies(e.segs_per_body, e.blobs_per_body)
                load(x, e.x_segs, e.x_blobs, e.f_segs, e.f_blobs)
            plain.set_symmetric(P32, False)
            print(f"case 64 bodies dof={seg_dof}", flush=True)
            torch.cuda.synchronize()
            before = torch.cuda.mem_get_info()[0]
            h.evaluate()
            got = read(h, e.num_segs, e.num_blobs)
            used = (before - torch.cuda.mem_get_info()[0]) / 2**30
            plain.evaluate()
            want = read(plain, e.num_segs, e.num_blobs)
            print(f"  {used:.2f} GiB, rel diff {rel(got, want):.2e}", flush=True)
            assert rel(got, want) <= TOLS[P32] and not np.array_equal(got, want)
            assert used <= 4.0 + 200 * (e.num_segs + e.num_blobs) / 2**30
            if seg_dof == 3:
                assert h.symmetric(P32) and h.symmetric(P64)
        finally:
            h.close()
            plain.close()
    for n, takes in ((170_000, True), (400_000, False)):
        h = RpyHandle(n, 0, seg_dof=3, precision=P32, bs_accumulate=True)
        try:
            assert h.symmetric(P32) == takes
        finally:
            h.close()


def test_the_autotuned_shape_set_again_gives_the_same_results():
    """6-DOF handles report the directed shape behind the symmetric form: setting
    what was reported after the autotuner brings its choice back, and switching
    the form off or setting another shape does not."""
    ns, nb = 12800, 9000                         # symmetric by a fifth
    xs, xb, fs, fb = cloud(ns, nb, 4)
    h = RpyHandle(ns, nb, seg_dof=6, precision=P64, bs_accumulate=True)
    try:
        load(h, xs, xb, fs, fb)
        h.autotune(P64, reps=1)
        h.evaluate()
        tuned, s = read(h, ns, nb), h.tile_shape(P64)
        put = h.set_split_shape if s["split"] else h.set_tile_shape
        other = (h.set_tile_shape, (256, 2, 1024))
        for first, args in (other, (h.set_symmetric, (False,))):
            first(P64, *args)
            h.evaluate()
            assert not np.array_equal(read(h, ns, nb), tuned)
            put(P64, s["block"], s["per_thread"], s["chunk"])
            h.evaluate()
            assert np.array_equal(read(h, ns, nb), tuned)
    finally:
        h.close()


def test_a_six_dof_handle_switched_off_gets_its_own_choice_back():
    ns, nb = 2500, 2300
    h = RpyHandle(ns, nb, seg_dof=6, precision=P64, bs_accumulate=True)
    try:
        load(h, *cloud(ns, nb, 4))
        with pytest.raises(RuntimeError):
            h.set_symmetric(P64)                 # cannot be set, only left
        results = []
        for enable in (None, False, True, False):
            if enable is not None:
                h.set_symmetric(P64, enable)
            h.evaluate()
            results.append(read(h, ns, nb))
        own, off = results[:2]
        assert rel(own, off) <= 1e-12 and not np.array_equal(own, off)
        assert np.array_equal(results[2], own) and np.array_equal(results[3], off)
        s = h.tile_shape(P64)
        (h.set_split_shape if s["split"] else h.set_tile_shape)(P64, s["block"], s["per_thread"], s["chunk"])
        with pytest.raises(RuntimeError):
            h.set_symmetric(P64)                 # a shape was set
    finally:
        h.close()


def test_many_small_bodies_keep_the_directed_form():
    """Bodies that leave their 64-particle tiles mostly empty, or have few tiles,
    take the directed form bit for bit; the same particles in bodies that fill
    them do not."""
    for bodies, takes in (([(20, 30)] * 1000, False), ([(64, 64)] * 1000, False), ([(129, 65)] * 300, False),
                          ([(640, 640)] * 40, True)):
        ns, nb = sum(s for s, _ in bodies), sum(b for _, b in bodies)
        xs, xb, fs, fb = cloud(ns, nb, 6)
        h, plain = (RpyHandle(ns, nb, seg_dof=6, precision=P64, bs_accumulate=True) for _ in range(2))
        try:
            print(f"case {len(bodies)} bodies of {bodies[0]}", flush=True)
            for x in (h, plain):
                x.set_bodies([s for s, _ in bodies], [b for _, b in bodies])
                load(x, xs, xb, fs, fb)
            plain.set_symmetric(P64, False)
            h.evaluate()
            plain.evaluate()
            a, b = read(h, ns, nb), read(plain, ns, nb)
            assert rel(a, b) <= 1e-12 and np.array_equal(a, b) != takes
        finally:
            h.close()
            plain.close()


def test_autotune_tries_both_kinds_without_rotations():
    """Twelve bodies of 320 + 2,000 particles with 3-DOF segments, FP64: one
    particle per lane, the handle's own choice, is a tenth faster than two or the
    directed shapes; the autotuner keeps it, or has found something faster."""
    import time

    bodies = [(320, 2000)] * 12
    ns, nb = (sum(b[k] for b in bodies) for k in (0, 1))
    xs, xb, fs, fb = cloud(ns, nb, 6)
    own, tuned = (RpyHandle(ns, nb, seg_dof=3, precision=P64, bs_accumulate=True) for _ in range(2))
    try:
        for h in (own, tuned):
            h.set_bodies([s for s, _ in bodies], [b for _, b in bodies])
            load(h, xs, xb, fs, fb)
            h.evaluate()
        want = read(own, ns, nb)
        assert np.array_equal(read(tuned, ns, nb), want)
        ms = 1e9
        for _ in range(5):
            t0 = time.perf_counter()
            for _ in range(20):
                own.evaluate()
            own.sync()
            ms = min(ms, (time.perf_counter() - t0) * 50)
        best = tuned.autotune(P64, reps=20)
        print(f"case own {ms * 1e3:.1f} us, tuned {best * 1e3:.1f}, shape {tuned.tile_shape(P64)}", flush=True)
        tuned.evaluate()
        got = read(tuned, ns, nb)
        assert rel(got, want) <= 1e-12
        assert np.array_equal(got, want) or best < ms
    finally:
        own.close()
        tuned.close()
