"""The half-space matvec at the sizes where its work list changes (tiles of 64
targets, source shares of the four waves, items of several staged batches),
against the oracle's half-space sums.

Bars: those of the half-space matvec, 1e-12 (FP64) and 2e-6 (FP32 tiles)."""
import numpy as np
import pytest

from oracle import oracle as O
from timfilsimmod_amd import _lib as L
from timfilsimmod_amd.mobility import RpyHandle

pytestmark = pytest.mark.gpu

P32, P64 = L.PRECISION_FP32_ACC64, L.PRECISION_FP64
TOLS = {P32: 2e-6, P64: 1e-12}


def carpet(n, seed):
    """n particles at least 2.3 apart on a jittered grid above the wall."""
    rng = np.random.default_rng(seed)
    side = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), -1).reshape(-1, 3)[rng.permutation(side ** 3)[:n]]
    return (2.7 * g + rng.uniform(-0.2, 0.2, (n, 3)) + [0.0, 0.0, 1.5]).reshape(-1)


def evaluate(xs, xb, fs, fb, seg_dof, precision, blocks):
    ns, nb = xs.size // 3, xb.size // 3
    h = RpyHandle(ns, nb, seg_dof=seg_dof, precision=precision, bs_accumulate=True)
    try:
        h.set_domain(L.DOMAIN_HALF_SPACE)
        for what, a in ((L.SEG_POSITIONS, xs), (L.BLOB_POSITIONS, xb), (L.SEG_FORCES, fs), (L.BLOB_FORCES, fb)):
            if a.size:
                h.upload(what, a)
        h.evaluate(blocks)
        vs, vb = np.zeros(6 * ns), np.zeros(3 * nb)
        if ns:
            h.download(L.SEG_VELOCITIES, vs)
        if nb:
            h.download(L.BLOB_VELOCITIES, vb)
        h.sync()
        return np.concatenate([vs, vb])
    finally:
        h.close()


@pytest.mark.parametrize("precision", [P32, P64])
@pytest.mark.parametrize("seg_dof", [6, 3])
@pytest.mark.parametrize("ns,nb", [(1, 0), (1, 1), (3, 2), (63, 1), (64, 0), (65, 0), (0, 129), (64, 64), (255, 0),
                                   (257, 66), (400, 513)])
def test_tile_edges(ns, nb, seg_dof, precision):
    print(f"case dof={seg_dof} ns={ns} nb={nb} precision={precision}", flush=True)
    x, rng = carpet(ns + nb, ns + 7 * nb), np.random.default_rng(3)
    xs, xb, fs, fb = x[:3 * ns], x[3 * ns:], rng.normal(size=6 * ns), rng.normal(size=3 * nb)
    got = evaluate(xs, xb, fs, fb, seg_dof, precision, L.BLOCK_ALL)
    with O.domain(O.HALF_SPACE):
        want = np.concatenate(O.full_mobility(xs, xb, fs, fb, seg_dof=seg_dof, bs_accumulate=True))
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"  rel err {err:.2e}", flush=True)
    assert err <= TOLS[precision]


@pytest.mark.parametrize("precision", [P32, P64])
def test_items_of_several_batches(precision):
    """Few segments among 15,000 blobs: items of 576 sources, two staged batches and a quarter."""
    ns, nb = 70, 15000
    print(f"case ns={ns} nb={nb} precision={precision}", flush=True)
    x, rng = carpet(ns + nb, 1), np.random.default_rng(4)
    xs, xb, fs, fb = x[:3 * ns], x[3 * ns:], rng.normal(size=6 * ns), rng.normal(size=3 * nb)
    got = evaluate(xs, xb, fs, fb, 6, precision, L.BLOCK_SB | L.BLOCK_BS)
    with O.domain(O.HALF_SPACE):
        want = np.concatenate([O.block("sb", xs, xb, fs, fb, np.zeros(6 * ns), seg_dof=6),
                               O.block("bs", xs, xb, fs, fb, np.zeros(3 * nb), seg_dof=6, bs_accumulate=True)])
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"  rel err {err:.2e}", flush=True)
    assert err <= TOLS[precision]
