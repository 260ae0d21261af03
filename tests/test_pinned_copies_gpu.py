"""Uploads and downloads of host memory that a kernel reaches (pinned arrays of up
to 1 MB, whole ones and views inside them) and that it does not (larger ones,
pageable arrays): the same evaluation from each, bit for bit, and again from
other values (nothing is kept from the first); the kernel's copies are counted,
one for every array that it reaches and none for the others."""
import numpy as np
import pytest

from timfilsimmod_amd import _lib as L
from timfilsimmod_amd.mobility import PinnedArray, RpyHandle

pytestmark = pytest.mark.gpu


def evaluate(h, arrays, vs, vb):
    for what, a in zip((L.SEG_POSITIONS, L.BLOB_POSITIONS, L.SEG_FORCES, L.BLOB_FORCES), arrays):
        h.upload(what, a)
    h.evaluate()
    h.download(L.SEG_VELOCITIES, vs)
    h.download(L.BLOB_VELOCITIES, vb)
    h.sync()
    return vs.copy(), vb.copy()


# 48 ns bytes of segment forces: one page, more, on both sides of 1 MB
@pytest.mark.parametrize("ns,nb", [(5, 7), (342, 683), (3000, 1500), (21845, 1), (21846, 800)])
def test_pinned_equals_pageable(ns, nb):
    print(f"case ns={ns} nb={nb}", flush=True)
    rng = np.random.default_rng(ns)
    lens = (3 * ns, 3 * nb, 6 * ns, 3 * nb, 6 * ns, 3 * nb)
    pinned = [PinnedArray(n + 3) for n in lens]
    h = RpyHandle(ns, nb, seg_dof=6, precision=L.PRECISION_FP64, bs_accumulate=True)
    try:
        for _ in range(2):
            box = 2.0 * (ns + nb) ** (1 / 3)
            plain = [rng.uniform(-box, box, lens[0]), rng.uniform(-box, box, lens[1]), rng.normal(size=lens[2]),
                     rng.normal(size=lens[3])]
            before = h.kernel_copies()
            want = evaluate(h, plain, np.zeros(lens[4]), np.zeros(lens[5]))
            assert h.kernel_copies() == before
            for off in (0, 3):
                views = [p.array[off:off + n] for p, n in zip(pinned, lens)]
                for v, a in zip(views, plain):
                    v[:] = a
                got = evaluate(h, views[:4], views[4], views[5])
                assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
                reached = sum(8 * n <= 1 << 20 for n in lens)
                assert h.kernel_copies() == before + reached
                before += reached
    finally:
        h.close()
        for p in pinned:
            p.free()
