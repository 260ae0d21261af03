"""The block inverse at the sizes where its form changes (up to 64, 128 and 192
rows in registers, more in memory), with pivots in any order, uneven blocks,
and singular and non-finite ones.

Tolerance: n eps times the condition number, 193 x 2.2e-16 x 3 for these blocks
(a random part of norm 2 sqrt(n) beside 3 sqrt(n) I) = 1.3e-13, and a factor 8
for the growth of the entries."""
import numpy as np
import pytest

from oracle import broyden_oracle as BO
from timfilsimmod_amd import _lib as L
from timfilsimmod_amd.broyden import BroydenSolver

pytestmark = pytest.mark.gpu


def block(n, rng):
    m = rng.normal(size=(n, n)) + 3.0 * np.sqrt(n) * np.eye(n)
    return m[rng.permutation(n)]            # the large entries anywhere: every step looks for its pivot


@pytest.mark.parametrize("sizes", [[1, 2, 63, 64], [64] * 5, [65, 1, 64], [127, 128, 120, 3], [129, 128], [191, 192, 7],
                                   [193, 40]])
def test_inverse_matches_numpy(sizes):
    print(f"case sizes={sizes}", flush=True)
    rng = np.random.default_rng(sum(sizes))
    blocks = [block(n, rng) for n in sizes]
    eng = BroydenSolver(sizes, confidence=1.0)
    try:
        eng.set_jacobian(blocks)
        e = rng.normal(size=sum(sizes))
        eng.start(e)
        want = -BO.block_diag_apply([np.linalg.inv(b) for b in blocks], e)
        err = np.linalg.norm(eng.find_update() - want) / np.linalg.norm(want)
        print(f"  rel err {err:.2e}", flush=True)
        assert err <= 1e-12
    finally:
        eng.close()


@pytest.mark.parametrize("n", [5, 64, 100, 128, 150, 192, 200])
@pytest.mark.parametrize("what", ["rank", "nan", "inf", "zero"])
def test_bad_blocks_are_reported(n, what):
    print(f"case n={n} {what}", flush=True)
    rng = np.random.default_rng(n)
    good, bad = block(n, rng), block(n, rng)
    if what == "rank":
        bad[:, n // 2] = 0.0                # a column without a pivot
    else:
        bad[n // 3, n // 2] = {"nan": np.nan, "inf": np.inf, "zero": 0.0}[what]
    if what == "zero":
        bad[:] = 0.0
    eng = BroydenSolver([n, n])
    try:
        with pytest.raises(L.TfsError) as err:
            eng.set_jacobian([good, bad])
        assert err.value.code == L.TFS_ERR_NON_FINITE and "block 1" in str(err.value)
    finally:
        eng.close()
