"""Three-way BF16 split products (FP32 under fast math) whose planes are built
from the tensors in place: runs of 3, 4 and 5 elements (the dispatch's line
lies at 4) and longer ones, rows and k on either side of a 64-wide tile and of the 32-wide k
blocks, sums over several K chunks, contracted groups in reversed orders and of
up to five dimensions (five are matricized), both orientations, accumulating
and not (D then holds NaN). Against float64 sums, and beside the matricized
form of the same contraction.

Bound 1e-6: every operand is held to 2^-24 of itself and the products are
summed in FP32 (2^-24 each, errors of either sign) with FP64 sums across
chunks; relative to the result's norm that leaves a few 2^-24 times the square
root of a chunk's MFMA steps, below 5e-7."""
import numpy as np
import pytest

from exatensor_amd import talsh as T
from gpu_util import contract, engine, rel_err

pytestmark = pytest.mark.gpu

# D, L, R index orders, extents
CASES = [
    ("bi", "ki", "kb", dict(i=65, b=63, k=33)),
    ("ib", "ik", "bk", dict(i=16, b=17, k=31)),
    ("ib", "ik", "kb", dict(i=15, b=64, k=64)),
    ("iajb", "iakl", "lkjb", dict(i=3, a=25, b=7, j=9, k=11, l=5)),
    ("iajb", "iakl", "lkjb", dict(i=4, a=19, b=13, j=5, k=16, l=4)),
    ("aibj", "klia", "ljkb", dict(i=5, a=5, b=21, j=3, k=5, l=13)),
    ("bi", "ik", "bk", dict(i=130, b=16, k=65)),
    ("aibj", "kalj", "likb", dict(a=17, i=3, b=16, j=5, k=16, l=7)),
    ("jbia", "aklj", "lkbi", dict(a=16, j=33, b=3, i=5, k=4, l=18)),
    ("abij", "aikl", "kblj", dict(a=16, b=5, i=9, j=4, k=48, l=47)),
    ("ab", "kalmn", "nmblk", dict(a=70, b=66, k=17, l=2, m=3, n=16)),
    ("ab", "klmnoa", "onmlkb", dict(a=20, b=18, k=16, l=2, m=3, n=2, o=16)),
    ("ab", "ka", "kb", dict(a=64, b=64, k=9001)),
]


@pytest.mark.parametrize("do,lo,ro,ext", CASES)
def test_split_planes_in_place(do, lo, ro, ext):
    L = engine().lib
    rng = np.random.default_rng(sum(ext.values()))
    dims = {t: [ext[x] for x in o] for t, o in (("D", do), ("L", lo), ("R", ro))}
    l, r, d = (rng.uniform(-1, 1, dims[t]).astype(np.float32) for t in "LRD")
    prod = 0.5 * np.einsum(f"{lo},{ro}->{do}", l.astype(np.float64), r.astype(np.float64), optimize=True)
    flat = lambda x: x.ravel(order="F")
    for acc in (True, False):
        want = prod + d if acc else prod
        d0 = d if acc else np.full_like(d, np.nan)
        pat = "D(%s)%s=L(%s)*R(%s)" % (",".join(do), "+" if acc else "", ",".join(lo), ",".join(ro))
        assert L.talshEnableFastMath(T.DEV_AMD_GPU, 0) == 0
        try:
            for v in (-1, 0):
                L.talshAmdSetPlanVariant(v, -1)
                e, got = contract(pat, flat(d0), dims["D"], flat(l), dims["L"], flat(r), dims["R"], 0.5, acc)
                assert e == 0, (v, acc, e)
                assert rel_err(got, flat(want)) <= 1e-6, (v, acc)
        finally:
            L.talshAmdSetPlanVariant(-1, -1)
            L.talshDisableFastMath(T.DEV_AMD_GPU, 0)
