"""Which plan an R4 contraction under fast math runs: in place (a fused-gather
candidate) where the tensors have runs of four elements and would be
transposed, the matricized form where they are matrices as they lie; what the
choice query names, and what the autotuner times."""
import ctypes as C

import numpy as np
import pytest

from exatensor_amd import talsh as T

# D, L, R index orders, extents, in place
CASES = [
    ("ib", "ki", "kb", dict(i=200, b=150, k=170), False),
    ("bi", "ik", "bk", dict(i=200, b=150, k=170), False),
    ("abij", "klab", "klij", dict(a=12, b=13, i=14, j=15, k=16, l=11), False),
    ("ib", "wki", "kwb", dict(i=200, b=150, k=170, w=1), True),  # matrices, but for the order of a unit index
    ("abij", "kalb", "klij", dict(a=12, b=13, i=14, j=15, k=16, l=11), True),
    ("aibj", "klab", "klij", dict(a=12, b=13, i=14, j=15, k=16, l=11), True),
    ("aibj", "klab", "klij", dict(a=3, b=13, i=14, j=15, k=16, l=11), False),
]


def _args(do, lo, ro, ext):
    dims = [[ext[x] for x in o] for o in (do, lo, ro)]
    pat = "D(%s)+=L(%s)*R(%s)" % tuple(",".join(o) for o in (do, lo, ro))
    return pat, dims


@pytest.mark.parametrize("do,lo,ro,ext,in_place", CASES)
def test_choice(do, lo, ro, ext, in_place):
    L = T.load_library()
    pat, dims = _args(do, lo, ro, ext)
    v, t = C.c_int(), C.c_int()
    assert L.talshAmdGetPlanMode() == 1
    for fast in (0, 1):
        assert L.talshAmdSelectorChoice(pat.encode(), len(do), T.ints(dims[0]), len(lo), T.ints(dims[1]), len(ro),
                                        T.ints(dims[2]), T.R4, T.YEP, fast, C.byref(v), C.byref(t)) == 0
        if fast:
            assert (v.value >= T.FUSED_VARIANT) == in_place


def _runs(L, a):
    """Whether some fused-gather candidate has runs of four elements in both
    operands and along the result's rows."""
    n, info, ext, st = C.c_int(), T.ints([0] * 9), T.ints([0] * 96), (C.c_longlong * 96)()
    assert L.talshAmdPlanFusedCandidates(*a, C.byref(n)) == 0
    for i in range(n.value):
        assert L.talshAmdPlanFusedMaps(*a, i, info, ext, st) == 0
        run = [info[3 + g] > 0 and st[16 * g] == 1 and ext[16 * g] >= 4 for g in range(6)]
        if (run[0] or run[1]) and (run[2] or run[3]) and run[4]:
            return True
    return False


def test_matrices_are_left_as_matrices():
    """Over random index orders: the fast-math plan is in place exactly where
    the cheapest matricization moves something and the runs allow it."""
    L = T.load_library()
    rng = np.random.default_rng(3)
    v, t, n, moved = C.c_int(), C.c_int(), C.c_int(), (C.c_double * 64)()
    seen = set()
    for _ in range(3000):
        nk, nl, nr = (int(x) for x in rng.integers(1, 3, 3))
        k, l, r = "kl"[:nk], "ab"[:nl], "ij"[:nr]
        ext = {x: int(rng.integers(2, 9)) for x in k + l + r}
        do, lo, ro = ("".join(rng.permutation(list(x))) for x in (l + r, k + l, k + r))
        pat, dims = _args(do, lo, ro, ext)
        a = (pat.encode(), len(do), T.ints(dims[0]), len(lo), T.ints(dims[1]), len(ro), T.ints(dims[2]), T.R4, T.YEP)
        assert L.talshAmdPlanCandidates(*a, 64, moved, C.byref(n)) == 0
        assert L.talshAmdSelectorChoice(*a, 1, C.byref(v), C.byref(t)) == 0
        runs = _runs(L, a[:7])
        assert (v.value >= T.FUSED_VARIANT) == (moved[0] > 0 and runs), (pat, ext)
        seen.add((moved[0] > 0, runs))
    assert len(seen) == 4


@pytest.mark.gpu
def test_autotuner_times_the_split_in_place():
    """Plan mode 2 tunes an R4 contraction under fast math too, the in-place
    form among the candidates, and every forced candidate agrees with float64
    sums (bound: that of the in-place tests)."""
    from gpu_util import contract, engine, rel_err
    L = engine().lib
    rng = np.random.default_rng(9)
    do, lo, ro, ext, _ = CASES[4]
    pat, dims = _args(do, lo, ro, ext)
    d, l, r = (rng.uniform(-1, 1, x).astype(np.float32) for x in dims)
    want = d + 0.5 * np.einsum(f"{lo},{ro}->{do}", l.astype(np.float64), r.astype(np.float64), optimize=True)
    flat = lambda x: x.ravel(order="F")
    v, t = C.c_int(), C.c_int()
    key = (pat.encode(), 4, T.ints(dims[0]), 4, T.ints(dims[1]), 4, T.ints(dims[2]), T.R4, T.YEP, 1, C.byref(v), C.byref(t))
    nf, nc = C.c_int(), C.c_int()
    assert L.talshAmdPlanFusedCandidates(*key[:7], C.byref(nf)) == 0 and nf.value > 0
    assert L.talshAmdPlanCandidates(*key[:9], 0, None, C.byref(nc)) == 0
    assert L.talshEnableFastMath(T.DEV_AMD_GPU, 0) == 0
    try:
        L.talshAmdAutotuneClear()
        assert L.talshAmdSetPlanMode(2) == 0
        assert L.talshAmdAutotuneChoice(*key) == T.TALSH_NOT_FOUND
        run = lambda: contract(pat, flat(d), dims[0], flat(l), dims[1], flat(r), dims[2], 0.5, True)
        e, got = run()
        assert e == 0 and rel_err(got, flat(want)) <= 1e-6
        assert L.talshAmdAutotuneChoice(*key) == 0
        for x in list(range(nc.value)) + [T.FUSED_VARIANT + i for i in range(nf.value)]:
            L.talshAmdSetPlanVariant(x, -1)
            e, got = run()
            assert e == 0 and rel_err(got, flat(want)) <= 1e-6, x
    finally:
        L.talshAmdSetPlanVariant(-1, -1)
        L.talshAmdSetPlanMode(1)
        L.talshAmdAutotuneClear()
        L.talshDisableFastMath(T.DEV_AMD_GPU, 0)
