"""Gathered products by offset tables in LDS, and operands beyond 32-bit offsets: contracted groups of more than
three dimensions or with runs that are no multiple of a k-tile, several chunks
of 64 k-values per k-group, as many dimensions as a group can have, sums cut
along K, and tensors of more than 4 GB read in place. Tolerances of the index
walk tests (float64 / complex128 products); whole numbers exactly."""
import ctypes as C

import numpy as np
import pytest

from exatensor_amd import talsh as T
from gpu_util import contract, engine, rel_err

pytestmark = pytest.mark.gpu

TOL = {T.R8: 1e-13, T.C8: 1e-13, T.R4: 1e-5, T.C4: 1e-5}

# contracted extents, whether L / R hold their stride-1 index among them, free extents of L and of R
GROUPS = [
    ((5, 3, 7, 2, 3), True, False, (65,), (3, 43)),
    ((9, 7, 11), False, True, (2, 3, 2, 3, 2), (63,)),
    ((3, 5, 4, 3), False, False, (3, 3, 3, 3, 3), (2, 5, 2, 3)),
    ((16, 3, 3, 5), True, True, (130,), (5, 7)),
    ((2,) * 16, True, True, (33,), (17,)),
    # four dimensions in every group, the short form of the arguments at its limit; five in one group
    ((3, 5, 4, 3), True, False, (3, 2, 5, 4), (2, 5, 2, 3)),
    ((5, 9), False, True, (3, 3, 3, 2, 2), (6,)),
    ((5, 9), True, True, (7,), (2, 3, 2, 2, 5)),
]


@pytest.mark.parametrize("kind", [T.R8, T.R4, T.C8, T.C4])
@pytest.mark.parametrize("ks,lk,rk,lf,rf", GROUPS)
def test_groups(kind, ks, lk, rk, lf, rf):
    L = engine().lib
    rng = np.random.default_rng(len(ks) * 100 + ks[0])
    kn, ln, rn = "abcdefghijklmnop"[:len(ks)], "qrstu"[:len(lf)], "vwxyz"[:len(rf)]
    ext = dict(zip(kn + ln + rn, ks + lf + rf))
    # R's contracted indices reversed, D's free ones too: no two runs line up
    lord, rord = (kn + ln if lk else ln + kn), (kn[::-1] + rn if rk else rn + kn[::-1])
    dord = rn[::-1] + ln[::-1]
    dims = {t: [ext[x] for x in o] for t, o in (("D", dord), ("L", lord), ("R", rord))}

    def rand(o):
        x = rng.uniform(-1, 1, dims[o])
        return (x + 1j * rng.uniform(-1, 1, dims[o]) if kind in (T.C4, T.C8) else x).astype(T.NP_DTYPE[kind])

    l, r, d = (rand(t) for t in "LRD")
    wide = np.complex128 if kind in (T.C4, T.C8) else np.float64
    K = int(np.prod(ks))
    lm = np.moveaxis(l, [lord.index(x) for x in kn], range(len(kn))).reshape(K, *lf).astype(wide)
    rm = np.moveaxis(r, [rord.index(x) for x in kn], range(len(kn))).reshape(K, *rf).astype(wide)
    p = np.tensordot(lm, rm, (0, 0))  # ln, rn
    want = d.astype(wide) + 0.5 * np.transpose(p, [(ln + rn).index(x) for x in dord])
    pat = "D(%s)+=L(%s)*R(%s)" % tuple(",".join(o) for o in (dord, lord, rord))
    nf = C.c_int()
    assert L.talshAmdPlanFusedCandidates(pat.encode(), len(dord), T.ints(dims["D"]), len(lord), T.ints(dims["L"]),
                                         len(rord), T.ints(dims["R"]), C.byref(nf)) == 0 and nf.value > 0
    flat = lambda x: x.ravel(order="F")
    try:
        for v in range(nf.value):
            for tile in ((0, 1, 2) if kind in (T.R8, T.R4) else (0,)):
                L.talshAmdSetPlanVariant(T.FUSED_VARIANT + v, tile)
                e, got = contract(pat, flat(d), dims["D"], flat(l), dims["L"], flat(r), dims["R"], 0.5, True)
                assert e == 0, (v, tile, e)
                assert rel_err(got, flat(want)) <= TOL[kind], (v, tile)
    finally:
        L.talshAmdSetPlanVariant(-1, -1)


@pytest.mark.parametrize("order", ["akb", "kab", "abk"])
def test_tensor_beyond_4gb(order):
    """L is 4.6 GB: the coordinates along its three dimensions are told apart by
    whole numbers that the sums keep exactly."""
    import torch
    L, gpu = engine().lib, engine().gpu(0)
    ext = dict(a=33, b=133001, k=131, x=5)
    dev = "cuda"
    val = {"a": 1.0, "b": 64.0, "k": 1024.0}
    mod = {"a": 33, "b": 13, "k": 7}
    vec = {c: val[c] * (torch.arange(ext[c], dtype=torch.float64, device=dev) % mod[c]) for c in "abk"}
    o = order[::-1]  # torch's last dimension is the tensor's first
    shape = lambda c: [-1 if y == c else 1 for y in o]
    l = vec["a"].view(shape("a")) + vec["b"].view(shape("b")) + vec["k"].view(shape("k"))
    kx = (torch.arange(131, dtype=torch.float64, device=dev) % 3)[None, :] + torch.arange(5, dtype=torch.float64, device=dev)[:, None]
    d = torch.zeros(5, ext["b"], ext["a"], dtype=torch.float64, device=dev)  # D(a,b,x)
    torch.cuda.synchronize()
    ts = []
    for t, dims in ((d, [33, 133001, 5]), (l, [ext[c] for c in order]), (kx, [131, 5])):
        h = T.TalshTens()
        L.talshTensorClean(C.byref(h))
        assert L.talshTensorConstruct(C.byref(h), T.R8, len(dims), T.ints(dims), gpu, C.c_void_p(t.data_ptr()), -1, None,
                                      0.0, 0.0) == 0
        ts.append(h)
    sk = kx.sum(1)
    want = (vec["a"][None, None, :] + vec["b"][None, :, None]) * sk[:, None, None] + (kx * vec["k"][None, :]).sum(1)[:, None, None]
    pat = ("D(a,b,x)=L(%s)*R(k,x)" % ",".join(order)).encode()
    try:
        for v in (0, 1):
            for tile in (0, 1, 2):
                d.fill_(float("nan"))
                torch.cuda.synchronize()
                L.talshAmdSetPlanVariant(T.FUSED_VARIANT + v, tile)
                assert L.talshTensorContract(pat, C.byref(ts[0]), C.byref(ts[1]), C.byref(ts[2]), 1.0, 0.0, gpu, T.DEV_NULL,
                                             T.COPY_MTT, T.NOPE, None) == 0
                assert torch.equal(d, want), (v, tile)
    finally:
        L.talshAmdSetPlanVariant(-1, -1)
        for h in ts:
            L.talshTensorDestruct(C.byref(h))


@pytest.mark.parametrize("ak", [1, 0])
@pytest.mark.parametrize("m,n,k", [(70000, 40, 8192), (70001, 41, 8195), (130, 6, 4194320)])
def test_matrix_beyond_4gb(m, n, k, ak):
    """A matrix of more than 4 GB on either side of the product, in whole
    vectors and not, and with k-values so far apart that a tile does not fit 32
    bits either (130 rows of 34 MB): whole numbers that the sums keep exactly,
    every tile."""
    import torch
    L = engine().lib
    dev = "cuda"
    rows = torch.arange(m, dtype=torch.float64, device=dev) % 97
    ks = torch.arange(k, dtype=torch.float64, device=dev) % 11
    a = rows[:, None] + 100 * ks[None, :] if ak else rows[None, :] + 100 * ks[:, None]
    b = (torch.arange(n, dtype=torch.float64, device=dev)[:, None] + (ks[None, :] % 3)).contiguous()
    bs, bk = b.sum(1), (b * ks[None, :]).sum(1)
    want = rows[None, :] * bs[:, None] + 100 * bk[:, None]
    c = torch.empty(m * n, dtype=torch.float64, device=dev)
    for swap in (False, True):
        for tile in (0, 1, 2):
            c.fill_(float("nan"))
            torch.cuda.synchronize()
            x, y = ((m, a, ak), (n, b, 1)) if not swap else ((n, b, 1), (m, a, ak))
            assert L.talshAmdGemm(T.R8, 0, x[0], y[0], k, x[1].data_ptr(), x[2], y[1].data_ptr(), y[2], c.data_ptr(), 1.0,
                                  0.0, 1, tile, None, 0) == 0
            assert torch.equal(c.view(n, m) if not swap else c.view(m, n).t(), want), (swap, tile)
