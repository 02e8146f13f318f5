"""Index walks of the native-precision matrix kernels: contracted groups of one
to five dimensions with odd extents (carries, the offset tables beyond three
dimensions and for runs that are no multiple of a k-tile, the long argument
form), k-tails on both sides of a k-tile and of a workgroup's share of them,
row and column edges, and operands of more than 4 GB, against float64 /
complex128 products."""
import ctypes as C

import numpy as np
import pytest

from exatensor_amd import talsh as T
from gpu_util import contract, engine, rel_err

pytestmark = pytest.mark.gpu

TOL = {T.R8: 1e-13, T.C8: 1e-13, T.R4: 1e-5, T.C4: 1e-5}


def _rand(rng, kind, dims):
    x = rng.uniform(-1, 1, dims)
    if kind in (T.C4, T.C8):
        x = x + 1j * rng.uniform(-1, 1, dims)
    return x.astype(T.NP_DTYPE[kind])


# contracted extents (in L's order), whether L / R hold their stride-1 index among them, free extents of L and R
WALKS = [
    ((7, 5), True, True, (65,), (9, 13)),
    ((7, 5, 3), True, False, (33, 3), (67,)),
    ((3, 5, 7, 2), False, True, (5, 13), (64,)),
    ((2, 3, 5, 2, 3), True, True, (63,), (31, 2)),
    ((3, 2, 3, 2, 3), False, False, (3, 43), (1, 65)),
    ((16, 3), True, True, (64,), (64,)),
    ((32, 5), True, False, (66,), (130,)),
    ((48, 2, 3), False, True, (130,), (18,)),
]


@pytest.mark.parametrize("kind", [T.R8, T.R4, T.C8, T.C4])
@pytest.mark.parametrize("ks,lk,rk,lf,rf", WALKS)
def test_contracted_groups(kind, ks, lk, rk, lf, rf):
    L = engine().lib
    rng = np.random.default_rng(len(ks) * 100 + ks[0])
    names = "klmno"[:len(ks)]
    ln, rn = "ab"[:len(lf)], "xy"[:len(rf)]
    ext = dict(zip(names + ln + rn, ks + lf + rf))
    # R's contracted indices reversed: L's runs along k do not line up with R's
    lord, rord = (names + ln if lk else ln + names), (names[::-1] + rn if rk else rn + names[::-1])
    dord = rn[::-1] + ln
    dims = {t: [ext[x] for x in o] for t, o in (("D", dord), ("L", lord), ("R", rord))}
    l, r, d = (_rand(rng, kind, dims[t]) for t in "LRD")
    wide = np.complex128 if kind in (T.C4, T.C8) else np.float64
    want = d.astype(wide) + 0.5 * np.einsum(f"{lord},{rord}->{dord}", l.astype(wide), r.astype(wide), optimize=True)
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


@pytest.mark.parametrize("kind", [T.R8, T.R4, T.C8])
@pytest.mark.parametrize("k", [1, 2, 8, 15, 16, 17, 24, 31, 33, 63, 64, 65, 72, 127, 130, 264])
def test_k_tails(kind, k):
    """Products of 66 x 62 (edges of 64-wide tiles, even: pair loads where k
    allows) and 65 x 129, every orientation and tile choice, K uncut (pieces of
    K: test_gpu_k_pieces.py)."""
    import torch
    L = engine().lib
    cx = kind == T.C8
    dt = {T.R8: torch.float64, T.R4: torch.float32, T.C8: torch.complex128}[kind]
    for m, n in ((66, 62), (65, 129)):
        gen = torch.Generator(device="cuda").manual_seed(k * 1000 + m)
        a, b = (torch.rand(x * k * (2 if cx else 1), dtype=torch.float64, device="cuda", generator=gen) - 0.5 for x in (m, n))
        a, b = ((torch.view_as_complex(x.view(-1, 2)) if cx else x).to(dt) for x in (a, b))
        for ak in (0, 1):
            for bk in (0, 1):
                A = a.view(m, k) if ak else a.view(k, m).t()
                B = b.view(n, k) if bk else b.view(k, n).t()
                wide = torch.complex128 if cx else torch.float64
                want = (A.to(wide).cpu() @ B.to(wide).cpu().t()).t().contiguous().view(-1).numpy()
                for tile in ((0,) if cx else (0, 1, 2)):
                    c = torch.full((m * n,), 7.0, dtype=dt, device="cuda")
                    torch.cuda.synchronize()
                    e = L.talshAmdGemm(kind, 0, m, n, k, a.data_ptr(), ak, b.data_ptr(), bk, c.data_ptr(), 1.0, 0.0, 1,
                                       tile, None, 0)
                    assert e == 0
                    assert rel_err(c.cpu().numpy(), want) <= TOL[kind], (m, n, ak, bk, tile)


@pytest.mark.parametrize("ak", [1, 0])
def test_operand_beyond_4gb(ak):
    """A is 4.6 GB: its rows and k-values are told apart by whole numbers that
    the sums keep exactly."""
    import torch
    L = engine().lib
    m, n, k = 70001, 40, 8195
    dev = "cuda"
    rows = torch.arange(m, dtype=torch.float64, device=dev) % 97
    ks = torch.arange(k, dtype=torch.float64, device=dev) % 11
    a = rows[:, None] + 100 * ks[None, :] if ak else rows[None, :] + 100 * ks[:, None]
    b = (torch.arange(n, dtype=torch.float64, device=dev)[:, None] + (ks[None, :] % 3)).contiguous()
    c = torch.zeros(m * n, dtype=torch.float64, device=dev)
    torch.cuda.synchronize()
    e = L.talshAmdGemm(T.R8, 0, m, n, k, a.data_ptr(), ak, b.data_ptr(), 1, c.data_ptr(), 1.0, 0.0, 1, -1, None, 0)
    assert e == 0
    bs = b.sum(1)
    want = rows[None, :] * bs[:, None] + 100 * (b * ks[None, :]).sum(1)[:, None]
    assert torch.equal(c.view(n, m), want)
