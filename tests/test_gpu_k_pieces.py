"""Native-precision contractions whose leftover tiles are cut along K: a little
over one round of 64x64 and 128x128 tiles with ragged rows, columns and k, so
whole tiles, padded partials and a chain of tiles in pieces occur together,
accumulating and not. Against float64 / complex128 products; and in an arena
with no room for the partials, bit for bit what the same call gives in an empty
one, also with several such tasks in flight on the engine's streams.

Bounds: the pieces' sums are held in the kind's own precision and added in
FP64, so the error is that of an uncut product, a few roundings times the
square root of k, as in the tests of the uncut walks."""
import ctypes as C

import numpy as np
import pytest

from exatensor_amd import talsh as T
from gpu_util import engine

pytestmark = pytest.mark.gpu

TOL = {T.R8: 1e-13, T.C8: 1e-13, T.R4: 1e-5}
PAT = b"D(a,b)%s=L(k,a)*R(k,b)"
# kind, tile choice, m, n, k
CASES = [
    (T.R8, 1, 1030, 1111, 3001),
    (T.R8, 2, 1990, 1111, 2999),
    (T.R8, 0, 2999, 3001, 1537),
    (T.R4, 1, 1030, 1111, 3001),
    (T.R4, 2, 1990, 1111, 3000),
    (T.R4, 0, 2999, 3001, 1537),
    (T.C8, 0, 1030, 1111, 701),
]


def _wrap(L, x, dims, kind):
    t = T.TalshTens()
    L.talshTensorClean(C.byref(t))
    assert L.talshTensorConstruct(C.byref(t), kind, len(dims), T.ints(dims), engine().gpu(0), C.c_void_p(x.data_ptr()),
                                  -1, None, 0.0, 0.0) == 0
    return t


def _parts(L, kind, tile, m, n, k, acc):
    """Pieces of K that the planner's description gives the forced plan."""
    nf = L.talshAmdPlanFeatureCount()
    v, t, f, nc = (C.c_int * 64)(), (C.c_int * 64)(), (C.c_float * (64 * nf))(), C.c_int()
    assert L.talshAmdPlanFeatures(PAT % (b"+" if acc else b""), 2, T.ints([m, n]), 2, T.ints([k, m]), 2, T.ints([k, n]),
                                  kind, T.YEP if acc else T.NOPE, 0, 64, v, t, f, C.byref(nc)) == 0
    i = [j for j in range(nc.value) if v[j] == 0 and t[j] == tile][0]
    return round(2.0 ** f[i * nf + 53])


class _FullArena:
    """Holds the arena's free blocks down to less than a MiB each."""

    def __enter__(self):
        L, gpu = engine().lib, engine().gpu(0)
        self.held = []
        while True:
            n = L.talshDeviceTensorSize(0, T.DEV_AMD_GPU) // 8
            if n < 1 << 17:
                return self
            t = T.Tensor(L, T.R8, [min(n, 1 << 30)], gpu)
            assert t.err == 0, t.err
            self.held.append(t)

    def __exit__(self, *a):
        for t in self.held:
            t.destruct()


@pytest.mark.parametrize("kind,tile,m,n,k", CASES)
def test_pieces_of_k(kind, tile, m, n, k):
    import torch
    L, gpu = engine().lib, engine().gpu(0)
    dt = {T.R8: torch.float64, T.R4: torch.float32, T.C8: torch.complex128}[kind]
    wide = torch.complex128 if kind == T.C8 else torch.float64
    gen = torch.Generator(device="cuda").manual_seed(m + k)

    def rand(rows, cols):
        x = torch.rand(rows, cols, dtype=torch.float64, device="cuda", generator=gen) - 0.5
        if kind == T.C8:
            x = torch.complex(x, torch.rand(rows, cols, dtype=torch.float64, device="cuda", generator=gen) - 0.5)
        return x.to(dt)

    a, b, d = rand(m, k), rand(n, k), rand(n, m)  # bodies with k, k and D's rows fastest
    prod = (b.to(wide) @ a.to(wide).t().contiguous())
    try:
        L.talshAmdSetPlanVariant(0, tile)
        for acc in (True, False):
            assert _parts(L, kind, tile, m, n, k, acc) > 1
            want = prod + d.to(wide) if acc else prod
            outs = []
            for full in (False, True):
                nt = 4 if full else 1
                ds = [d.clone() if acc else torch.full_like(d, float("nan")) for _ in range(nt)]
                torch.cuda.synchronize()
                ts = [(_wrap(L, x, [m, n], kind), _wrap(L, a, [k, m], kind), _wrap(L, b, [k, n], kind), T.TalshTask())
                      for x in ds]
                held = _FullArena().__enter__() if full else None
                try:
                    for D, A, B, task in ts:
                        L.talshTaskClean(C.byref(task))
                        assert L.talshTensorContract(PAT % (b"+" if acc else b""), C.byref(D), C.byref(A), C.byref(B), 1.0,
                                                     0.0, gpu, T.DEV_NULL, T.COPY_MTT, T.YEP if acc else T.NOPE,
                                                     C.byref(task)) == 0
                    st = C.c_int()
                    for D, A, B, task in ts:
                        assert L.talshTaskWait(C.byref(task), C.byref(st)) == 0 and st.value == T.TALSH_TASK_COMPLETED
                        assert L.talshTaskDestruct(C.byref(task)) == 0
                finally:
                    if held:
                        held.__exit__()
                outs += ds
                for q in ts:
                    for t in q[:3]:
                        L.talshTensorDestruct(C.byref(t))
            err = float(torch.linalg.norm(outs[0].to(wide) - want) / torch.linalg.norm(want))
            assert err <= TOL[kind], (acc, err)
            for x in outs[1:]:
                assert torch.equal(outs[0], x), acc
    finally:
        L.talshAmdSetPlanVariant(-1, -1)
