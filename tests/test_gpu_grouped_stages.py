"""Chains of the grouped kernel whose block products have contracted extents on
either side of a 16-wide and a 32-wide k-stage, in both orders (a half stage in
the middle and at the end of a chain), with rows and columns on either side of a
64-wide tile, against float64 / complex128 sums."""
import ctypes as C

import numpy as np
import pytest

from exatensor_amd import talsh as T
from gpu_util import engine, gpu_tensor, rel_err

pytestmark = pytest.mark.gpu

TOL = {T.R8: 1e-13, T.C8: 1e-13, T.R4: 1e-5, T.C4: 1e-5}
CHAINS = [(1,), (16, 17), (48,), (33, 5, 64), (32, 48, 16, 1, 96), (80, 80)]


@pytest.mark.parametrize("kind", [T.R8, T.R4, T.C8, T.C4])
@pytest.mark.parametrize("m,n", [(1, 1), (63, 65), (64, 130), (129, 3)])
def test_chain_stages(kind, m, n):
    lib = engine().lib
    rng = np.random.default_rng(m * 1000 + n)
    cx = kind in (T.C4, T.C8)
    wide = np.complex128 if cx else np.float64

    def block(*dims):
        x = rng.uniform(-1, 1, dims) + (1j * rng.uniform(-1, 1, dims) if cx else 0)
        x = x.astype(T.NP_DTYPE[kind])
        return x, gpu_tensor(x.ravel(order="F"), list(dims))

    outs, tens, D, L, R = [], [], [], [], []
    for chain in CHAINS:
        d, td = block(m, n)
        want = d.astype(wide)
        for k in chain:
            (l, tl), (r, tr) = block(m, k), block(k, n)
            want = want + 0.75 * (l.astype(wide) @ r.astype(wide))
            D.append(td); L.append(tl); R.append(tr)
            tens += [tl, tr]
        outs.append((chain, td, want))
        tens.append(td)
    nops = len(D)
    arr = lambda ts: (T._TP * nops)(*[C.pointer(t.t) for t in ts])
    b = C.c_void_p()
    assert lib.talshAmdBatchCreate(b"D(a,b)+=L(a,k)*R(k,b)", nops, arr(D), arr(L), arr(R), 0.75, T.YEP, 0, C.byref(b)) == 0
    assert lib.talshAmdBatchExecute(b, 0) == 0
    assert lib.talshAmdBatchDestroy(b) == 0
    for chain, td, want in outs:
        assert rel_err(td.download(), want.ravel(order="F")) <= TOL[kind], chain
    for t in tens:
        t.destruct()
