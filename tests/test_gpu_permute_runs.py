"""Permutations and permuted additions by runs: odd and tiny extents, tiles
that overlap along every dimension, runs of several dimensions, bodies aligned
to one element only, operands that overlap in memory. Copies bit for bit,
additions equal to separately rounded products and sums (numpy in the data
kind's own precision)."""
import ctypes as C

import numpy as np
import pytest

from exatensor_amd import talsh as T
from gpu_util import engine

pytestmark = pytest.mark.gpu

SHAPES = [
    ((2, 2), (1, 0)),
    ((3, 5), (1, 0)),
    ((1, 7, 1, 3), (3, 2, 1, 0)),
    ((129, 127), (1, 0)),
    ((1023, 1025), (1, 0)),
    ((5, 3, 7, 11, 13), (4, 2, 0, 3, 1)),
    ((37, 29, 41, 23), (2, 3, 1, 0)),
    ((67, 31, 29), (0, 2, 1)),
    ((2, 3, 2, 3, 2, 3, 2, 3, 2, 3, 2), (10, 8, 6, 4, 2, 0, 1, 3, 5, 7, 9)),
    ((31, 2, 65, 66), (3, 0, 2, 1)),
    ((4099, 3, 5), (2, 0, 1)),
    ((6, 4001), (1, 0)),
    ((128, 64, 32), (2, 1, 0)),   # whole lines: the vector form
]


def _pattern(perm, sign, conj=False):
    d = [""] * len(perm)
    for i, q in enumerate(perm):
        d[q] = "i%d" % i
    return ("D(%s)%sL%s(%s)" % (",".join(d), sign, "+" if conj else "", ",".join("i%d" % i for i in range(len(perm))))).encode()


def _wrap(L, ptr, kind, dims):
    t = T.TalshTens()
    L.talshTensorClean(C.byref(t))
    assert L.talshTensorConstruct(C.byref(t), kind, len(dims), T.ints(dims), engine().gpu(0), C.c_void_p(ptr), -1, None,
                                  0.0, 0.0) == 0
    return t


def _axpy(d, x, f):
    """d + f x, every product and sum rounded in the kind's precision."""
    if not np.iscomplexobj(d):
        return d + x * d.dtype.type(f.real)
    r = d.real.dtype.type
    fr, fi = r(f.real), r(f.imag)
    out = np.empty_like(d)
    out.real = d.real + (x.real * fr - x.imag * fi)
    out.imag = d.imag + (x.real * fi + x.imag * fr)
    return out


@pytest.mark.parametrize("kind", [T.R4, T.R8, T.C4, T.C8])
@pytest.mark.parametrize("shift", [0, 1])
def test_copy_and_add(kind, shift):
    import torch
    L, gpu = engine().lib, engine().gpu(0)
    dt = T.NP_DTYPE[kind]
    f = complex(-0.75, 0.5 if kind in (T.C4, T.C8) else 0.0)
    for si, (dims, perm) in enumerate(SHAPES):
        n = int(np.prod(dims))
        rng = np.random.default_rng(100 * si + kind)
        mk = lambda: (rng.uniform(-1, 1, n) + (1j * rng.uniform(-1, 1, n) if kind in (T.C4, T.C8) else 0)).astype(dt)
        x, d0 = mk(), mk()
        od = [0] * len(dims)
        for i, q in enumerate(perm):
            od[q] = dims[i]
        inv = [perm.index(q) for q in range(len(perm))]
        want = np.transpose(x.reshape(dims, order="F"), inv).ravel(order="F")
        # bodies one element into their buffers (shift) end one element before their buffers' ends
        guard = np.full(1, 7, dt)
        bx = torch.from_numpy(np.concatenate([guard] * shift + [x, guard])).cuda()
        for conj in ((False, True) if kind in (T.C4, T.C8) else (False,)):
            w = np.conj(want) if conj else want
            for sign, res in (("=", w), ("+=", _axpy(d0, w, f))):
                bd = torch.from_numpy(np.concatenate([guard] * shift + [d0, guard])).cuda()
                torch.cuda.synchronize()
                tl = _wrap(L, bx.data_ptr() + shift * dt().itemsize, kind, dims)
                td = _wrap(L, bd.data_ptr() + shift * dt().itemsize, kind, od)
                p = _pattern(perm, sign, conj)
                if sign == "=":
                    e = L.talshTensorCopy(p, C.byref(td), C.byref(tl), gpu, T.DEV_NULL, T.COPY_MT, None)
                else:
                    e = L.talshTensorAdd(p, C.byref(td), C.byref(tl), f.real, f.imag, gpu, T.DEV_NULL, T.COPY_MT, None)
                assert e == 0, (dims, perm, sign, e)
                got = bd.cpu().numpy()
                assert np.all(got[:shift] == 7) and got[-1] == 7, (dims, perm, sign)
                same = got[shift:-1]
                if sign == "=" or not np.any(same != res):
                    assert same.tobytes() == res.tobytes() or (sign == "+=" and np.array_equal(same, res)), (dims, perm, sign)
                else:
                    raise AssertionError((dims, perm, conj, float(np.max(np.abs(same - res)))))
                L.talshTensorDestruct(C.byref(tl))
                L.talshTensorDestruct(C.byref(td))


def test_add_of_a_tensor_to_itself():
    """D(b,a) += f D(a,b) over one body: the sum takes the permuted copy."""
    import torch
    L, gpu = engine().lib, engine().gpu(0)
    n = 77
    x = np.random.default_rng(4).uniform(-1, 1, n * n)
    b = torch.from_numpy(x.copy()).cuda()
    torch.cuda.synchronize()
    t1, t2 = _wrap(L, b.data_ptr(), T.R8, (n, n)), _wrap(L, b.data_ptr(), T.R8, (n, n))
    e = L.talshTensorAdd(b"D(b,a)+=L(a,b)", C.byref(t1), C.byref(t2), 0.5, 0.0, gpu, T.DEV_NULL, T.COPY_MT, None)
    assert e == 0
    m = x.reshape(n, n, order="F")
    assert np.array_equal(b.cpu().numpy().reshape(n, n, order="F"), m + m.T * 0.5)
    for t in (t1, t2):
        L.talshTensorDestruct(C.byref(t))


def test_permuted_addition_is_profiled():
    """An addition that permutes is a launch of the transpose class, in one pass
    or (over overlapping bodies) with a permuted copy."""
    import torch
    L, gpu = engine().lib, engine().gpu(0)
    n = 33
    b = torch.zeros(3 * n * n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ms, count = C.c_double(), C.c_longlong()
    L.talshAmdProfile(1)
    try:
        for at in (0, n, 2 * n * n):  # the same body, overlapping, apart
            t1, t2 = _wrap(L, b.data_ptr(), T.R8, (n, n)), _wrap(L, b.data_ptr() + 8 * at, T.R8, (n, n))
            L.talshAmdProfileQuery(T.KERNEL_TRANSPOSE, C.byref(ms), C.byref(count))
            assert L.talshTensorAdd(b"D(b,a)+=L(a,b)", C.byref(t1), C.byref(t2), 0.5, 0.0, gpu, T.DEV_NULL, T.COPY_MT, None) == 0
            L.talshAmdProfileQuery(T.KERNEL_TRANSPOSE, C.byref(ms), C.byref(count))
            assert count.value == 1 and ms.value > 0, at
            for t in (t1, t2):
                L.talshTensorDestruct(C.byref(t))
    finally:
        L.talshAmdProfile(0)
