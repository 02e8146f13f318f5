"""The decomposition on matrices of every regime of its sweeps: all columns in
one workgroup's LDS, windows of columns that neighbours share, one launch per
round (columns too long for a window of twelve pairs); odd and even numbers of
columns, tall and wide, real and complex. Singular values against numpy's,
orthonormal factors, reconstruction."""
import numpy as np
import pytest

from exatensor_amd import talsh as T
from gpu_util import engine, gpu_tensor

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2), (3, 2), (17, 17), (64, 33), (96, 96), (186, 150), (150, 186), (300, 97), (257, 40), (40, 257),
          (1500, 31), (5000, 7), (12000, 6)]


@pytest.mark.parametrize("kind", [T.R8, T.C8, T.R4])
@pytest.mark.parametrize("rows,cols", SHAPES)
def test_windows(kind, rows, cols):
    eng = engine()
    lib = eng.lib
    rng = np.random.default_rng(rows * 1000 + cols)
    n = min(rows, cols)
    u, v = rng.uniform(-1, 1, (rows, n)), rng.uniform(-1, 1, (n, cols))
    if kind == T.C8:
        u, v = u + 1j * rng.uniform(-1, 1, u.shape), v + 1j * rng.uniform(-1, 1, v.shape)
    a = ((u * np.logspace(0, -3, n)) @ v).astype(T.NP_DTYPE[kind])
    td = gpu_tensor(a.ravel(order="F"), [rows, cols])
    tl = gpu_tensor(np.zeros(rows * n, T.NP_DTYPE[kind]), [rows, n])
    tr = gpu_tensor(np.zeros(n * cols, T.NP_DTYPE[kind]), [n, cols])
    ts = gpu_tensor(np.zeros(n, T.NP_DTYPE[kind]), [n])
    e = lib.talshTensorDecomposeSVD(b"D(a,b)=L(a,k)*R(k,b)", td.ptr, tl.ptr, tr.ptr, ts.ptr, b"N", eng.gpu(0), T.DEV_NULL)
    assert e == 0
    L = tl.download().reshape((rows, n), order="F").astype(np.complex128)
    R = tr.download().reshape((n, cols), order="F").astype(np.complex128)
    S = ts.download().real.astype(np.float64)
    for t in (td, tl, tr, ts):
        t.destruct()
    tol = 2e-4 if kind == T.R4 else 1e-12
    want = np.linalg.svd(a.astype(np.complex128), compute_uv=False)
    assert np.max(np.abs(S - want)) <= tol * want[0]
    assert np.linalg.norm(L.conj().T @ L - np.eye(n)) <= tol * n
    assert np.linalg.norm(R @ R.conj().T - np.eye(n)) <= tol * n
    assert np.linalg.norm((L * S) @ R - a) <= tol * np.linalg.norm(a)
