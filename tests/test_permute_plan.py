"""Tiles of the permutation kernels, described on the host (talshAmdPermutePlan):
the run form's vectors, counted with the partial one at every run's end, fit
four per thread, and a dimension of many tiles is cut into whole cache lines."""
import numpy as np
import pytest

from exatensor_amd import talsh as T

THREADS, PER_THREAD, LINE = 512, 4, 128
SIZE = {T.R4: 4, T.R8: 8, T.C4: 8, T.C8: 16}


def _plan(kind, dims, o2n):
    lib = T.load_library()
    info = T.ints([0] * 7)
    assert lib.talshAmdPermutePlan(kind, len(dims), T.ints(dims), T.ints(o2n), info) == 0
    return dict(zip(("rank", "path", "vol", "in_run", "out_run", "grid", "vec"), info))


def _vectors(p):
    return max(-(-p[s] // p["vec"]) * (p["vol"] // p[s]) for s in ("in_run", "out_run"))


def test_vectors_per_thread():
    rng = np.random.default_rng(5)
    cases = [(T.R4, [90, 4000, 95], [1, 2, 0])]
    for _ in range(3000):
        n = int(rng.integers(2, 7))
        dims = [int(x) for x in np.rint(np.exp(rng.uniform(np.log(2), np.log(150), n)))]
        cases.append((int(rng.choice(list(SIZE))), dims, [int(x) for x in rng.permutation(n)]))
    seen = 0
    for kind, dims, o2n in cases:
        p = _plan(kind, dims, o2n)
        if p["path"] != 1 or all(p[s] * SIZE[kind] % LINE == 0 for s in ("in_run", "out_run")):
            continue  # whole lines on both sides: the vector form, which holds up to eight
        seen += 1
        assert _vectors(p) <= THREADS * PER_THREAD, (kind, dims, o2n, p)
    assert seen > 500


@pytest.mark.parametrize("kind,dims,o2n", [
    (T.C4, [2350648, 16], [1, 0]),
    (T.C8, [8132, 2, 32, 5, 7], [2, 4, 3, 0, 1]),
    (T.C4, [3014, 6, 8, 32, 2, 6], [4, 3, 0, 5, 1, 2]),
    (T.R4, [4001, 4003], [1, 0]),
])
def test_long_dimensions_are_cut_in_lines(kind, dims, o2n):
    p = _plan(kind, dims, o2n)
    assert p["path"] == 1 and p["in_run"] * SIZE[kind] % LINE == 0, p
