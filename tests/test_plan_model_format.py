"""Plan model files name the format of their features: the shipped model and a
saved one carry the present format; one of the format before is still accepted,
keeps its format, and installing it says so on stderr."""
import ctypes as C

from exatensor_amd import selector as S
from exatensor_amd import talsh as T


def _tag(path):
    with open(path) as f:
        return f.readline().split()


def test_formats(tmp_path, capfd):
    L = T.load_library()
    now = _tag(S.DEFAULT_MODEL)
    assert now[0] == "talsh_plan_mlp"
    m = C.c_void_p()
    assert L.talshAmdMlpCreate(L.talshAmdPlanFeatureCount(), 1, 8, 5, C.byref(m)) == 0
    p = str(tmp_path / "m.txt")
    assert L.talshAmdMlpSave(m, p.encode()) == 0 and _tag(p) == now
    L.talshAmdMlpDestroy(m)
    with open(p) as f:
        body = f.read().split("\n", 1)[1]
    for fmt, accepted in ((int(now[1]), True), (1, True), (0, False), (int(now[1]) + 1, False)):
        q = str(tmp_path / ("f%d.txt" % fmt))
        with open(q, "w") as f:
            f.write("talsh_plan_mlp %d\n%s" % (fmt, body))
        assert (L.talshAmdMlpLoad(q.encode(), C.byref(m)) == 0) == accepted, fmt
        if not accepted:
            continue
        capfd.readouterr()
        try:
            assert L.talshAmdSelectorInstall(m) == 0
        finally:
            L.talshAmdSelectorInstall(None)
        assert ("format 1" in capfd.readouterr().err) == (fmt == 1)
        assert L.talshAmdMlpSave(m, (q + "s").encode()) == 0 and _tag(q + "s")[1] == str(fmt)
        L.talshAmdMlpDestroy(m)
