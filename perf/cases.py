"""The work whose speed this engine is judged by: contractions, transposes,
scaled additions, block-sparse batches and decompositions, each through the
entry points that a program calls, with operands resident on the GPU.

A case names an operation ("op"), a data kind and either a symbolic pattern
with the extents of its indices or the sizes of that operation. Bodies are
torch tensors handed to the engine as external memory (first tensor dimension
fastest, as the engine stores them), so a pass leaves its result in memory
that the caller owns. Every pass overwrites its results: running it again on
the same inputs gives the same outputs.
"""
import ctypes as C
import math
import random
import re

import torch

from exatensor_amd import talsh as T

KINDS = {"r4": T.R4, "r8": T.R8, "c4": T.C4, "c8": T.C8}
DTYPES = {"r4": torch.float32, "r8": torch.float64, "c4": torch.complex64, "c8": torch.complex128}
SIZES = {"r4": 4, "r8": 8, "c4": 8, "c8": 16}
ARENA_BYTES = 48 << 30  # temporaries and batch descriptors; bodies are torch tensors

BLOCK_PATTERN = "D(a,b,c,d)+=L(a,k,c,l)*R(l,b,k,d)"
BLOCK_EXTENTS = (8, 12, 16, 24, 32, 48, 64)  # segment extents of the block-sparse workload

_engine = None


def engine():
    global _engine
    if _engine is None:
        _engine = T.Engine(gpus=[0], arena_bytes=ARENA_BYTES)
    return _engine


# ---- the cases ----------------------------------------------------------------------


def listed():
    return [
        # one block contraction of the smallest size a block-level caller issues: latency, launches
        dict(name="contract_tiny_r8", op="contract", kind="r8", pattern="D(a,b,c,d)+=L(d,i,b,j)*R(j,c,i,a)",
             extents="a=8,b=8,c=8,d=8,i=8,j=8", terms=1, fast=False),
        # an ordinary tile of a blocked tensor, two terms summed into one result (the second accumulates)
        dict(name="contract_ext32_r8", op="contract", kind="r8", pattern="D(a,b,c,d)+=L(d,i,b,j)*R(j,c,i,a)",
             extents="a=32,b=32,c=32,d=32,i=32,j=32", terms=2, fast=False),
        # orbital counts are seldom round: a particle-particle style term with odd extents
        dict(name="contract_odd_r8", op="contract", kind="r8", pattern="D(a,b,i,j)+=L(a,k,i,l)*R(l,b,k,j)",
             extents="a=53,b=51,i=29,j=31,k=53,l=47", terms=1, fast=False),
        # a tensor-network step in double complex, one operand conjugated
        dict(name="contract_conj_c8", op="contract", kind="c8", pattern="D(a,s,t,b)+=L+(a,k,s,l)*R(k,t,l,b)",
             extents="a=60,s=12,t=12,b=72,k=48,l=20", terms=1, fast=False),
        # one quarter of a four-index transformation: a large tensor times a small matrix (memory-bound)
        dict(name="transform_r8", op="contract", kind="r8", pattern="D(p,q,r,t)+=L(q,s,p,r)*R(s,t)",
             extents="p=60,q=58,r=60,s=62,t=50", terms=1, fast=False),
        # single precision with the three-way split the caller enables for speed, odd free extents
        dict(name="contract_fast_r4", op="contract", kind="r4", pattern="D(a,b,i,j)+=L(a,k,i,l)*R(l,b,k,j)",
             extents="a=66,b=64,i=39,j=40,k=64,l=48", terms=1, fast=True),
        # the benchmark's large contraction, on the FP64 matrix cores
        dict(name="contract_large_r8", op="contract", kind="r8", pattern="D(a,b,i,j)+=L(a,k,i,l)*R(l,b,k,j)",
             extents="a=96,b=96,i=96,j=96,k=128,l=128", terms=1, fast=False),
        # the benchmark's rank-6 tensor under one of its permutations
        dict(name="transpose_rank6_r8", op="transpose", kind="r8", dims="24,24,24,24,24,24", perm="3,5,0,4,1,2"),
        # odd extents, single precision: no side has a run that is a whole number of lines
        dict(name="transpose_odd_r4", op="transpose", kind="r4", dims="37,29,41,23,31", perm="2,4,1,0,3"),
        # spin summation of an amplitude block, 2 T(a,b,i,j) - T(b,a,i,j), assembled with Init and two Adds
        dict(name="add_spinsum_r8", op="add", kind="r8", dims="88,88,44,44", perm="1,0,2,3"),
        # a block-level worker's list of uneven block contractions as one batch, replayed from a graph
        dict(name="blocksparse_r4", op="blocks", kind="r4", segments=7, fill=0.2, ops=4096, structure=2026, fast=False),
        # truncated decomposition of a two-site tensor
        dict(name="svd_twosite_r8", op="svd", kind="r8", left=62, s=3, t=3, right=50, bond=96),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["contract"] * 8 + ["transpose"] * 4 + ["add"] * 2 + ["blocks", "svd"])
    if op == "contract":
        return _draw_contract(rng)
    if op == "blocks":
        kind = rng.choice(["r8", "r4", "r4", "c8"])
        return dict(op=op, kind=kind, segments=rng.randint(3, 6), fill=round(rng.uniform(0.15, 0.4), 3),
                    ops=_spread(rng, 64, 1024), structure=rng.randint(0, 1 << 20),
                    fast=kind == "r4" and rng.random() < 0.5)
    if op == "svd":
        left, right = _spread(rng, 6, 72), _spread(rng, 6, 72)
        s, t = rng.randint(2, 3), rng.randint(2, 3)
        return dict(op=op, kind=rng.choice(["r8", "r8", "c8", "r4"]), left=left, s=s, t=t, right=right,
                    bond=max(2, int(min(left * s, t * right) * rng.uniform(0.4, 1.0))))
    # transposes and additions: ranks 2 to 6, bodies of 64 KB to 2 GB
    kind = rng.choice(["r8", "r8", "r4", "r4", "c8"])
    top = math.log2(2 << 30) - math.log2(SIZES[kind]) - (2 if op == "add" else 0)
    target = rng.uniform(14.0, top)
    while True:
        rank = rng.randint(2, 6)
        dims = [_spread(rng, 3, 2000) for _ in range(rank)]
        if abs(math.log2(math.prod(dims)) - target) > 0.5:
            continue
        perm = list(range(rank))
        if op == "add":  # exchanges two indices of one extent
            i, j = sorted(rng.sample(range(rank), 2))
            dims[j] = dims[i]
            perm[i], perm[j] = j, i
        else:
            rng.shuffle(perm)
        if perm != list(range(rank)) and 14.0 <= math.log2(math.prod(dims)) <= top:
            return dict(op=op, kind=kind, dims=",".join(map(str, dims)), perm=",".join(map(str, perm)))


def _draw_contract(rng):
    """Ranks 2 to 6, every operand with a free and a contracted index, the
    largest tensor of 2^12 to 2^25 elements, at most 2^35 flops."""
    kind, fast = rng.choice([("r8", False)] * 4 + [("r4", False)] * 3 + [("c8", False)] * 2 + [("r4", True)])
    target = rng.uniform(12.0, 25.0 - (1.0 if kind == "c8" else 0.0))
    while True:
        nc, nl, nr = (rng.randint(1, 3) for _ in range(3))
        labels = "abcdefghi"[:nc + nl + nr]
        ext = {x: _spread(rng, 2, 96) for x in labels}
        c, l, r = labels[:nc], labels[nc:nc + nl], labels[nc + nl:]

        def vol(names):
            return math.prod(ext[x] for x in names)
        if abs(math.log2(max(vol(c + l), vol(c + r), vol(l + r))) - target) > 0.5:
            continue
        if math.log2((8.0 if kind == "c8" else 2.0) * vol(labels)) > 35.0:
            continue
        names = [rng.sample(x, len(x)) for x in (l + r, c + l, c + r)]
        conj = ("+" if kind == "c8" and rng.random() < 0.3 else "")
        return dict(op="contract", kind=kind, pattern="D(%s)+=L%s(%s)*R(%s)" % (
            ",".join(names[0]), conj, ",".join(names[1]), ",".join(names[2])),
            extents=",".join("%s=%d" % (x, ext[x]) for x in labels), terms=rng.choice([1, 1, 2]), fast=fast)


# ---- inputs -------------------------------------------------------------------------


def _random(kind, n, gen):
    """n values: uniform in [-1, 1], both components for complex kinds."""
    real = torch.float32 if kind in ("r4", "c4") else torch.float64
    parts = 2 if kind in ("c4", "c8") else 1
    x = torch.rand(n * parts, dtype=real, device="cuda", generator=gen).mul_(2).sub_(1)
    return torch.view_as_complex(x.view(n, 2)) if parts == 2 else x


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _parse(case):
    """(index names of D, L, R; conjugation of L, R; extents by name)."""
    ext = {k: int(v) for k, v in (x.split("=") for x in case["extents"].split(","))}
    names = [g.split(",") for g in re.findall(r"\(([^)]*)\)", case["pattern"])]
    return names, ("L+" in case["pattern"], "R+" in case["pattern"]), ext


def _dims(text):
    return [int(x) for x in text.split(",")]


def _copy_pattern(sign, perm):
    """Pattern whose L index i becomes D index perm[i]."""
    d = [""] * len(perm)
    for i, q in enumerate(perm):
        d[q] = "i%d" % i
    return "D(%s)%sL(%s)" % (",".join(d), sign, ",".join("i%d" % i for i in range(len(perm))))


def _permuted_dims(dims, perm):
    out = [0] * len(dims)
    for i, q in enumerate(perm):
        out[q] = dims[i]
    return out


def _block_structure(case):
    """Segment extents per mode and the (D, L, R) block keys of the batch."""
    rng = random.Random(case["structure"])
    seg = range(case["segments"])
    ext = {m: [rng.choice(BLOCK_EXTENTS) for _ in seg] for m in "abcdkl"}
    left = [(a, k, c, l) for a in seg for k in seg for c in seg for l in seg if rng.random() < case["fill"]]
    right = {(l, b, k, d) for l in seg for b in seg for k in seg for d in seg if rng.random() < case["fill"]}
    ops = [((a, b, c, d), (a, k, c, l), (l, b, k, d)) for a, k, c, l in left for b in seg for d in seg
           if (l, b, k, d) in right]
    if len(ops) > case["ops"]:
        ops = sorted(rng.sample(ops, case["ops"]))
    return ext, ops


def _block_layout(case):
    """Per tensor: {block key: (offset, dims)} in one buffer each (blocks start
    at multiples of 256 bytes) and the buffers' lengths in elements."""
    ext, ops = _block_structure(case)
    align = 256 // SIZES[case["kind"]]
    places, lengths = [], []
    for which, modes in enumerate(("abcd", "akcl", "lbkd")):
        at, place = 0, {}
        for key in sorted({o[which] for o in ops}):
            dims = [ext[m][s] for m, s in zip(modes, key)]
            place[key] = (at, dims)
            at += (math.prod(dims) + align - 1) // align * align
        places.append(place)
        lengths.append(at)
    return ops, places, lengths


def _inputs(case, seed):
    gen, kind = _gen(seed), case["kind"]
    if case["op"] == "contract":
        (_, ln, rn), _, ext = _parse(case)
        return [_random(kind, math.prod(ext[x] for x in names), gen) for _ in range(case["terms"]) for names in (ln, rn)]
    if case["op"] in ("transpose", "add"):
        return [_random(kind, math.prod(_dims(case["dims"])), gen)]
    if case["op"] == "blocks":
        _, _, lengths = _block_layout(case)
        return [_random(kind, lengths[1], gen), _random(kind, lengths[2], gen)]
    # a two-site tensor with singular values that fall over four decades
    rows, cols = case["left"] * case["s"], case["t"] * case["right"]
    n = min(rows, cols)
    weight = torch.logspace(0, -4, n, dtype=torch.float64, device="cuda")
    wide = "c8" if kind in ("c4", "c8") else "r8"
    u = _random(wide, rows * n, gen).view(rows, n)
    v = _random(wide, n * cols, gen).view(n, cols)
    theta = (u * weight) @ v
    return [theta.t().contiguous().view(-1).to(DTYPES[kind])]  # rows fastest


# ---- a program's state and one pass ----------------------------------------------------


class State:
    """Tensors, handles and buffers of one case; released with the object."""

    def __init__(self, case):
        self.case, self.lib = case, engine().lib
        self.gpu = engine().gpu(0)
        self.kind = KINDS[case["kind"]]
        self.tensors, self.batch, self.outputs = [], None, {}

    def wrap(self, body, dims):
        """A tensor of extents dims over the body's memory."""
        t = T.TalshTens()
        self.lib.talshTensorClean(C.byref(t))
        e = self.lib.talshTensorConstruct(C.byref(t), self.kind, len(dims), T.ints(dims), self.gpu,
                                          C.c_void_p(body.data_ptr()), -1, None, 0.0, 0.0)
        if e:
            raise RuntimeError("talshTensorConstruct: %d" % e)
        self.tensors.append((t, body))
        return t

    def empty(self, n):
        return torch.zeros(n, dtype=DTYPES[self.case["kind"]], device="cuda")

    def __del__(self):
        if self.batch is not None:
            self.lib.talshAmdBatchDestroy(self.batch)
        for t, _ in self.tensors:
            self.lib.talshTensorDestruct(C.byref(t))


def prepare(case, seed):
    st = State(case)
    bodies = _inputs(case, seed)
    torch.cuda.synchronize()
    if case["op"] == "contract":
        names, _, ext = _parse(case)
        dims = [[ext[x] for x in n] for n in names]
        out = st.empty(math.prod(dims[0]))
        st.d = st.wrap(out, dims[0])
        st.lr = [(st.wrap(bodies[2 * i], dims[1]), st.wrap(bodies[2 * i + 1], dims[2])) for i in range(case["terms"])]
        st.pattern = case["pattern"].encode()
        st.outputs = {"d": out}
    elif case["op"] in ("transpose", "add"):
        dims, perm = _dims(case["dims"]), _dims(case["perm"])
        out = st.empty(bodies[0].numel())
        st.src = st.wrap(bodies[0], dims)
        st.dst = st.wrap(out, _permuted_dims(dims, perm))
        st.pattern = _copy_pattern("=" if case["op"] == "transpose" else "+=", perm).encode()
        st.same = _copy_pattern("+=", range(len(dims))).encode()
        st.outputs = {"d": out}
    elif case["op"] == "blocks":
        ops, places, lengths = _block_layout(case)
        bufs = [st.empty(lengths[0])] + bodies
        made = []
        for buf, place in zip(bufs, places):
            made.append({key: st.wrap(buf[at:at + math.prod(dims)], dims) for key, (at, dims) in place.items()})
        arrays = [(T._TP * len(ops))(*[C.pointer(made[w][o[w]]) for o in ops]) for w in range(3)]
        if case["fast"]:
            st.lib.talshEnableFastMath(T.DEV_AMD_GPU, 0)
        handle = C.c_void_p()
        torch.cuda.synchronize()
        e = st.lib.talshAmdBatchCreate(BLOCK_PATTERN.encode(), len(ops), *arrays, 1.0, T.NOPE, 0, C.byref(handle))
        if case["fast"]:
            st.lib.talshDisableFastMath(T.DEV_AMD_GPU, 0)
        if e:
            raise RuntimeError("talshAmdBatchCreate: %d" % e)
        st.batch = handle
        st.outputs = {"d": bufs[0]}
    else:
        left, s, t, right, bond = (case[k] for k in ("left", "s", "t", "right", "bond"))
        outs = [st.empty(n) for n in (left * s * bond, bond * t * right, bond)]
        st.d = st.wrap(bodies[0], [left, s, t, right])
        st.l, st.r, st.s = (st.wrap(o, dims) for o, dims in zip(outs, ([left, s, bond], [bond, t, right], [bond])))
        st.outputs = {"left": outs[0], "right": outs[1], "values": outs[2]}
    torch.cuda.synchronize()
    return st


def _check(e, what):
    if e:
        raise RuntimeError("%s: %d" % (what, e))


def run(st):
    lib, case, gpu, b = st.lib, st.case, st.gpu, C.byref
    if case["op"] == "contract":
        if case["fast"]:
            lib.talshEnableFastMath(T.DEV_AMD_GPU, 0)
        for i, (l, r) in enumerate(st.lr):
            _check(lib.talshTensorContract(st.pattern, b(st.d), b(l), b(r), 1.0, 0.0, gpu, T.DEV_NULL, T.COPY_MTT,
                                           T.YEP if i else T.NOPE, None), "talshTensorContract")
        if case["fast"]:
            lib.talshDisableFastMath(T.DEV_AMD_GPU, 0)
    elif case["op"] == "transpose":
        _check(lib.talshTensorCopy(st.pattern, b(st.dst), b(st.src), gpu, T.DEV_NULL, T.COPY_MT, None),
               "talshTensorCopy")
    elif case["op"] == "add":
        _check(lib.talshTensorInit(b(st.dst), 0.0, 0.0, gpu, T.DEV_NULL, T.COPY_M, None), "talshTensorInit")
        _check(lib.talshTensorAdd(st.same, b(st.dst), b(st.src), 2.0, 0.0, gpu, T.DEV_NULL, T.COPY_MT, None),
               "talshTensorAdd")
        _check(lib.talshTensorAdd(st.pattern, b(st.dst), b(st.src), -1.0, 0.0, gpu, T.DEV_NULL, T.COPY_MT, None),
               "talshTensorAdd")
    elif case["op"] == "blocks":
        _check(lib.talshAmdBatchExecute(st.batch, 1), "talshAmdBatchExecute")
    else:
        _check(lib.talshTensorDecomposeSVD(b"D(a,b,c,d)=L(a,b,k)*R(k,c,d)", b(st.d), b(st.l), b(st.r), b(st.s), b"N",
                                           gpu, T.DEV_NULL), "talshTensorDecomposeSVD")
    return st.outputs


# ---- what a pass cannot do without, and its exact result --------------------------------


def work(case):
    es, cx = SIZES[case["kind"]], 4.0 if case["kind"] in ("c4", "c8") else 1.0
    if case["op"] == "contract":
        names, _, ext = _parse(case)
        vols = [math.prod(ext[x] for x in n) for n in names]
        return {"bytes": es * (vols[0] + case["terms"] * (vols[1] + vols[2])),
                "flops": cx * case["terms"] * 2.0 * math.prod(ext.values())}
    if case["op"] in ("transpose", "add"):
        n = math.prod(_dims(case["dims"]))
        return {"bytes": 2 * es * n, "flops": 3.0 * n if case["op"] == "add" else 0.0}
    if case["op"] == "blocks":
        ops, places, _ = _block_layout(case)
        flops = 0.0
        for d, l, r in ops:
            dd, ll = places[0][d][1], places[1][l][1]
            flops += cx * 2.0 * math.prod(dd) * ll[1] * ll[3]
        return {"bytes": es * sum(math.prod(dims) for place in places for _, dims in place.values()), "flops": flops}
    # a singular value decomposition with both factors: about 14 m n^2 + 8 n^3 operations
    m, n = sorted((case["left"] * case["s"], case["t"] * case["right"]), reverse=True)
    return {"bytes": es * (m * n + (m + n) * case["bond"] + case["bond"]), "flops": cx * (14.0 * m * n * n + 8.0 * n ** 3)}


def _full(body, dims):
    """The body as a torch tensor indexed in the order of its dimensions."""
    wide = torch.complex128 if body.is_complex() else torch.float64
    return body.to(wide).view(list(reversed(dims))).permute(list(reversed(range(len(dims)))))


def _flat(x):
    """The values of x with its first dimension fastest."""
    return x.permute(list(reversed(range(x.dim())))).contiguous().view(-1)


def _product(l, ln, r, rn, dn):
    """sum over the shared names of l(ln) r(rn), as a tensor in the order dn."""
    k = [x for x in ln if x in rn]
    lf, rf = [x for x in ln if x not in k], [x for x in rn if x not in k]
    lm = l.permute([ln.index(x) for x in lf + k])
    rm = r.permute([rn.index(x) for x in k + rf])
    shape = list(lm.shape[:len(lf)]) + list(rm.shape[len(k):])
    inner = math.prod(lm.shape[len(lf):])
    d = (lm.reshape(-1, inner) @ rm.reshape(inner, -1)).view(shape)
    return d.permute([(lf + rf).index(x) for x in dn])


def exact(case, seed):
    bodies = _inputs(case, seed)
    if case["op"] == "contract":
        (dn, ln, rn), (lc, rc), ext = _parse(case)
        out = 0
        for i in range(case["terms"]):
            l, r = _full(bodies[2 * i], [ext[x] for x in ln]), _full(bodies[2 * i + 1], [ext[x] for x in rn])
            out = out + _product(l.conj() if lc else l, ln, r.conj() if rc else r, rn, dn)
        return {"d": _flat(out)}
    if case["op"] in ("transpose", "add"):
        dims, perm = _dims(case["dims"]), _dims(case["perm"])
        x = _full(bodies[0], dims)
        inverse = [perm.index(q) for q in range(len(perm))]
        y = x.permute(inverse)
        return {"d": _flat(y if case["op"] == "transpose" else 2.0 * x - y)}
    if case["op"] == "blocks":
        ops, places, lengths = _block_layout(case)
        wide = torch.complex128 if case["kind"] in ("c4", "c8") else torch.float64
        out = torch.zeros(lengths[0], dtype=wide, device="cuda")
        for keys in ops:
            (da, dd), (la, ld), (ra, rd) = (place[key] for place, key in zip(places, keys))
            l = _full(bodies[0][la:la + math.prod(ld)], ld)
            r = _full(bodies[1][ra:ra + math.prod(rd)], rd)
            out[da:da + math.prod(dd)] += _flat(_product(l, list("akcl"), r, list("lbkd"), list("abcd")))
        return {"d": out}
    # the factors are unique up to a phase per singular value, the values are unique
    left, s, t, right = (case[k] for k in ("left", "s", "t", "right"))
    wide = torch.complex128 if case["kind"] in ("c4", "c8") else torch.float64
    theta = bodies[0].to(wide).view(t * right, left * s).cpu()
    values = torch.linalg.svdvals(theta)[:case["bond"]]
    return {"left": None, "right": None, "values": values.to(wide) if wide == torch.complex128 else values}
