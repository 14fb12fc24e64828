"""The work that a user of this backend has it do, as cases that can be timed.

A case is one compiled plan and the tensors it is bound to; one pass is one
HipPlan.run() on buffers that already lie in device memory.  The schedules are the
reference scheduler's: for the sizes that polygrad_amd/plans ships they are those
files kernel by kernel (same ranges, buffers and arithmetic), for every other size
they are put together here in the same form and handed over as plan files.

    gpt2     GPT-2 forward, whole model: prefill of long, ragged and short prompts
             (without a key cache a short prompt is also what decoding runs), 16-bit
             weights as the headline benchmark has them, or fp32 as the reference's
             own builder makes them
    train    one GPT-2 medium block with head and loss: forward, backward and AdamW
    mlp      two-layer classifier: forward, backward and SGD step in fp32
    adamw    optimizer update of a flat fp32 parameter
    rows     elementwise chain into a row sum, row max, softmax or LayerNorm, fp32
    matmul   C = A B in bf16, fp16 or fp32 with fp32 result, the operand layouts of a
             linear layer's forward and backward
"""
import math
import os
import struct
import tempfile

import torch

import polygrad_amd
from polygrad_amd import HipPlan
from polygrad_amd.inputs import torch_dtype

PLANS = os.path.join(os.path.dirname(os.path.abspath(polygrad_amd.__file__)), "plans")
VOCAB = 50257


# ── the cases ────────────────────────────────────────────────────────────────

def _gpt2(batch, ctx, dtype, layers=12, heads=12, d_model=768):
    return dict(kind="gpt2", batch=batch, ctx=ctx, dtype=dtype, layers=layers, heads=heads, d_model=d_model)


def listed():
    return [
        # the headline: GPT-2 small over a full batch of full contexts
        dict(name="gpt2_small_bf16_b8_t1024", **_gpt2(8, 1024, "bfloat16")),
        # a few prompts of some length that no tile divides
        dict(name="gpt2_small_bf16_b3_t345", **_gpt2(3, 345, "bfloat16")),
        # one short prompt: launches and weight reads
        dict(name="gpt2_small_bf16_b1_t12", **_gpt2(1, 12, "bfloat16")),
        # the same model as the reference's builder makes it, in fp32
        dict(name="gpt2_small_f32_b1_t128", **_gpt2(1, 128, "float32")),
        # training of a transformer block: mixed precision forward, backward, AdamW
        dict(name="gpt2_medium_block_train_b4_t1024", kind="train"),
        # training of a small classifier, at the benchmark's batch and at a small odd one
        dict(name="mlp_train_f32_b4096", kind="mlp", batch=4096, d_in=784, d_hid=512, d_out=10),
        dict(name="mlp_train_f32_b33", kind="mlp", batch=33, d_in=784, d_hid=129, d_out=10),
        # the optimizer step of GPT-2 medium
        dict(name="adamw_f32_355m", kind="adamw", numel=354823168),
        # row operations: the benchmark's, and rows of odd length
        dict(name="softmax_f32_8192x8192", kind="rows", op="softmax", rows=8192, cols=8192),
        dict(name="layernorm_f32_4097x1001", kind="rows", op="layernorm", rows=4097, cols=1001),
        # products: the benchmark's, and one with all three extents odd
        dict(name="matmul_bf16_4096x4096x4096", kind="matmul", m=4096, n=4096, k=4096, dtype="bfloat16", layout="nn"),
        dict(name="matmul_bf16_1111x999x1501", kind="matmul", m=1111, n=999, k=1501, dtype="bfloat16", layout="nn"),
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]; odd as often as not, and now and then a
    multiple of 64, which sizes in use often are."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if n >= 128 and rng.random() < 0.3:
        n = n // 64 * 64
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["gpt2", "gpt2", "mlp", "adamw", "rows", "rows", "matmul", "matmul", "matmul"])
    if kind == "gpt2":
        dtype = rng.choice(["bfloat16", "bfloat16", "float32"])
        ctx = _log(rng, 2, 1024 if dtype == "bfloat16" else 256)
        batch = _log(rng, 1, max(1, min(8, (8192 if dtype == "bfloat16" else 512) // ctx)))
        if rng.random() < 0.3:
            return _gpt2(min(batch, 4), ctx, dtype, layers=rng.randint(1, 12), heads=16, d_model=1024)
        return _gpt2(batch, ctx, dtype, layers=rng.choice([2, 4, 6, 12]))
    if kind == "mlp":
        return dict(kind=kind, batch=_log(rng, 2, 4096), d_in=_log(rng, 8, 1024), d_hid=_log(rng, 8, 1024), d_out=_log(rng, 2, 100))
    if kind == "adamw":
        return dict(kind=kind, numel=_log(rng, 1000, 354823168))
    if kind == "rows":
        cols = _log(rng, 8, 50257)
        return dict(kind=kind, op=rng.choice(["sum", "max", "softmax", "layernorm"]), rows=_log(rng, 4, max(4, min(65536, (1 << 26) // cols))), cols=cols)
    dtype = rng.choice(["bfloat16", "bfloat16", "float16", "float32"])
    top = 8192 if dtype != "float32" else 2048
    m, n, k = (_log(rng, 16, top) for _ in range(3))
    while m * n * k > 4096 ** 3:
        m, n, k = max(16, m // 2), max(16, n // 2), max(16, k // 2)
    return dict(kind=kind, m=m, n=n, k=k, dtype=dtype, layout=rng.choice(["nn", "nn", "nt", "tn"]))


# ── schedules ────────────────────────────────────────────────────────────────
#
# What the reference's scheduler hands a backend: kernels SINK(END*(STORE(INDEX(PARAM, i), v),
# RANGE...)) over numbered buffers.  Op and dtype codes are those of include/polygrad_abi.h,
# the file layout that of csrc/planfile.cc.

_OPS = dict(PARAM=8, SINK=14, INDEX=19, LOAD=20, STORE=21, CAST=23, EXP2=25, LOG2=26, SQRT=28, RECIPROCAL=29, NEG=30, ADD=32, MUL=33, IDIV=36,
            MAX=37, MOD=38, CMPLT=39, CMPNE=40, SUB=46, FDIV=47, WHERE=49, RANGE=52, END=54, CONST=57)
_REDUCE = 83
_DT = dict(void=0, bool=1, int32=6, float16=10, bfloat16=11, float32=12)
_SIZE = dict(bool=1, int32=4, float16=2, bfloat16=2, float32=4)
F32 = "float32"
LOG2E, LN2 = 1.4426950408889634, 0.6931471805599453


class E:
    """A node of a kernel's expression graph."""
    __slots__ = ("op", "dt", "src", "arg", "extent")

    def __init__(self, op, dt, src=(), arg=None, extent=None):
        self.op, self.dt, self.src, self.arg, self.extent = op, dt, tuple(src), arg, extent

    def _bin(self, op, o, dt=None):
        return E(op, dt or self.dt, (self, const(o, self.dt)))

    def __add__(self, o): return self if self.dt == "int32" and _is_zero(o) else self._bin("ADD", o)
    def __mul__(self, o): return self._bin("MUL", o)
    def __rmul__(self, o): return const(o, self.dt)._bin("MUL", self)
    def __radd__(self, o): return const(o, self.dt)._bin("ADD", self)
    def __sub__(self, o): return self._bin("SUB", o)
    def __truediv__(self, o): return self._bin("FDIV", o)
    def __floordiv__(self, o): return self._bin("IDIV", o)
    def __mod__(self, o): return self._bin("MOD", o)
    def __neg__(self): return E("NEG", self.dt, (self,))
    def lt(self, o): return self._bin("CMPLT", o, "bool")
    def ne(self, o): return self._bin("CMPNE", o, "bool")
    def un(self, op): return E(op, self.dt, (self,))
    def cast(self, dt): return self if dt == self.dt else E("CAST", dt, (self,))


def _is_zero(o):
    return (o.op == "CONST" and o.arg == 0) if isinstance(o, E) else o == 0


def const(v, dt="int32"):
    return v if isinstance(v, E) else E("CONST", dt, arg=v)


def where(c, a, b):
    t = a if isinstance(a, E) else b
    return E("WHERE", t.dt, (c, const(a, t.dt), const(b, t.dt)))


class Buf:
    def __init__(self, index, name, dt, numel):
        self.index, self.name, self.dt, self.numel = index, name, dt, numel

    def __getitem__(self, i):
        return E("LOAD", self.dt, (E("INDEX", self.dt, (E("PARAM", self.dt, arg=self), const(i))),))


class Schedule:
    def __init__(self):
        self.bufs, self.items, self._axis = [], [], 0

    def buf(self, name, numel, dt=F32):
        """A buffer of the caller's, or with no name an intermediate."""
        self.bufs.append(Buf(len(self.bufs), name, dt, numel))
        return self.bufs[-1]

    def tmp(self, numel, dt=F32):
        return self.buf("", numel, dt)

    def range(self, extent, reduce=False):
        self._axis += 1
        if extent == 1:
            return const(0)
        return E("RANGE", "int32", (const(extent),), (self._axis - 1, 5 if reduce else 3), extent)

    def ranges(self, *extents):
        self._axis = 0
        return [self.range(e) for e in extents]

    def rrange(self, extent):
        return self.range(extent, True)

    def reduce(self, op, value, *over):
        over = [r for r in over if r.op == "RANGE"]
        return E("REDUCE", value.dt, (value,) + tuple(over), _OPS[op]) if over else value

    def store(self, out, index, value, *ranges):
        nodes, params, seen = [], [out], {}

        def add(op, dt, src, arg, ptr=0, vcount=1, size=0):
            kinds = dict(PARAM="i", CONST="c", RANGE="r", REDUCE="i")
            b = struct.pack("<HBBHHqiH", _REDUCE if op == "REDUCE" else _OPS[op], _DT[dt], ptr, 1, vcount, size, 0, len(src))
            b += b"".join(struct.pack("<I", s) for s in src)
            k = kinds.get(op)
            if k == "i":
                b += struct.pack("<Bq", 1, arg)
            elif k == "c":
                b += struct.pack("<Bq", 1, arg) if dt == "int32" else struct.pack("<BB", 3, arg) if dt == "bool" else struct.pack("<Bd", 2, arg)
            elif k == "r":
                b += struct.pack("<BqII", 9, arg[0], arg[1], 0)
            else:
                b += b"\0"
            if b not in seen:
                seen[b] = len(nodes)
                nodes.append(b)
            return seen[b]

        memo = {}

        def emit(e):
            if id(e) in memo:
                return memo[id(e)][0]
            src = [emit(s) for s in e.src]
            if e.op == "PARAM":
                if e.arg not in params:
                    params.append(e.arg)
                n = add("PARAM", e.dt, src, params.index(e.arg), ptr=1, size=e.arg.numel)
            elif e.op == "INDEX":
                n = add("INDEX", e.dt, src, None, ptr=1, size=1)
            else:
                n = add(e.op, e.dt, src, e.arg, vcount=1 if e.op == "LOAD" else 0)
            memo[id(e)] = (n, e)
            return n

        to = add("INDEX", out.dt, [add("PARAM", out.dt, [], 0, ptr=1, size=out.numel), emit(const(index))], None, ptr=1, size=out.numel)
        assert value.dt == out.dt, (value.dt, out.dt)
        n = add("STORE", "void", [to, emit(value)], None, vcount=0)
        for r in ranges:
            if r.op == "RANGE":
                n = add("END", "void", [n, emit(r)], None, vcount=0)
        add("SINK", "void", [n], None, vcount=0)
        self.items.append(struct.pack("<I", len(params)) + b"".join(struct.pack("<i", p.index) for p in params) + struct.pack("<II", 0, len(nodes)) + b"".join(nodes))
        return out

    def plan(self):
        head = b"POLYPLN1" + struct.pack("<IIII", len(self.bufs), len(self.items), 0, 0)
        ext = 0
        for b in self.bufs:
            name = b.name.encode()
            head += struct.pack("<BBiqqH", _DT[b.dt], 0 if name else 1, ext if name else -1, b.numel, b.numel * _SIZE[b.dt], len(name)) + name
            ext += 1 if name else 0
        data = head + b"".join(self.items) + struct.pack(f"<{len(self.items)}I", *range(len(self.items)))
        fd, path = tempfile.mkstemp(suffix=".polyplan")
        try:
            with os.fdopen(fd, "wb") as f:
                f.write(data)
            return HipPlan.from_file(path)
        finally:
            os.unlink(path)


def _gpt2_schedule(c):
    """GPT-2 forward: embedding as masked sums, pre-LayerNorm blocks, head tied to the token embedding; every
    tensor of the model builder realized (src/modelzoo/models/gpt2.c:320-526).  16-bit models reduce in fp32."""
    B, T, D, H, L, V, w = c["batch"], c["ctx"], c["d_model"], c["heads"], c["layers"], VOCAB, c["dtype"]
    hd = D // H
    s = Schedule()
    out, x, va = s.buf("output", B * T * V, w), s.buf("x", B * T), s.buf("vocab_arange", V)
    wte, pos, ar, wpe = s.buf("wte.weight", V * D, w), s.buf("positions", T), s.buf("arange", T), s.buf("wpe.weight", T * D, w)
    P = []
    for i in range(L):
        shapes = dict(ln1_w=("ln_1.weight", D), ln1_b=("ln_1.bias", D), attn_w=("attn.c_attn.weight", 3 * D * D), attn_b=("attn.c_attn.bias", 3 * D),
                      proj_w=("attn.c_proj.weight", D * D), proj_b=("attn.c_proj.bias", D), ln2_w=("ln_2.weight", D), ln2_b=("ln_2.bias", D),
                      fc_w=("mlp.c_fc.weight", 4 * D * D), fc_b=("mlp.c_fc.bias", 4 * D), fc2_w=("mlp.c_proj.weight", 4 * D * D), fc2_b=("mlp.c_proj.bias", D))
        P.append({k: s.buf(f"h.{i}.{n}", e, w) for k, (n, e) in shapes.items()})
    lnf_w, lnf_b = s.buf("ln_f.weight", D, w), s.buf("ln_f.bias", D, w)

    def btd(t, d, *e):
        """Ranges of a [B, T, d] tensor and its flat index."""
        b, q, j = s.ranges(B, T, d)
        return b, q, j, b * (T * d) + q * d + j

    def embed(dst, ids, arange, table, n, rows, cols, id_of, at, rs):
        v = s.rrange(n)
        hit = where(ids[id_of].ne(arange[v]), const(0.0, F32), const(1.0, F32))
        pick = where(hit, table[v * D + cols].cast(F32), const(0.0, F32))
        return s.store(dst, at, s.reduce("ADD", pick, v).cast(w), *rs)

    b, q, j, at = btd(T, D)
    tok = embed(s.tmp(B * T * D, w), x, va, wte, V, None, j, b * T + q, at, (b, q, j))
    q, j = s.ranges(T, D)
    pe0 = embed(s.tmp(T * D, w), pos, ar, wpe, T, None, j, q, q * D + j, (q, j))
    pe = pe0
    if B > 1:                        # (broadcast over the batch: realized before it is expanded)
        q, j = s.ranges(T, D)
        pe = s.store(s.tmp(T * D, w), q * D + j, pe0[q * D + j], q, j)
    b, q, j, at = btd(T, D)
    h = s.store(s.tmp(B * T * D, w), at, tok[at] + pe[q * D + j], b, q, j)

    def layernorm(src, gamma, beta):
        b, q = s.ranges(B, T)
        k = s.rrange(D)
        mean = s.store(s.tmp(B * T), b * T + q, s.reduce("ADD", src[b * (T * D) + q * D + k].cast(F32), k) / float(D), b, q)
        b, q = s.ranges(B, T)
        k = s.rrange(D)
        d = src[b * (T * D) + q * D + k].cast(F32) + (-mean[b * T + q])
        var = s.store(s.tmp(B * T), b * T + q, s.reduce("ADD", d * d, k) / float(D), b, q)
        b, q, j, at = btd(T, D)
        y = ((src[at].cast(F32) + (-mean[b * T + q])) * (var[b * T + q] + 1e-5).un("SQRT").un("RECIPROCAL")).cast(w)
        y = s.store(s.tmp(B * T * D, w), at, y * gamma[j] + beta[j], b, q, j)
        if w == F32:                 # (the fp32 graph copies some of what its layers read)
            b, q, j, at = btd(T, D)
            y = s.store(s.tmp(B * T * D, w), at, y[at], b, q, j)
        return y

    def linear(src, weight, bias, n_in, n_out, heads=False):
        b, q, j, at = btd(T, n_out)
        k = s.rrange(n_in)
        a = b * (H * T * hd) + (k // hd) * (T * hd) + q * hd + k % hd if heads else b * (T * n_in) + q * n_in + k
        acc = s.reduce("ADD", src[a].cast(F32) * weight[k * n_out + j].cast(F32), k).cast(w)
        return s.store(s.tmp(B * T * n_out, w), at, acc + bias[j], b, q, j)

    def add(u, v):
        b, q, j, at = btd(T, D)
        return s.store(s.tmp(B * T * D, w), at, u[at] + v[at], b, q, j)

    mask = None
    for p in P:
        ln1 = layernorm(h, p["ln1_w"], p["ln1_b"])
        qkv = linear(ln1, p["attn_w"], p["attn_b"], D, 3 * D)
        if w == F32:
            b, q, j, at = btd(T, 3 * D)
            qkv = s.store(s.tmp(B * T * 3 * D, w), at, qkv[at], b, q, j)

        def part(o):
            b, q, j, at = btd(T, D)
            return s.store(s.tmp(B * T * D, w), at, qkv[b * (T * 3 * D) + q * (3 * D) + (j + o)], b, q, j)

        Q, K = part(0), part(D)
        b, e, q, n = s.ranges(B, H, T, T)
        k = s.rrange(hd)
        prod = Q[b * (T * D) + q * D + e * hd + k].cast(F32) * K[b * (T * D) + n * D + e * hd + k].cast(F32)
        at = b * (H * T * T) + e * (T * T) + q * T + n
        sc = s.store(s.tmp(B * H * T * T, w), at, s.reduce("ADD", prod, k).cast(w), b, e, q, n)
        if mask is None:
            q, n = s.ranges(T, T)
            mask = s.store(s.tmp(T * T, w), q * T + n, where(ar[q].lt(ar[n]), const(-1e9, w), const(0.0, w)), q, n)
        b, e, q, n = s.ranges(B, H, T, T)
        at = b * (H * T * T) + e * (T * T) + q * T + n
        sc = s.store(s.tmp(B * H * T * T, w), at, sc[at] * (1.0 / math.sqrt(hd)) + mask[q * T + n], b, e, q, n)

        def row(op, value):
            b, e, q = s.ranges(B, H, T)
            n = s.rrange(T)
            r = b * (H * T) + e * T + q
            return s.store(s.tmp(B * H * T), r, s.reduce(op, value(b * (H * T * T) + e * (T * T) + q * T + n, r), n), b, e, q)

        top = row("MAX", lambda a, r: sc[a].cast(F32))
        tot = row("ADD", lambda a, r: ((sc[a].cast(F32) - top[r]) * LOG2E).un("EXP2"))
        b, e, q, n = s.ranges(B, H, T, T)
        at, r = b * (H * T * T) + e * (T * T) + q * T + n, b * (H * T) + e * T + q
        pr = s.store(s.tmp(B * H * T * T, w), at, (((sc[at].cast(F32) - top[r]) * LOG2E).un("EXP2") / tot[r]).cast(w), b, e, q, n)
        Vv = part(2 * D)
        b, e, q, j = s.ranges(B, H, T, hd)
        n = s.rrange(T)
        prod = pr[b * (H * T * T) + e * (T * T) + q * T + n].cast(F32) * Vv[b * (T * D) + n * D + e * hd + j].cast(F32)
        at = b * (H * T * hd) + e * (T * hd) + q * hd + j
        o = s.store(s.tmp(B * T * D, w), at, s.reduce("ADD", prod, n).cast(w), b, e, q, j)
        if w == F32:
            b, e, q, j = s.ranges(B, H, T, hd)
            at = b * (H * T * hd) + e * (T * hd) + q * hd + j
            o = s.store(s.tmp(B * T * D, w), at, o[at], b, e, q, j)
        h = add(h, linear(o, p["proj_w"], p["proj_b"], D, D, heads=True))
        ff = linear(layernorm(h, p["ln2_w"], p["ln2_b"]), p["fc_w"], p["fc_b"], D, 4 * D)
        b, q, j, at = btd(T, 4 * D)
        u = ff[at]
        inner = 2.0 * (0.7978845608028654 * (u + 0.044715 * (u * (u * u))))
        tanh = 2.0 * (1.0 + (inner * -LOG2E).un("EXP2")).un("RECIPROCAL") + -1.0
        if w != F32:
            tanh = 2.0 * (1.0 + (inner * -LOG2E).un("EXP2")).un("RECIPROCAL") - 1.0
        g = s.store(s.tmp(B * T * 4 * D, w), at, 0.5 * (u * (1.0 + tanh)), b, q, j)
        h = add(h, linear(g, p["fc2_w"], p["fc2_b"], 4 * D, D))
    h = layernorm(h, lnf_w, lnf_b)
    (r,) = s.ranges(B * T * V)
    k = s.rrange(D)
    acc = s.reduce("ADD", h[(r // V) * D + k].cast(F32) * wte[(r % V) * D + k].cast(F32), k).cast(w)
    s.store(out, r, acc, r)
    return s


def _mlp_schedule(c):
    """Two-layer classifier, softmax cross-entropy against one-hot labels, gradients of the reference's reverse
    mode, one SGD step written back into the parameters."""
    N, I, Hd, O, lr = c["batch"], c["d_in"], c["d_hid"], c["d_out"], 0.01
    s = Schedule()
    logits, X, W1, b1, W2, b2, loss, Y = (s.buf(n, e) for n, e in (("logits", N * O), ("X", N * I), ("W1", Hd * I), ("b1", Hd), ("W2", O * Hd),
                                                                   ("b2", O), ("loss", 1), ("Y", N * O)))
    relu = lambda u: where(const(0.0, F32).lt(u), u, const(0.0, F32))  # noqa: E731
    r, j = s.ranges(N, Hd)
    k = s.rrange(I)
    pre = s.store(s.tmp(N * Hd), r * Hd + j, s.reduce("ADD", X[r * I + k] * W1[j * I + k], k) + b1[j], r, j)
    r, j = s.ranges(N, O)
    k = s.rrange(Hd)
    lg = s.store(s.tmp(N * O), r * O + j, s.reduce("ADD", relu(pre[r * Hd + k]) * W2[j * Hd + k], k) + b2[j], r, j)

    def row(op, value):
        (r,) = s.ranges(N)
        j = s.rrange(O)
        return s.store(s.tmp(N), r, s.reduce(op, value(r, r * O + j), j), r)

    top = row("MAX", lambda r, a: lg[a])
    ex = lambda r, a, m: ((lg[a] - m[r]) * LOG2E).un("EXP2")  # noqa: E731
    tot = row("ADD", lambda r, a: ex(r, a, top))
    (r,) = s.ranges(N)
    j = s.rrange(O)
    d_tot = s.store(s.tmp(N), r, s.reduce("ADD", -(Y[r * O + j] * (-1.0 / N)), j) * LN2 * LOG2E / tot[r], r)
    r, j = s.ranges(N, O)
    at = r * O + j
    d_lg = s.store(s.tmp(N * O), at, Y[at] * (-1.0 / N) + d_tot[r] * (ex(r, at, top) * LN2) * LOG2E, r, j)
    (r,) = s.ranges(N)
    top1 = s.store(s.tmp(N), r, top[r], r)
    is_top = lambda r, a: lg[a].ne(top1[r]).ne(const(True, "bool")).cast(F32)  # noqa: E731
    cnt = row("ADD", is_top)
    (r,) = s.ranges(N)
    cnt1 = s.store(s.tmp(N), r, cnt[r], r)
    d_top = row("ADD", lambda r, a: -d_lg[a])
    r, j = s.ranges(N, O)
    at = r * O + j
    g = s.store(s.tmp(N * O), at, d_lg[at] + is_top(r, at) / cnt1[r] * d_top[r], r, j)
    r, j = s.ranges(N, Hd)
    k = s.rrange(O)
    d_h = s.reduce("ADD", g[r * O + k] * W2[k * Hd + j], k)
    d_pre = s.store(s.tmp(N * Hd), r * Hd + j, where(const(0.0, F32).lt(pre[r * Hd + j]), d_h, const(0.0, F32)), r, j)

    def update(p, grad):
        (i,) = s.ranges(p.numel)
        r = s.rrange(N)
        new = s.store(s.tmp(p.numel), i, p[i] - s.reduce("ADD", grad(i, r), r) * lr, i)
        (i,) = s.ranges(p.numel)
        s.store(p, i, new[i], i)

    update(W1, lambda i, r: d_pre[r * Hd + i // I] * X[r * I + i % I])
    update(b1, lambda i, r: d_pre[r * Hd + i])
    update(W2, lambda i, r: g[r * O + i // Hd] * relu(pre[r * Hd + i % Hd]))
    update(b2, lambda i, r: g[r * O + i])
    (i,) = s.ranges(N * O)
    s.store(logits, i, lg[i], i)
    s.ranges()
    r, j = s.rrange(N), s.rrange(O)
    at = r * O + j
    nll = ((lg[at] - top[r]) - tot[r].un("LOG2") * LN2) * Y[at]
    s.store(loss, 0, s.reduce("ADD", s.reduce("ADD", nll, j), r) * (-1.0 / N))
    return s


def _adamw_schedule(c):
    """Decoupled AdamW of a flat parameter: p through a temporary, then p, m and v in place (src/instance.c:1162-1224)."""
    n = c["numel"]
    s = Schedule()
    p, m, g, bc1, v, bc2 = s.buf("p", n), s.buf("m", n), s.buf("g", n), s.buf("bc1", 1), s.buf("v", n), s.buf("bc2", 1)
    new_m = lambda i: 0.9 * m[i] + (1.0 - 0.9) * g[i]  # noqa: E731
    new_v = lambda i: 0.999 * v[i] + (1.0 - 0.999) * (g[i] * g[i])  # noqa: E731
    (i,) = s.ranges(n)
    step = new_m(i) * bc1[0] * ((new_v(i) * bc2[0]).un("SQRT") + 1e-8).un("RECIPROCAL")
    t = s.store(s.tmp(n), i, p[i] * (1.0 - 3e-4 * 0.1) - 3e-4 * step, i)
    s.store(p, i, t[i], i)
    s.store(m, i, new_m(i), i)
    s.store(v, i, new_v(i), i)
    return s


def _rows_schedule(c):
    """y = clamp(exp2(a b + c), -4, 4), never stored, and an operation over its rows."""
    R, C, op = c["rows"], c["cols"], c["op"]
    s = Schedule()
    out = s.buf("out", R if op in ("sum", "max") else R * C)
    a, b, d = s.buf("a", R * C), s.buf("b", R * C), s.buf("c", R * C)

    def y(i):
        u = (a[i] * b[i] + d[i]).un("EXP2")
        lo = where(u.lt(-4.0), const(-4.0, F32), u)
        return where(const(4.0, F32).lt(lo), const(4.0, F32), lo)

    def row(dst, over, value):
        (r,) = s.ranges(R)
        k = s.rrange(C)
        v = s.reduce(over, value(r * C + k), k)
        return s.store(dst, r, v / float(C) if op == "layernorm" else v, r)

    if op in ("sum", "max"):
        row(out, "MAX" if op == "max" else "ADD", y)
        return s
    st = row(s.tmp(R), "MAX" if op == "softmax" else "ADD", y)
    r, k = s.ranges(R, C)
    i = r * C + k
    mid = s.store(s.tmp(R * C), i, ((y(i) - st[r]) * LOG2E).un("EXP2") if op == "softmax" else y(i) + (-st[r]), r, k)
    sm = row(s.tmp(R), "ADD", lambda i: mid[i] if op == "softmax" else mid[i] * mid[i])
    (i,) = s.ranges(R * C)
    v = mid[i] / sm[i // C] if op == "softmax" else mid[i] * (sm[i // C] + 1e-5).un("SQRT").un("RECIPROCAL")
    s.store(out, i, v, i)
    return s


def _matmul_schedule(c):
    M, N, K, dt = c["m"], c["n"], c["k"], c["dtype"]
    s = Schedule()
    C, A, B = s.buf("C", M * N), s.buf("A", M * K, dt), s.buf("B", K * N, dt)
    (r,) = s.ranges(M * N)
    k = s.rrange(K)
    m, n = r // N, r % N
    a = k * M + m if c["layout"][0] == "t" else m * K + k
    b = n * K + k if c["layout"][1] == "t" else k * N + n
    s.store(C, r, s.reduce("ADD", A[a].cast(F32) * B[b].cast(F32), k), r)
    return s


_SCHEDULES = dict(gpt2=_gpt2_schedule, mlp=_mlp_schedule, adamw=_adamw_schedule, rows=_rows_schedule, matmul=_matmul_schedule)


# ── inputs ───────────────────────────────────────────────────────────────────

def _fill(case, name, n, dt, g):
    """The contents of buffer `name`, on the device."""
    normal = lambda scale: (torch.randn(n, generator=g, device="cuda") * scale).to(dt)  # noqa: E731
    kind = case["kind"]
    if name in ("positions", "arange", "vocab_arange") or name.startswith("__arange_"):
        return torch.arange(n, device="cuda").to(dt)
    if name in ("x", "target"):                       # token and class ids, which the reference keeps as floats
        return torch.randint(0, VOCAB, (n,), generator=g, device="cuda").to(dt)
    if name in ("output", "logits", "loss", "out", "C"):
        return torch.zeros(n, dtype=dt, device="cuda")
    if kind in ("gpt2", "train"):
        if name == "h0":
            return normal(1.0)
        if name in ("bc1", "bc2"):                    # bias corrections after a thousand steps
            return torch.full((n,), 1.0 / (1.0 - (0.9 if name == "bc1" else 0.999) ** 1000), device="cuda")
        if name.endswith(".m"):                       # moments of a run under way
            return normal(1e-4)
        if name.endswith(".v"):
            return normal(1e-4) ** 2 + 1e-10
        leaf = name.split(".")[-2] if kind == "gpt2" and "." in name else name.split(".")[-1]
        if leaf.startswith("ln") and (name.endswith(".weight") or name.endswith("_w")):
            return (1.0 + torch.randn(n, generator=g, device="cuda") * 0.1).to(dt)
        return normal(0.02)
    if kind == "mlp":
        if name == "Y":
            labels = torch.randint(0, case["d_out"], (case["batch"],), generator=g, device="cuda")
            return torch.nn.functional.one_hot(labels, case["d_out"]).to(dt).reshape(-1)
        if name == "X":
            return torch.rand(n, generator=g, device="cuda")
        return normal(dict(W1=case["d_in"], W2=case["d_hid"]).get(name, 10000) ** -0.5)
    if kind == "adamw":
        if name in ("bc1", "bc2"):
            return torch.full((n,), 1.0 / (1.0 - (0.9 if name == "bc1" else 0.999) ** 1000), device="cuda")
        return normal(1e-3) ** 2 + 1e-10 if name == "v" else normal(dict(p=0.02).get(name, 1e-3))
    if kind == "rows":
        return torch.rand(n, generator=g, device="cuda") * 2 - 1
    return normal(1.0)


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    if case["kind"] == "train":
        plan = HipPlan.from_file(os.path.join(PLANS, "gpt2_medium_block_train_b4_t1024.polyplan"))
    else:
        plan = _SCHEDULES[case["kind"]](case).plan()
    data, by_name = [None] * len(plan.slots), {}
    for slot in plan.external_slots():
        data[slot.index] = by_name[slot.name] = _fill(case, slot.name, slot.numel, torch_dtype(slot.dtype), g)
    names = dict(gpt2=["output"], mlp=["logits", "loss", "W1", "b1", "W2", "b2"], adamw=["p", "m", "v"], rows=["out"], matmul=["C"]).get(case["kind"])
    if names is None:                                 # every parameter and both its moments, and the loss
        names = ["loss"] + [n for n in by_name if n.endswith((".m", ".v")) or n + ".m" in by_name]
    return dict(plan=plan, data=data, out={n: by_name[n] for n in names})


def run(state):
    state["plan"].run(state["data"], sync=False)
    return state["out"]


# ── what a pass cannot do without ────────────────────────────────────────────

def work(case):
    kind = case["kind"]
    if kind == "gpt2":
        B, T, D, L, e = case["batch"], case["ctx"], case["d_model"], case["layers"], _SIZE[case["dtype"]]
        tokens, block = B * T, 12 * D * D + 13 * D
        # (token ids; the embedding rows are rows of the head's weights; a causal score and its value count half)
        flops = 2.0 * tokens * (L * 12 * D * D + VOCAB * D) + L * 2.0 * tokens * (T + 1) * D
        return dict(bytes=e * (VOCAB * D + T * D + L * block + 2 * D + tokens * VOCAB) + 4 * tokens, flops=flops)
    if kind == "train":
        B, T, D = 4, 1024, 1024
        params = 12 * D * D + 13 * D + 2 * D + VOCAB * D
        # forward once, backward twice (not towards the block's input)
        flops = 6.0 * B * T * (12 * D * D + VOCAB * D) - 2.0 * B * T * 3 * D * D + 3 * 2.0 * B * T * (T + 1) * D
        return dict(bytes=4.0 * params * 6 + 2 * B * T * D + 4 * B * T, flops=flops)
    if kind == "mlp":
        N, I, H, O = case["batch"], case["d_in"], case["d_hid"], case["d_out"]
        return dict(bytes=4.0 * (N * I + 2 * N * O + 2 * (H * I + H + O * H + O) + 1), flops=4.0 * N * I * H + 6.0 * N * H * O)
    if kind == "adamw":
        return dict(bytes=4.0 * 7 * case["numel"] + 8, flops=0)
    if kind == "rows":
        n = case["rows"] * case["cols"]
        return dict(bytes=4.0 * (3 * n + (case["rows"] if case["op"] in ("sum", "max") else n)), flops=0)
    M, N, K = case["m"], case["n"], case["k"]
    return dict(bytes=_SIZE[case["dtype"]] * (M * K + K * N) + 4.0 * M * N, flops=2.0 * M * N * K)


def tolerance(case):
    """About four times the largest difference seen between a path and itself in other orders of summation (other
    tiles, K splits, the two-pass attention, unfused kernels), and for the fp32 paths between it and float64."""
    kind = case["kind"]
    if kind == "gpt2" and case["dtype"] != F32:
        return {"rel": 4e-2, "max": 0.3}              # seen: 1.2e-2 and 0.084, a rounding to 16 bits after every operation
    if kind == "train":
        return {"rel": 4e-2, "max": 0.5}              # seen: 1.1e-2 and 0.13, first moments of the smallest gradients
    return {"rel": dict(gpt2=1e-5, mlp=4e-6, adamw=4e-7, rows=2e-6, matmul=4e-6)[kind]}
