"""The work a user of sa3k has it do, as cases that can be prepared, run, priced and checked.

Six kinds of call, each through the Python binding of the C ABI:

  dit    the DiT LoRA/DoRA training update (accumulate: forward, velocity MSE, backward; then average,
         clip and AdamW), or the forward alone (the velocity)
  block  one DiT block: adapter refresh, forward and backward
  lin    one adapted linear (lora or dora-rows): adapter refresh, forward and backward
  chain  inference: the forward of a composed adapter chain over a frozen base
  attn   differential attention, forward and backward (self, windowed or dense; cross)
  adamw  average, global clip and AdamW over a flat arena

Sizes: the model of the benchmark (24 blocks x 1536, 24 heads of 64, FFN 6144, 64 memory + up to
1024 latent tokens, 128 conditioning tokens, rank 32), its linears, and the ranges around them.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HP = (1e-4, 0.9, 0.999, 1e-8, 0.01, 1.0)   # lr, beta1, beta2, eps, weight decay, clip


def _binding():
    if "sa3k" not in sys.modules:
        spec = importlib.util.spec_from_file_location("sa3k", os.path.join(ROOT, "sa3.cpp_amd", "sa3k.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules["sa3k"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["sa3k"]


_CTX = []


def _ctx():
    """the program's one context"""
    if not _CTX:
        torch.cuda.init()
        _CTX.append(_binding().Context(0))
    return _CTX[0]


# ------------------------------------------------------------------------------------------ cases
def listed():
    return [
        # one optimizer update of the benchmark's model: 24 blocks, batch 2 x 1024 frames, window 256,
        # dora-rows r32 on all 180 targets over an f16 base
        dict(name="dit_update_b2_t1024", kind="dit", mode="update", depth=24, heads=24, inner=6144, batch=2, frames=1024,
             ctx=128, window=256, rank=32, dora=True, local=0, recompute=False),
        # the reference's per-sample call on a shorter clip, inpaint model, dense attention, lora r16:
        # the forward that previews and validates while training
        dict(name="dit_velocity_inpaint_b1_t215", kind="dit", mode="velocity", depth=8, heads=24, inner=6144, batch=1,
             frames=215, ctx=128, window=0, rank=16, dora=False, local=257, recompute=False),
        # one block of the benchmark's model, trained
        dict(name="block_dora_b2_s1088_w256", kind="block", heads=24, inner=6144, batch=2, seq=1088, ctx=128, window=256,
             rank=32, dora=True, base="f16"),
        # one block at the reference's per-sample call: dense attention, an odd length, lora r16
        dict(name="block_lora_b1_s343_dense", kind="block", heads=24, inner=6144, batch=1, seq=343, ctx=77, window=0,
             rank=16, dora=False, base="f16"),
        # the FFN linear over a quantised base, trained
        dict(name="lin_dora_q8_0_2048x1536x6144", kind="lin", tokens=2048, inp=1536, out=6144, rank=32, dora=True,
             base="q8_0", prec="bf16"),
        # an out-projection trained in full f32
        dict(name="lin_lora_f32_2048x1536x1536", kind="lin", tokens=2048, inp=1536, out=1536, rank=16, dora=False,
             base="f32", prec="f32"),
        # the modulation linear: one row per sample, so launches and latency count
        dict(name="lin_lora_f16_2x1536x9216", kind="lin", tokens=2, inp=1536, out=9216, rank=16, dora=False, base="f16",
             prec="bf16"),
        # inference over a quantised base with three composed adapters, a whole clip of two samples
        dict(name="chain_q8_0_2176x1536x6144", kind="chain", tokens=2176, inp=1536, out=6144, adapters=3, rank=16,
             base="q8_0"),
        # inference of the conditioning tokens' linear with one adapter: a small call
        dict(name="chain_f16_77x768x1536", kind="chain", tokens=77, inp=768, out=1536, adapters=1, rank=16, base="f16"),
        # windowed self-attention at the benchmark's size, forward and backward
        dict(name="attn_b2_s1088_w256", kind="attn", batch=2, heads=24, sq=1088, sk=1088, window=256),
        # the reference's dense self-attention of one odd-length sample
        dict(name="attn_b1_s607_dense", kind="attn", batch=1, heads=24, sq=607, sk=607, window=0),
        # clip and AdamW over the adapters of the benchmark's model
        dict(name="adamw_38m", kind="adamw", n=38417600, count=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["dit", "block", "lin", "chain", "attn", "adamw"], [1, 3, 4, 3, 3, 1])[0]
    heads = rng.choice([4, 8, 12, 16, 24])
    rank = rng.choice([8, 16, 24, 32])
    window = rng.choice([0, 0, 64, 256])
    dora = rng.random() < 0.6
    if kind == "dit":
        return dict(kind=kind, mode=rng.choice(["update", "update", "velocity"]), depth=rng.randint(1, 4), heads=heads,
                    inner=256 * heads, batch=rng.randint(1, 3), frames=_log(rng, 32, 1024), ctx=rng.choice([64, 77, 128]),
                    window=window, rank=rank, dora=dora, local=rng.choice([0, 0, 257]), recompute=rng.random() < 0.3)
    if kind == "block":
        return dict(kind=kind, heads=heads, inner=256 * heads, batch=rng.randint(1, 3), seq=_log(rng, 48, 1088),
                    ctx=rng.choice([32, 77, 128]), window=window, rank=rank, dora=dora,
                    base=rng.choice(["f16", "f16", "f32", "bf16"]))
    if kind == "lin":
        base = rng.choice(["f16", "f16", "f32", "bf16", "q8_0"])
        prec = rng.choice(["bf16", "f32"]) if base in ("f16", "f32") else "bf16"
        return dict(kind=kind, tokens=_log(rng, 1, 4096), inp=64 * _log(rng, 1, 96), out=64 * _log(rng, 1, 144), rank=rank,
                    dora=dora, base=base, prec=prec)
    if kind == "chain":
        return dict(kind=kind, tokens=_log(rng, 1, 4096), inp=64 * _log(rng, 4, 96), out=64 * _log(rng, 4, 144),
                    adapters=rng.randint(1, 4), rank=rank, base=rng.choice(["q8_0", "f16", "bf16"]))
    if kind == "attn":
        sq = _log(rng, 32, 2048)
        cross = rng.random() < 0.4
        return dict(kind=kind, batch=rng.randint(1, 3), heads=heads, sq=sq, sk=_log(rng, 16, 256) if cross else sq,
                    window=0 if cross else window)
    return dict(kind=kind, n=_log(rng, 10_000, 40_000_000), count=rng.choice([1, 2, 4]))


# ---------------------------------------------------------------------------------- inputs, weights
class _Draw:
    """seeded tensors on the GPU, in the order they are asked for"""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, shape, sd=1.0, mean=0.0):
        t = torch.empty(shape, device="cuda", dtype=torch.float32)
        return t.normal_(mean, sd, generator=self.g)

    def uniform(self, shape, lo, hi):
        t = torch.empty(shape, device="cuda", dtype=torch.float32)
        return t.uniform_(lo, hi, generator=self.g)

    def adapter(self, inp, out, rank, norms, b_sd=0.01):
        """A Kaiming-uniform, B part-trained, magnitudes near the base's row norms (norms None: lora)"""
        A = self.uniform((rank, inp), -1 / math.sqrt(inp), 1 / math.sqrt(inp))
        B = self.normal((out, rank), b_sd)
        m = (norms * self.normal((out,), 0.05, 1.0)).float() if norms is not None else None
        return A, B, m


def _q8_0(W):
    """(blocks uint8 [out][in/32][34], the weight they decode to): 32-element blocks of an f16 scale and int8s"""
    out, inp = W.shape
    w = W.reshape(out, inp // 32, 32)
    scale = (w.abs().amax(2) / 127.0).half()
    s = scale.float()[:, :, None]
    q = torch.where(s > 0, torch.round(w / torch.where(s > 0, s, torch.ones_like(s))), torch.zeros_like(w)).clamp(-127, 127)
    blocks = torch.cat([scale.contiguous().view(torch.uint8).reshape(out, inp // 32, 2), q.to(torch.int8).view(torch.uint8)], 2)
    return blocks.contiguous(), (s * q).reshape(out, inp)


def _base(d, inp, out, base):
    """(what the loader takes, the decoded weight) of a frozen base ~ N(0, 0.02)"""
    W = d.normal((out, inp), 0.02)
    if base == "q8_0":
        return _q8_0(W)
    t = W.to({"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[base])
    return t, t.float()


def _type(base):
    s = _binding()
    return {"f32": s.TYPE_F32, "f16": s.TYPE_F16, "bf16": s.TYPE_BF16, "q8_0": s.TYPE_Q8_0}[base]


def _host(t):
    """a base weight as the loader's host array"""
    return (t.view(torch.int16) if t.dtype == torch.bfloat16 else t).cpu().numpy()


def _norms(W):
    return W.double().square().sum(1).sqrt()


def _dev(t):
    """a device tensor as the binding's array (the tensor keeps its memory)"""
    kind = {torch.float32: np.float32, torch.bfloat16: np.uint16, torch.float16: np.float16, torch.uint8: np.uint8}[t.dtype]
    return _binding().DeviceArray(_ctx(), t.data_ptr(), t.shape, kind, owner=False)


class _Handles:
    """library objects, given back the last made first once nothing refers to them or their memory"""

    def __init__(self):
        self.made = []

    def __del__(self):
        try:
            torch.cuda.synchronize()
            while self.made:
                self.made.pop().destroy()
        except Exception:
            pass


class _Raw:
    """device memory of the library, for torch to look at: it lives as long as the tensors over it"""

    def __init__(self, a, handles):
        self.handles = handles
        self.__cuda_array_interface__ = dict(shape=a.shape, typestr="<f4", data=(a.ptr, False), version=2, strides=None)


class _State:
    """what a program keeps between calls"""

    def __init__(self, case):
        self.case, self.handles = case, _Handles()

    def keep(self, h):
        self.handles.made.append(h)
        return h

    def see(self, a):
        return torch.as_tensor(_Raw(a, self.handles), device="cuda")


def _arena(state, shapes):
    """one zeroed f32 arena cut into tensors of the shapes: a user clears its gradients in one call"""
    sizes = [math.prod(s) for s in shapes]
    state.flat = torch.zeros(sum(-(-n // 64) * 64 for n in sizes), device="cuda")
    out, at = [], 0
    for s, n in zip(shapes, sizes):
        out.append(state.flat[at:at + n].view(s))
        at += -(-n // 64) * 64
    return out


def _clear(state):
    c = _ctx()
    c.check(c.lib.sa3k_memset(c.h, state.flat.data_ptr(), 0, state.flat.numel() * 4))


# ------------------------------------------------------------------------------------------ linears
def _lin_inputs(case, seed):
    d = _Draw(seed)
    stored, W = _base(d, case["inp"], case["out"], case["base"])
    A, B, m = d.adapter(case["inp"], case["out"], case["rank"], _norms(W) if case["dora"] else None)
    X = d.normal((case["tokens"], case["inp"]))
    dY = d.normal((case["tokens"], case["out"]), 1e-2)
    return stored, W, A, B, m, X, dY


def _prepare_lin(case, seed):
    c, k, s = _ctx(), _binding(), _State(case)
    stored, W, s.A, s.B, s.m, s.X, s.dY = _lin_inputs(case, seed)
    h = _host(stored)
    s.w = s.keep(c.weight((h, case["inp"], case["out"]) if case["base"] == "q8_0" else h, _type(case["base"])))
    s.lin = s.keep(c.lin(s.w, case["rank"], k.PREC_F32 if case["prec"] == "f32" else k.PREC_BF16, case["tokens"]))
    s.bnsq = s.w.row_norm_sq() if case["dora"] else None
    n, i, o, r = case["tokens"], case["inp"], case["out"], case["rank"]
    s.Y, s.dX = torch.empty((n, o), device="cuda"), torch.empty((n, i), device="cuda")
    s.dA, s.dB, s.dm = _arena(s, [(r, i), (o, r), (o,) if case["dora"] else (0,)])
    return s


def _run_lin(s):
    c = s.case
    n = c["tokens"]
    s.lin.prepare(_dev(s.A), _dev(s.B), 1.0, c["dora"], _dev(s.m) if c["dora"] else None, s.bnsq)
    _clear(s)
    s.lin.forward(_dev(s.X), n, _dev(s.Y))
    s.lin.backward(_dev(s.X), n, _dev(s.dY), _dev(s.dX), _dev(s.dA), _dev(s.dB), _dev(s.dm) if c["dora"] else None)
    return [s.Y, s.dX, s.dA, s.dB] + ([s.dm] if c["dora"] else [])


def _lin64(X, W, A, B, m, scale, bias=None):
    """the adapted linear in 64 bits: (X W^T + s (X A^T) B^T) (.) m / |W + s B A|, + bias"""
    y = X @ W.t() + scale * ((X @ A.t()) @ B.t())
    if m is not None:
        We = W + scale * (B @ A)
        y = y * (m / torch.sqrt(We.square().sum(1) + W.shape[1] * 1e-12))
    return y if bias is None else y + bias


def _leaf(t):
    return t.double().requires_grad_() if t is not None else None


def _exact_lin(case, seed):
    _, W, A, B, m, X, dY = _lin_inputs(case, seed)
    X, A, B, m = _leaf(X), _leaf(A), _leaf(B), _leaf(m)
    Y = _lin64(X, W.double(), A, B, m, 1.0)
    Y.backward(dY.double())
    return [Y.detach(), X.grad, A.grad, B.grad] + ([m.grad] if m is not None else [])


def _lin_work(n, i, o, r, dora):
    """flops of forward and backward of an adapted linear over n tokens (no gradient of the frozen base)"""
    extra = 2.0 * r * i * o if dora else 0.0
    return 2 * (2.0 * n * i * o) + 3 * (2.0 * n * r * i) + 3 * (2.0 * n * r * o) + 2 * extra


_STORED = {"f32": 4.0, "f16": 2.0, "bf16": 2.0, "q8_0": 34 / 32}


# ------------------------------------------------------------------------------------------- chains
def _chain_inputs(case, seed):
    d = _Draw(seed)
    stored, W = _base(d, case["inp"], case["out"], case["base"])
    ads = []
    for k in range(case["adapters"]):   # dora and lora in turn, as a user stacks them, at falling strengths
        dora = k % 2 == 0
        A, B, m = d.adapter(case["inp"], case["out"], case["rank"], _norms(W) if dora else None, 0.02)
        ads.append((dora, case["rank"], float(case["rank"]), (1.0, 0.7, 0.5, 0.3)[k], A, B, m))
    return stored, W, ads, d.normal((case["tokens"], case["inp"])), d.normal((case["out"],), 0.02)


def _prepare_chain(case, seed):
    c, s = _ctx(), _State(case)
    stored, _, ads, s.X, s.bias = _chain_inputs(case, seed)
    h = _host(stored)
    torch.cuda.synchronize()
    s.w = s.keep(c.weight((h, case["inp"], case["out"]) if case["base"] == "q8_0" else h, _type(case["base"])))
    if case["base"] == "q8_0":
        s.w.drop_working_copy()   # what a user keeps a quantised base for: its size
    s.chain = s.keep(c.lora_chain(s.w, [(a, r, al, st, _dev(A), _dev(B), _dev(m) if m is not None else None)
                                        for a, r, al, st, A, B, m in ads], case["tokens"]))
    c.sync()   # the adapters are read by the fold only
    s.Y = torch.empty((case["tokens"], case["out"]), device="cuda")
    return s


def _run_chain(s):
    s.chain.forward(_dev(s.X), s.case["tokens"], _dev(s.Y), _dev(s.bias))
    return s.Y


def _exact_chain(case, seed):
    _, W, ads, X, bias = _chain_inputs(case, seed)
    W = W.double()
    for dora, r, alpha, strength, A, B, m in ads:   # merged one after another
        W = W + (alpha / r * strength) * (B.double() @ A.double())
        if dora:
            W = W * (m.double() / torch.sqrt(W.square().sum(1)))[:, None]
    return X.double() @ W.t() + bias.double()


# ---------------------------------------------------------------------------------------- attention
def _attn_inputs(case, seed):
    d = _Draw(seed)
    bh = case["batch"] * case["heads"]

    def rows(n):   # the per-head RMS-normed queries and keys
        x = d.normal((bh, n, 64))
        return (x / x.square().mean(2, keepdim=True).sqrt()).bfloat16()

    q1, q2, k1, k2 = rows(case["sq"]), rows(case["sq"]), rows(case["sk"]), rows(case["sk"])
    v = d.normal((bh, case["sk"], 64)).bfloat16()
    return q1, k1, q2, k2, v, d.normal((case["batch"], case["sq"], case["heads"] * 64), 1e-2)


def _prepare_attn(case, seed):
    s = _State(case)
    s.q1, s.k1, s.q2, s.k2, s.v, s.dO = _attn_inputs(case, seed)
    b, h, sq, sk = case["batch"], case["heads"], case["sq"], case["sk"]
    half = lambda *n: torch.empty(n, device="cuda", dtype=torch.bfloat16)   # noqa: E731
    full = lambda *n: torch.empty(n, device="cuda")   # noqa: E731
    s.o, s.o1, s.o2, s.doh = half(b, sq, h * 64), half(b * h, sq, 64), half(b * h, sq, 64), half(b * h, sq, 64)
    s.l1, s.l2, s.dn = full(b * h, sq), full(b * h, sq), full(2, b * h, sq)
    s.g = [full(b * h, n, 64) for n in (sq, sk, sq, sk, sk)]
    return s


def _run_attn(s):
    c, a = _ctx(), s.case
    p = lambda *ts: [t.data_ptr() for t in ts]   # noqa: E731
    shape = (a["batch"], a["heads"], a["sq"], a["sk"], 64, a["window"], 0.125)
    c.check(c.lib.sa3k_diff_attn_fwd(c.h, *p(s.q1, s.k1, s.q2, s.k2, s.v), *shape, *p(s.o, s.o1, s.o2, s.l1, s.l2)))
    c.check(c.lib.sa3k_diff_attn_bwd(c.h, *p(s.q1, s.k1, s.q2, s.k2, s.v, s.o1, s.o2, s.l1, s.l2, s.dO), *shape,
                                     *p(s.doh, s.dn, *s.g)))
    return [s.o, s.o1, s.o2, s.l1, s.l2] + s.g


def _branch64(q, k, v, window):
    s = (q @ k.transpose(-1, -2)) * 0.125
    if window > 0:
        i = torch.arange(q.shape[-2], device=q.device)
        s = s.masked_fill(2 * (i[:, None] - i[None, :]).abs() > window, float("-inf"))
    return torch.softmax(s, -1) @ v, torch.logsumexp(s, -1)


def _exact_attn(case, seed):
    q1, k1, q2, k2, v, dO = _attn_inputs(case, seed)
    q1, k1, q2, k2, v = (_leaf(t) for t in (q1, k1, q2, k2, v))
    b, h, sq = case["batch"], case["heads"], case["sq"]
    (o1, l1), (o2, l2) = _branch64(q1, k1, v, case["window"]), _branch64(q2, k2, v, case["window"])
    o = (o1 - o2).reshape(b, h, sq, 64).transpose(1, 2).reshape(b, sq, h * 64)
    o.backward(dO.double())
    log2e = 1 / math.log(2.0)
    return [t.detach() for t in (o, o1, o2, l1 * log2e, l2 * log2e)] + [t.grad for t in (q1, k1, q2, k2, v)]


def _pairs(s, window):
    if window <= 0:
        return float(s) * s
    h = window // 2
    return float(sum(min(q + h, s - 1) - max(q - h, 0) + 1 for q in range(s)))


# ------------------------------------------------------------------------------------------- blocks
def _targets(dim, inner):
    return [(dim, 5 * dim), (dim, dim), (dim, 2 * dim), (dim, 3 * dim), (dim, dim), (dim, 2 * inner), (inner, dim)]


_VECS = dict(ssg=None, pre_g="pre_norm.gamma", cross_g="cross_norm.gamma", ff_g="ff_norm.gamma",
             sq_g="self.q_norm.gamma", sk_g="self.k_norm.gamma", cq_g="cross.q_norm.gamma", ck_g="cross.k_norm.gamma")


def _block_vecs(d, dim):
    v = {"ssg": d.normal((6 * dim,), 0.1)}
    for n in ("pre_g", "cross_g", "ff_g"):
        v[n] = d.normal((dim,), 0.1, 1.0)
    for n in ("sq_g", "sk_g", "cq_g", "ck_g"):
        v[n] = d.normal((64,), 0.1, 1.0)
    return v


def _block_inputs(case, seed):
    d = _Draw(seed)
    dim, inner = 64 * case["heads"], case["inner"]
    tg = _targets(dim, inner)
    bases = [_base(d, i, o, case["base"]) for i, o in tg]
    bias = [None] * 5 + [d.normal((2 * inner,), 0.02), d.normal((dim,), 0.02)]
    vecs = _block_vecs(d, dim)
    ads = [d.adapter(i, o, case["rank"], _norms(W) if case["dora"] else None) for (i, o), (_, W) in zip(tg, bases)]
    b, n = case["batch"], case["seq"]
    x, cx, gc = d.normal((b, n, dim)), d.normal((b, case["ctx"], dim)), d.normal((b, 6 * dim), 0.1)
    return bases, bias, vecs, ads, x, cx, gc, d.normal((b, n, dim), 1e-2)


def _prepare_block(case, seed):
    c, k, s = _ctx(), _binding(), _State(case)
    bases, bias, vecs, s.ads, s.x, s.cx, s.gc, s.dout = _block_inputs(case, seed)
    dim, b, n, r = 64 * case["heads"], case["batch"], case["seq"], case["rank"]
    cfg = k.BlockConfig(dim, case["heads"], 64, case["inner"], 32, case["window"], 1e4, 1e-5, 1e-6)
    s.blk = s.keep(k.Block(c, cfg, [_host(t) for t, _ in bases], [None if t is None else t.cpu().numpy() for t in bias],
                           {m: t.cpu().numpy() for m, t in vecs.items()}, r, b * n, b * case["ctx"], _type(case["base"])))
    s.ws = s.keep(k.BlockWorkspace(c, cfg, b, n, case["ctx"]))
    s.out, s.dx = torch.empty_like(s.x), torch.empty_like(s.x)
    tg = _targets(dim, case["inner"])
    got = _arena(s, [s.cx.shape, s.gc.shape] + [(r, i) for i, _ in tg] + [(o, r) for _, o in tg] +
                 ([(o,) for _, o in tg] if case["dora"] else []))
    s.dcx, s.dgc, s.dA, s.dB, s.dm = got[0], got[1], got[2:9], got[9:16], got[16:]
    return s


def _run_block(s):
    each = lambda ts: [_dev(t) for t in ts]   # noqa: E731
    dora = s.case["dora"]
    s.blk.prepare(each(a[0] for a in s.ads), each(a[1] for a in s.ads), 1.0, dora, each(a[2] for a in s.ads) if dora else None)
    _clear(s)
    s.blk.forward(s.ws, _dev(s.x), _dev(s.cx), _dev(s.gc), _dev(s.out))
    s.blk.backward(s.ws, _dev(s.dout), _dev(s.dx), _dev(s.dcx), _dev(s.dgc), each(s.dA), each(s.dB), each(s.dm) if dora else None)
    return [s.out, s.dx, s.dcx, s.dgc, s.dA, s.dB] + ([s.dm] if dora else [])


def _rms64(x, g, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * g


def _rope64(x):
    """NeoX rotation of the first 32 dims of each head, position = row"""
    th = torch.arange(x.shape[-2], device=x.device, dtype=torch.float64)[:, None] * \
        1e4 ** (-2.0 * torch.arange(16, device=x.device, dtype=torch.float64) / 32)
    c, s, a, b = torch.cos(th), torch.sin(th), x[..., :16], x[..., 16:32]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., 32:]], -1)


def _block64(W, bias, v, ads, scale, x, cx, gc, window, add=None):
    """the block in 64 bits: W, bias by target; v the block's vectors; ads (A, B, m) by target"""
    B, S, dim = x.shape
    lin = lambda t, h: _lin64(h, W[t], *ads[t], scale, bias[t])   # noqa: E731
    heads = lambda h: h.reshape(B, h.shape[1], -1, 64).transpose(1, 2)   # noqa: E731
    sc_a, sh_a, g_a, sc_f, sh_f, g_f = [m[:, None, :] for m in (v["ssg"] + gc).split(dim, 1)]

    def attend(q, k, vv, qd, kd, win):
        o = _branch64(q, k, vv, win)[0] - _branch64(qd, kd, vv, win)[0]
        return o.transpose(1, 2).reshape(B, S, dim)

    h = _rms64(x, v["pre_g"], 1e-5) * (1 + sc_a) + sh_a
    q, k, vv, qd, kd = [heads(p) for p in lin(0, h).split(dim, 2)]
    nq, nk = (lambda t: _rope64(_rms64(t, v["sq_g"], 1e-6))), (lambda t: _rope64(_rms64(t, v["sk_g"], 1e-6)))
    x = x + lin(1, attend(nq(q), nk(k), vv, nq(qd), nk(kd), window)) * torch.sigmoid(1 - g_a)
    q, qd = [_rms64(heads(p), v["cq_g"], 1e-6) for p in lin(2, _rms64(x, v["cross_g"], 1e-5)).split(dim, 2)]
    k, kd, vv = [heads(p) for p in lin(3, cx).split(dim, 2)]
    k, kd = _rms64(k, v["ck_g"], 1e-6), _rms64(kd, v["ck_g"], 1e-6)
    x = x + lin(4, attend(q, k, vv, qd, kd, 0))
    if add is not None:
        x = x + add
    f = _rms64(x, v["ff_g"], 1e-5) * (1 + sc_f) + sh_f
    val, glu = lin(5, f).chunk(2, 2)
    return x + lin(6, val * torch.nn.functional.silu(glu)) * torch.sigmoid(1 - g_f)


def _exact_block(case, seed):
    bases, bias, vecs, ads, x, cx, gc, dout = _block_inputs(case, seed)
    W = [w.double() for _, w in bases]
    ads = [[_leaf(t) for t in a] for a in ads]
    x, cx, gc = _leaf(x), _leaf(cx), _leaf(gc)
    out = _block64(W, [None if t is None else t.double() for t in bias], {n: t.double() for n, t in vecs.items()}, ads, 1.0,
                   x, cx, gc, case["window"])
    out.backward(dout.double())
    return [out.detach(), x.grad, cx.grad, gc.grad] + [[a[j].grad for a in ads] for j in range(3 if case["dora"] else 2)]


def _block_work(b, s, ctx, heads, inner, r, window, dora):
    dim = 64 * heads
    fl = sum(_lin_work(b * (ctx if t == 3 else s), i, o, r, dora) for t, (i, o) in enumerate(_targets(dim, inner)))
    return fl + 3 * b * heads * (_pairs(s, window) + s * ctx) * 512


# --------------------------------------------------------------------------------------- the model
_IO, _COND, _TIME, _MEM = 64, 768, 256, 64
_BLOCK = ("self.qkv", "self.out", "cross.q", "cross.kv", "cross.out", "ff.proj", "ff.out")
_HEAD = ("pre_conv", "proj_in", "time_embed.0", "time_embed.2", "global_embed.0", "global_embed.2", "gce.0", "gce.2",
         "cond_embed.0", "cond_embed.2", "proj_out", "post_conv")


def _dit_shapes(case):
    """name -> shape of every tensor, weights first to last as the model holds them"""
    dim, inner = 64 * case["heads"], case["inner"]
    dims = [(_IO, _IO), (_IO, dim), (_TIME, dim), (dim, dim), (_COND, dim), (dim, dim), (dim, dim), (dim, 6 * dim),
            (_COND, dim), (dim, dim), (dim, _IO), (_IO, _IO)]
    got = {"dit.%s.weight" % n: (o, i) for n, (i, o) in zip(_HEAD, dims)}
    for n, (_, o) in zip(_HEAD, dims):
        if n.startswith(("time_embed", "gce")):
            got["dit.%s.bias" % n] = (o,)
    got["dit.memory_tokens"] = (_MEM, dim)
    for l in range(case["depth"]):
        for n, (i, o) in zip(_BLOCK, _targets(dim, inner)):
            got["dit.%d.%s.weight" % (l, n)] = (o, i)
        got["dit.%d.ff.proj.bias" % l], got["dit.%d.ff.out.bias" % l] = (2 * inner,), (dim,)
        got["dit.%d.ssg" % l] = (6 * dim,)
        for k, n in _VECS.items():
            if n:
                got["dit.%d.%s" % (l, n)] = (dim,) if k in ("pre_g", "cross_g", "ff_g") else (64,)
        if case["local"]:
            got["dit.%d.local.0.weight" % l], got["dit.%d.local.0.bias" % l] = (dim, case["local"]), (dim,)
            got["dit.%d.local.2.weight" % l], got["dit.%d.local.2.bias" % l] = (dim, dim), (dim,)
    return got


def _dit_tensor(d, name, shape):
    if name.endswith(".weight"):
        return d.normal(shape, 0.02).half()
    if name.endswith(".gamma"):
        return d.normal(shape, 0.1, 1.0)
    return d.normal(shape, 0.1 if name.endswith(".ssg") else 1.0 if name == "dit.memory_tokens" else 0.02)


def _dit_adapters(case, d, norms):
    """{weight name: (A, B, m)} of the full scope, in the arena's order; norms: row norms by name"""
    got = {}
    for n, s in sorted(_dit_shapes(case).items()):
        if n.endswith(".weight"):
            got[n] = d.adapter(s[1], s[0], case["rank"], norms[n] if case["dora"] else None)
    return got


def _dit_batch(case, d):
    b, t = case["batch"], case["frames"]
    x, target = d.normal((b, t, _IO)), d.normal((b, t, _IO))
    time, cross, glob = d.uniform((b,), 0.0, 1.0), d.normal((b, case["ctx"], _COND)), d.normal((b, _COND))
    return x, target, time, cross, glob, d.normal((b, t, case["local"])) if case["local"] else None


def _prepare_dit(case, seed):
    c, k, s = _ctx(), _binding(), _State(case)
    d = _Draw(seed)
    cfg = k.dit_config(_IO, 64 * case["heads"], case["depth"], case["heads"], _COND, _MEM, _TIME, case["inner"], case["window"],
                       local_dim=case["local"])
    s.dit = s.keep(k.Dit(c, cfg, k.TYPE_F16))
    norms = {}
    for n, shape in _dit_shapes(case).items():
        t = _dit_tensor(d, n, shape)
        if n.endswith(".weight"):
            norms[n] = _norms(t)
        s.dit.set_tensor(n, t.cpu().numpy())
    s.dit.setup(case["rank"], float(case["rank"]), case["dora"], k.SCOPE_FULL, case["batch"], case["frames"], case["ctx"],
                case["recompute"])
    s.dit.adapters_init(1, 0.0)   # clears gradients and moments
    ads = _dit_adapters(case, d, norms)
    s.p, _, s.m, s.v = (s.dit.arena(i) for i in range(4))
    p = s.see(s.p)
    c.sync()
    for n, i, o, a, b, m in s.dit.targets():
        A, B, mag = ads[n]
        p[a:a + A.numel()], p[b:b + B.numel()] = A.flatten(), B.flatten()
        if case["dora"]:
            p[m:m + o] = mag
    s.dit.adapters_changed()
    s.x, s.target, s.t, s.cross, s.glob, s.local = _dit_batch(case, d)
    if case["local"]:
        s.dit.set_local(_dev(s.local))
    s.step = 0
    # the moments too where they tell: over many blocks the rounding of 16-bit activations moves a gradient
    # by several percent, whatever the order of its sums, and the updated weights are what compares
    s.out = [s.see(a) for a in ((s.p, s.m, s.v) if case["depth"] <= 4 else (s.p,))]
    s.vel = torch.empty_like(s.x)
    torch.cuda.synchronize()
    if case["mode"] == "velocity":   # a program that samples has its adapters folded in already
        s.dit.forward(_dev(s.x), _dev(s.t), _dev(s.cross), _dev(s.glob), _dev(s.vel))
        c.sync()
    return s


def _run_dit(s):
    x, t, cross, glob = _dev(s.x), _dev(s.t), _dev(s.cross), _dev(s.glob)
    if s.case["mode"] == "velocity":
        s.dit.forward(x, t, cross, glob, _dev(s.vel))
        return s.vel
    s.step += 1
    s.dit.accumulate(x, _dev(s.target), t, cross, glob, want_loss=False)
    s.dit.apply_adamw(HP, s.step)
    return s.out


def _exact_dit(case, seed):
    d = _Draw(seed)
    T = {n: _dit_tensor(d, n, shape) for n, shape in _dit_shapes(case).items()}
    raw = _dit_adapters(case, d, {n: _norms(t) for n, t in T.items() if n.endswith(".weight")})
    x, target, time, cross, glob, local = _dit_batch(case, d)
    train = case["mode"] == "update"
    T = {n: t.double() for n, t in T.items()}
    ads = {n: tuple(t.double().requires_grad_(train) if t is not None else None for t in a) for n, a in raw.items()}
    silu = torch.nn.functional.silu
    L = lambda n, h: _lin64(h, T["dit.%s.weight" % n], *ads["dit.%s.weight" % n], 1.0, T.get("dit.%s.bias" % n))   # noqa: E731
    mlp = lambda n, h: L(n + ".2", silu(L(n + ".0", h)))   # noqa: E731
    # the time features, whose 32-bit argument is part of the model's input
    ramp = torch.arange(_TIME // 2, device="cuda", dtype=torch.float32) / (_TIME // 2 - 1)
    lo, hi = np.float32(math.log(0.5)), np.float32(math.log(1e4))
    f = torch.exp(ramp * float(hi - lo) + float(lo))
    vels = []
    with torch.set_grad_enabled(train):
        for b in range(case["batch"]):
            arg = (time[b] * f * float(np.float32(2 * math.pi))).double()
            g = mlp("global_embed", glob[b].double()[None]) + mlp("time_embed", torch.cat([torch.cos(arg), torch.sin(arg)])[None])
            gc, cx = mlp("gce", g), mlp("cond_embed", cross[b].double())[None]
            h = L("pre_conv", x[b].double()) + x[b].double()
            h = torch.cat([T["dit.memory_tokens"], L("proj_in", h)])[None]
            for l in range(case["depth"]):
                n = ["dit.%d.%s.weight" % (l, t) for t in _BLOCK]
                vecs = {k: T["dit.%d.%s" % (l, v or "ssg")] for k, v in _VECS.items()}
                add = None
                if local is not None:
                    e = mlp("%d.local" % l, local[b].double())
                    add = torch.cat([torch.zeros_like(T["dit.memory_tokens"]), e])[None]
                h = _block64([T[w] for w in n], [T.get(w[:-6] + "bias") for w in n], vecs, [ads[w] for w in n], 1.0, h, cx, gc,
                             case["window"], add)
            v = L("proj_out", h[0, _MEM:])
            v = L("post_conv", v) + v
            vels.append(v.detach())
            if train:
                ((v - target[b].double()).square().sum() / (_IO * case["frames"])).backward()
    if not train:
        return torch.stack(vels)
    flat = lambda pick: torch.cat([pick(t).flatten() for a in ads.values() for t in a if t is not None])   # noqa: E731
    p, g = flat(lambda t: t.detach()), flat(lambda t: t.grad)
    new = list(_adamw64(p, g, torch.zeros_like(p), torch.zeros_like(p), case["batch"]))
    return new if case["depth"] <= 4 else new[:1]


def _dit_work(case):
    b, t, ctx, r, dora, dim = case["batch"], case["frames"], case["ctx"], case["rank"], case["dora"], 64 * case["heads"]
    fl = case["depth"] * _block_work(b, _MEM + t, ctx, case["heads"], case["inner"], r, case["window"], dora)
    sh, weights, params = _dit_shapes(case), 0.0, 0.0
    for n, s in sh.items():
        if not n.endswith(".weight"):
            continue
        weights += math.prod(s)
        params += r * sum(s) + (s[0] if dora else 0)
        head = n.split(".")[1]
        if not head.isdigit():
            rows = b if head in ("time_embed", "global_embed", "gce") else b * ctx if head == "cond_embed" else b * t
            fl += _lin_work(rows, s[1], s[0], r, dora)
        elif ".local." in n:
            fl += _lin_work(b * t, s[1], s[0], r, dora)
    if case["mode"] == "velocity":
        return dict(bytes=2 * weights + 4 * params + 8 * b * t * _IO, flops=fl / 3)
    return dict(bytes=2 * weights + 24 * params + 8 * b * t * _IO, flops=fl)


# -------------------------------------------------------------------------------------------- AdamW
def _adamw_inputs(case, seed):
    d, n = _Draw(seed), case["n"]
    return d.normal((n,), 0.05), d.normal((n,), 1e-3), d.normal((n,), 1e-4), d.uniform((n,), 0.0, 1e-6)


def _prepare_adamw(case, seed):
    s = _State(case)
    s.p, s.g, s.m, s.v = _adamw_inputs(case, seed)
    s.step = 0
    return s


def _run_adamw(s):
    s.step += 1
    _ctx().adamw_clip(_dev(s.p), _dev(s.g), _dev(s.m), _dev(s.v), HP, s.step, s.case["count"])
    return [s.p, s.m, s.v]


def _adamw64(p, g, m, v, count, step=1):
    lr, b1, b2, eps, wd, clip = (float(np.float32(h)) for h in HP)
    g = g / count
    norm = g.norm()
    g = g * torch.where(norm > clip, clip / (norm + 1e-6), torch.ones_like(norm))
    m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
    return p - lr * ((m / (1 - b1 ** step)) / ((v / (1 - b2 ** step)).sqrt() + eps) + wd * p), m, v


def _exact_adamw(case, seed):
    return list(_adamw64(*(t.double() for t in _adamw_inputs(case, seed)), case["count"]))


# ---------------------------------------------------------------------------------------- the calls
def prepare(case, seed):
    s = dict(dit=_prepare_dit, block=_prepare_block, lin=_prepare_lin, chain=_prepare_chain, attn=_prepare_attn,
             adamw=_prepare_adamw)[case["kind"]](case, seed)
    torch.cuda.synchronize()   # the inputs are complete before the context's own stream reads them
    return s


def run(state):
    return dict(dit=_run_dit, block=_run_block, lin=_run_lin, chain=_run_chain, attn=_run_attn,
                adamw=_run_adamw)[state.case["kind"]](state)


def exact(case, seed):
    return dict(dit=_exact_dit, block=_exact_block, lin=_exact_lin, chain=_exact_chain, attn=_exact_attn,
                adamw=_exact_adamw)[case["kind"]](case, seed)


def work(case):
    k = case["kind"]
    if k == "dit":
        return _dit_work(case)
    if k == "block":
        b, s, dim, r = case["batch"], case["seq"], 64 * case["heads"], case["rank"]
        tg = _targets(dim, case["inner"])
        rows = 4 * b * (4 * s * dim + 2 * case["ctx"] * dim + 12 * dim)
        return dict(bytes=rows + sum(_STORED[case["base"]] * i * o + 8 * r * (i + o) + (8 * o if case["dora"] else 0) for i, o in tg),
                    flops=_block_work(b, s, case["ctx"], case["heads"], case["inner"], r, case["window"], case["dora"]))
    if k == "lin":
        n, i, o, r = case["tokens"], case["inp"], case["out"], case["rank"]
        return dict(bytes=_STORED[case["base"]] * i * o + 8 * n * (i + o) + 8 * r * (i + o) + (8 * o if case["dora"] else 0),
                    flops=_lin_work(n, i, o, r, case["dora"]))
    if k == "chain":
        n, i, o, r = case["tokens"], case["inp"], case["out"], case["rank"] * case["adapters"]
        return dict(bytes=_STORED[case["base"]] * i * o + 4 * n * (i + o) + 4 * r * (i + o) + 8 * o,
                    flops=2.0 * n * (i * o + r * i + r * o))
    if k == "attn":
        b, h, sq, sk = case["batch"], case["heads"], case["sq"], case["sk"]
        pairs = _pairs(sq, case["window"]) if case["window"] else float(sq) * sk
        # read q, k (2 branches), v in 16 bits and dO in 32; write o, o1, o2 in 16, the sums and five gradients in 32
        return dict(bytes=b * h * 64 * (4 * sq + 6 * sk + 4 * sq + 6 * sq + 8 * sq + 12 * sk) + 8 * b * h * sq,
                    flops=3 * b * h * pairs * 512)
    return dict(bytes=28.0 * case["n"], flops=14.0 * case["n"])


def tolerance(case):
    """about four times what another tile choice, attention kernel or contraction of W + s B A gives"""
    k = case["kind"]
    if k == "adamw":   # the one f32 clip scale, from a sum of squares in another order
        return {"rel": 1e-6, "max": 1e-5}
    if k == "lin" and case["prec"] == "f32":   # 32-bit sums in another order
        return {"rel": 1e-5, "max": 2e-4}
    if k == "dit":   # one rounding changed in an early layer travels through all that follow
        if case["mode"] == "update" and case["depth"] > 4:   # updated weights: a step is 1e-3 of them
            return {"rel": 8e-4, "max": 0.01}
        return {"rel": 0.03, "max": 0.9 if case["mode"] == "update" else 0.2}
    if k == "block":
        return {"rel": 0.025, "max": 0.2}
    return {"rel": 0.0125, "max": 0.1}   # one layer: bf16 operands rounded at other places
