"""The work that a user of this library has it do, as cases that can be timed.

Most cases are one call of `gpu_moe_forward` on an Ornith-shape layer (hidden
2048, 256 routed experts of width 512 and one shared expert, top 8), from one
token to a 2048-token prompt, on each kind of store a program can create:

  lean    MFMA layouts only (what an engine with its own weights keeps)
  file    the blocks of a model file in the file's orientation
  blocks  GGUF blocks only, in the reference's vec@mat orientation

The others are the 40-layer decode step, and the two large gpu.h operations
around the MoE block: attention and the LM head's product.  Weights are the
library's deterministic synthetic layers (the bytes depend on the seed
alone); `exact` generates the same bytes by itself and computes in 64 bits.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "ornith-flight_amd"))
import ornith_moe as om  # noqa: E402

STORES = {"lean": {"prefill_layout": 2}, "file": {"prefill_layout": False, "file_layout": True},
          "blocks": {"prefill_layout": False}}


def _layer(name, store, T, D=2048, H=512, E=256, k=8, norm=True, literal=False, zipf=0.0,
           wide=False):
    """One layer call.  norm: the input is normalised and added back (a
    model's MoE block); zipf: exponent of a Zipf router bias; wide: Q6_K
    sub-scales over the int8 range, as quantizers emit them, and not the
    generator's [-32, 31]."""
    c = {"kind": "layer", "store": store, "T": T, "D": D, "H": H, "E": E, "k": k, "norm": norm,
         "literal": literal, "zipf": zipf, "wide": wide}
    return dict(c, name=name) if name else c


def listed():
    return [
        # an engine's decode step: the call that replaces the MoE block of one layer
        _layer("decode_1", "lean", 1),
        # a decode batch, on the expert inputs as they are (the benchmark's headline)
        _layer("decode_16", "lean", 16, norm=False),
        # a batch whose router favours a few experts
        _layer("skew_256", "lean", 256, norm=False, zipf=1.1),
        # a prompt
        _layer("prefill_2048", "lean", 2048),
        # a shorter, ragged prompt on scales as real quantizers emit them
        _layer("prefill_wide_709", "lean", 709, wide=True),
        # the same sizes on a model file's own blocks
        _layer("file_1", "file", 1, wide=True),
        _layer("file_24", "file", 24, wide=True),
        _layer("file_1500", "file", 1500, wide=True),
        # a store that keeps the reference's blocks and nothing else
        _layer("blocks_300", "blocks", 300),
        # one token through all 40 layers
        {"name": "stack_1", "kind": "stack", "layers": 40, "T": 1},
        # one attention head over a 4096-token context
        {"name": "attention_4096", "kind": "attention", "S": 4096, "hd": 256},
        # the LM head for a decode batch: fp32 weights, vocabulary 248,320
        {"name": "lm_head_16", "kind": "matmul", "M": 16, "K": 2048, "N": 248320},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["layer"] * 8 + ["stack", "attention", "matmul"])
    if kind == "stack":
        return {"kind": "stack", "layers": rng.randint(4, 24), "T": _log(rng, 1, 16)}
    if kind == "attention":
        return {"kind": "attention", "S": _log(rng, 64, 4096), "hd": rng.choice([64, 96, 128, 256])}
    if kind == "matmul":
        return {"kind": "matmul", "M": rng.randint(1, 16), "K": rng.choice([1024, 2048]),
                "N": 4 * _log(rng, 8192, 62080)}
    store = rng.choice(["lean", "lean", "file", "blocks"])
    D, H, E = rng.choice([(2048, 512, 256)] * 3 + [(1024, 512, 128)])
    return _layer(None, store, _log(rng, 1, 512 if store == "blocks" else 2048), D=D, H=H, E=E,
                  norm=rng.random() < 0.6, literal=rng.random() < 0.2,
                  zipf=1.1 if rng.random() < 0.25 else 0.0, wide=rng.random() < 0.4)


# ---------------------------------------------------------------- preparation
_context = None


def _ctx():
    """The process's context: one stream and workspace, as an engine has."""
    global _context
    if _context is None:
        torch.cuda.init()
        _context = om.Context()
    return _context


class _Device:
    """A device buffer, freed with its last user; `tensor` shows it and keeps it."""

    def __init__(self, buf):
        self.buf, self.ptr, self.size = buf, buf.ptr, buf.size

    def tensor(self, shape, typestr):
        p = om.lib().gpu_device_ptr(_ctx().ptr, self.ptr)
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (p, False),
                                         "version": 2, "strides": None}
        return torch.as_tensor(self, device="cuda")

    def __del__(self):
        c = _ctx()
        c.sync()
        c._bufs = [b for b in c._bufs if b is not self.buf]
        self.buf.free()


class _State:
    """What a program holds: device buffers and, for the layers, a store."""

    store = None

    def __del__(self):
        if self.store is not None:
            self.store.close()


def _upload(a):
    return _Device(_ctx().upload(a))


def _output(shape, typestr="<f4"):
    """A result buffer and the tensor that shows it."""
    b = _Device(_ctx().alloc(int(np.prod(shape)) * 4))
    return b, b.tensor(shape, typestr)


def _tokens(seed, T, D):
    return om.synth_normal(seed, om.synth_stream(0, om.SYN_ACT, 0), T * D, 1.0).reshape(T, D)


def _randn(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator(device="cuda").manual_seed(seed),
                       device="cuda")


def _norm_w(seed, D):
    return np.random.default_rng(seed).uniform(0.5, 1.5, D).astype(np.float32)


def prepare(case, seed):
    s = _State()
    s.case, kind = case, case["kind"]
    if kind == "layer":
        T, D, k, E = case["T"], case["D"], case["k"], case["E"]
        st = s.store = om.Store(_ctx(), 1, D, case["H"], E, k, True, **STORES[case["store"]])
        st.fill_synthetic(0, seed, case["zipf"])
        st.set_norm(0, _norm_w(seed, D))
        if case["wide"]:
            st.set_experts(0, om.MAT_DOWN, 0, _down_blocks(case, seed, range(E + 1)).cpu().numpy(),
                           E + 1)
        s.x = _upload(_tokens(seed, T, D))
        s.out, o = _output((T, D))
        s.idx, i = _output((T, k), "<i4")
        s.w, w = _output((T, k))
        s.result = {"out": o, "idx": i, "w": w}
        s.opts = om.MoEOpts(om.ROUTE_LITERAL if case["literal"] else om.ROUTE_RENORM,
                            om.MOE_ASYNC | (om.MOE_NORM if case["norm"] else 0), 0, 0)
    elif kind == "stack":
        T, n, D = case["T"], case["layers"], 2048
        st = s.store = om.Store(_ctx(), n, D, 512, 256, 8, True, prefill_layout=2)
        for layer in range(n):
            st.fill_synthetic(layer, seed)
        s.tokens = _upload(_tokens(seed, T, D))
        s.x, s.result = _output((T, D))
        s.tmp, _ = _output((T, D))
        s.opts = om.MoEOpts(om.ROUTE_RENORM, om.MOE_ASYNC, 0, 0)
    else:
        a, b, c = _operands(case, seed)
        s.a, s.b = _upload(a.cpu().numpy()), _upload(b.cpu().numpy())
        s.c = _upload(c.cpu().numpy()) if c is not None else None
        s.out, s.result = _output((a.shape[0], a.shape[1] if c is not None else b.shape[1]))
    return s


def _operands(case, seed):
    """Q, K and V, or the hidden states and the head's matrix."""
    if case["kind"] == "attention":
        return tuple(_randn(seed * 3 + i, case["S"], case["hd"]) for i in range(3))
    return (_randn(seed * 2, case["M"], case["K"]), _randn(seed * 2 + 1, case["K"], case["N"]) * 0.02,
            None)


def run(s):
    L, ctx, kind = om.lib(), _ctx(), s.case["kind"]
    if kind == "layer":
        resid = s.x.ptr if s.case["norm"] else None
        ctx.check(L.gpu_moe_forward(ctx.ptr, s.store.ptr, 0, s.x.ptr, s.case["T"], resid,
                                    s.out.ptr, s.idx.ptr, s.w.ptr, C.byref(s.opts)), "forward")
    elif kind == "stack":  # the token's hidden state, then every layer in place
        L.gpu_copy_buffer(ctx.ptr, s.x.ptr, s.tokens.ptr, s.tokens.size)
        ctx.check(L.gpu_moe_forward_stack(ctx.ptr, s.store.ptr, 0, s.case["layers"], s.x.ptr,
                                          s.tmp.ptr, s.case["T"], C.byref(s.opts)), "stack")
    elif kind == "attention":
        L.gpu_attention(ctx.ptr, s.out.ptr, s.a.ptr, s.b.ptr, s.c.ptr, s.case["S"], s.case["hd"])
    else:
        L.gpu_matmul(ctx.ptr, s.out.ptr, s.a.ptr, s.b.ptr, s.case["M"], s.case["N"], s.case["K"],
                     0, 0)
    return s.result


# ---------------------------------------------------------------- bytes, operations
def _active(T, E, k, zipf):
    """Experts that T tokens are expected to use."""
    p = np.arange(1, E + 1, dtype=np.float64) ** -zipf
    p = np.minimum(p * (k / p.sum()), 1.0)
    return float((1.0 - (1.0 - p) ** T).sum())


def _layer_work(T, D, H, E, k, zipf):
    per = D * H // 256 * (2 * 144 + 210)
    rows = T * (k + 1)
    return {"bytes": (_active(T, E, k, zipf) + 1) * per + D * E * 4 + 2 * T * D * 4 + 8 * T * k,
            "flops": rows * 6 * D * H + 2 * T * D * E}


def work(case):
    if case["kind"] == "layer":
        return _layer_work(case["T"], case["D"], case["H"], case["E"], case["k"], case["zipf"])
    if case["kind"] == "stack":
        w = _layer_work(case["T"], 2048, 512, 256, 8, 0.0)
        return {n: v * case["layers"] for n, v in w.items()}
    if case["kind"] == "attention":
        S, hd = case["S"], case["hd"]
        return {"bytes": 16 * S * hd, "flops": 4 * S * S * hd}
    M, K, N = case["M"], case["K"], case["N"]
    return {"bytes": 4 * (M * K + K * N + M * N), "flops": 2 * M * K * N}


def tolerance(case):
    # The layers' products are fp32-class (two fp16 operands or fp32) and
    # their sums fp32: 0.4e-6 to 1.7e-6 off the 64-bit results, and two
    # correct orders of summation twice that apart.  The expert indices are
    # the rule's own.  The stack's errors grow with the residual stream
    # (1e-3 over 40 layers between its two routers).
    if case["kind"] == "stack":
        return {"rel": 4e-3, "max": 4e-2}
    return {"rel": 6e-6, "max": 1e-4, "differ": 0.0}


# ---------------------------------------------------------------- 64-bit results
# SplitMix64 on int64 tensors: products wrap, shifts are made logical.
_G = 0x9E3779B97F4A7C15


def _wrap(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _shr(z, n):
    return (z >> n) & ((1 << (64 - n)) - 1)


def _fmix(z):
    z = (z ^ _shr(z, 30)) * _wrap(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _wrap(0x94D049BB133111EB)
    return z ^ _shr(z, 31)


def _fmix_int(z):
    m = (1 << 64) - 1
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return z ^ (z >> 31)


def _key(seed, kind, expert):
    m = (1 << 64) - 1
    stream = (kind << 24) | expert
    return _fmix_int(_fmix_int((seed + _G) & m) ^ ((stream * _G + _G) & m))


def _words(key, first, n):
    i = torch.arange(first + 1, first + 1 + n, dtype=torch.int64, device="cuda")
    return _fmix(i * _wrap(_G) + _wrap(key))


def _halves(w):
    u = (w & 0xFFFFFFFF).double() * (1.0 / 4294967296.0)
    m, e = torch.frexp(0.001 + 0.009 * u)  # rounded once, to 11 bits
    return torch.ldexp(torch.round(m * 2048.0) / 2048.0, e).half()


def _synth_blocks(seed, kind, expert, n, nbytes):
    """Blocks of one matrix: their leading bytes, and the two halves."""
    w = _words(_key(seed, kind, expert), 0, n * 32).view(n, 32)
    return w[:, :18].contiguous().view(torch.uint8).view(n, 144) if nbytes == 144 else \
        w[:, :26].contiguous().view(torch.uint8).view(n, 208), _halves(w[:, 30]), _halves(w[:, 31])


def _down_blocks(case, seed, experts):
    """The Q6_K blocks of some experts' down matrices, 210 bytes each."""
    n, got = case["D"] * case["H"] // 256, []
    for e in experts:
        body, d, _ = _synth_blocks(seed, 3, e, n, 208)
        sc = body[:, 192:208]
        if case["wide"]:  # each block's first sub-scale at the range's end
            sc[:, 0] = torch.where(sc[:, 0] < 128, 127, 128).to(torch.uint8)
        else:
            sc.copy_(((sc & 63).to(torch.int16) - 32).to(torch.int8).view(torch.uint8))
        got.append(torch.cat([body, d.view(-1, 1).view(torch.uint8)], 1))
    return torch.cat(got)


def _q6k(blocks):
    b = blocks.to(torch.int64)
    ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
    low = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
    shift = torch.arange(0, 8, 2, device="cuda").view(1, 1, 4, 1)
    q = low + (((qh >> shift) & 3) << 4) - 32
    sc = blocks[:, 192:208].contiguous().view(torch.int8).double().view(-1, 2, 4, 2, 1)
    d = blocks[:, 208:210].contiguous().view(torch.half).double().view(-1, 1, 1, 1, 1)
    return (d * sc * q.view(-1, 2, 4, 2, 16).double()).reshape(-1)


def _q4k(seed, kind, expert, n):
    blk, d, dmin = _synth_blocks(seed, kind, expert, n, 144)
    s, qs = blk[:, 4:16].to(torch.int64), blk[:, 16:144].to(torch.int64).view(-1, 4, 1, 32)
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32).double()
    d = d.double().view(-1, 1)
    return ((d * sc.double()).unsqueeze(2) * q
            - (dmin.double().view(-1, 1) * mn.double()).unsqueeze(2)).reshape(-1)


def _matrices(case, seed, e):
    """Gate, up [D, H] and down [H, D] of one expert in 64 bits."""
    D, H, file = case["D"], case["H"], case["store"] == "file"
    n = D * H // 256

    def shape(flat, K, M):
        return flat.view(M, K).t() if file else flat.view(K, M)

    return (shape(_q4k(seed, 1, e, n), D, H), shape(_q4k(seed, 2, e, n), D, H),
            shape(_q6k(_down_blocks(case, seed, [e])), H, D))


def _zipf_bias(seed, E, s):
    key, rank = _key(seed, 6, 0), list(range(1, E + 1))
    m = (1 << 64) - 1
    for i in range(E - 1, 0, -1):
        j = _fmix_int((key + (i + 1) * _G) & m) % (i + 1)
        rank[i], rank[j] = rank[j], rank[i]
    bias = [-float(np.float32(s)) * math.log(r) for r in rank]
    return torch.tensor(bias, dtype=torch.float64, device="cuda").float()


def _normals(seed, kind, n, sigma):
    w = _words(_key(seed, kind, 0), 0, 3 * n)
    parts = sum((w >> 16 * i) & 0xFFFF for i in range(4)).view(n, 3).sum(1)
    return ((parts - 393210).double() / 65536.0 * sigma).float()


def exact(case, seed):
    """The layer in 64 bits; the choice of experts alone follows the engine's
    rule, the order of fp32 sums taken over the hidden index in sequence."""
    if case["kind"] == "stack":
        return None
    if case["kind"] != "layer":
        a, b, c = _operands(case, seed)
        if c is None:
            return a.double() @ b.double()
        return torch.softmax((a.double() @ b.double().t()) / math.sqrt(case["hd"]), 1) @ c.double()
    T, D, E, k = case["T"], case["D"], case["E"], case["k"]
    x = _normals(seed, 5, T * D, 1.0).view(T, D)
    router = _normals(seed, 4, D * E, 0.02)
    router = router.view(E, D).t().contiguous() if case["store"] == "file" else router.view(D, E)
    bias = _zipf_bias(seed, E, case["zipf"]) if case["zipf"] else None
    xin32, xin = x, x.double()
    if case["norm"]:
        w = torch.from_numpy(_norm_w(seed, D)).cuda()
        ss = torch.zeros(T, device="cuda")
        for d in range(D):
            ss = ss + x[:, d] * x[:, d]
        inv = 1.0 / torch.sqrt(ss / float(D) + 1e-6)
        xin32 = w * (x * inv[:, None])
        xin = w.double() * (xin * torch.rsqrt((xin * xin).mean(1, keepdim=True) + 1e-6))
    logits = torch.zeros(T, E, device="cuda")
    for d in range(D):
        logits = logits + xin32[:, d:d + 1] * router[d]
    if bias is not None:
        logits = logits + bias
    top = logits.topk(k, 1).indices
    z = xin @ router.double()
    if bias is not None:
        z = z + bias.double()
    w = torch.softmax(z, 1).gather(1, top) if case["literal"] else torch.softmax(z.gather(1, top), 1)
    out = x.double().clone() if case["norm"] else torch.zeros(T, D, dtype=torch.float64, device="cuda")
    for e in range(E + 1):
        rows, slot = (top == e).nonzero(as_tuple=True) if e < E else (slice(None), None)
        if e < E and rows.numel() == 0:
            continue
        g, u, dn = _matrices(case, seed, e)
        xe = xin[rows]
        y = (torch.nn.functional.silu(xe @ g) * (xe @ u)) @ dn
        if e < E:
            out.index_add_(0, rows, y * w[rows, slot].unsqueeze(1))
        else:
            out += y
    return {"idx": None, "out": out, "w": w}
