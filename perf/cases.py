"""The work that programs built on this package have it do, as cases that can be timed and
compared: the fp16 GEMM family, the W4A16 products and flash attention, each through the
package's public entry points.

    listed()              the cases by name
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   inputs, and the weights laid out once, on the GPU
    run(state)            one pass; its outputs whole
    exact(case, seed)     the same outputs in 64 bits from plain torch
    work(case)            bytes and operations that one pass cannot do without
    tolerance(case)       how far another correct implementation may be off
"""
from __future__ import annotations

import math

import torch

import wmma_ops_amd as wo

DEVICE = "cuda"

# The largest listed pass: no drawn case does more multiply-adds of its kind than these.
MOST_GEMM = 4096 ** 3
MOST_INT4 = 2048 * 14336 * 4096
MOST_ATTN = 4 * 32 * 4096 * 4096 * 128 // 2  # query-key pairs x d of [4, 32, 4096, 128] causal


def listed():
    return [
        # The smallest call: one 512^3 product, where launch latency and host time count.
        dict(name="gemm_512", op="gemm", m=512, n=512, k=512, layout="nn", out="new"),
        # The headline square product.
        dict(name="gemm_4096", op="gemm", m=4096, n=4096, k=4096, layout="nn", out="new"),
        # Sixteen rows against a wide layer (a small decoding batch): streams the weights.
        dict(name="gemm_rows16", op="gemm", m=16, n=11008, k=4096, layout="nn", out="new"),
        # Sizes off every grid (no dimension a multiple of 8) with the alpha / beta epilogue
        # into the caller's C: a program whose shapes come from its data.
        dict(name="gemm_ragged", op="gemm", m=1001, n=4100, k=4099, layout="nn", out="beta"),
        # A linear layer's training step on torch's [out, in] weight: y = x W^T,
        # dx = dy W, dW = dy^T x, the transposes passed as views.
        dict(name="linear_train", op="linear", m=2048, n=4096, k=4096),
        # One decoded token through a quantised layer, in the decode layout.
        dict(name="int4_decode", op="int4", m=1, n=14336, k=4096, group=128, layout="fused",
             half_out=False, act_order=False),
        # A decoding batch of sixteen, slice-major parameters.
        dict(name="int4_batch16", op="int4", m=16, n=4096, k=4096, group=128, layout="sliced",
             half_out=False, act_order=False),
        # Prefill of 2048 tokens through a quantised layer, fp16 activations out.
        dict(name="int4_prefill", op="int4", m=2048, n=14336, k=4096, group=128,
             layout="packed", half_out=True, act_order=False),
        # Causal grouped-query prefill on the [B, S, H, D] activations a projection leaves,
        # passed as transposed views.
        dict(name="attn_prefill", op="attn", b=1, h=32, hkv=8, sq=4096, sk=4096, d=128,
             causal=True, view=True),
        # One new token per sequence against a cache whose length is what it is.
        dict(name="attn_decode", op="attn", b=8, h=32, hkv=8, sq=1, sk=4001, d=128,
             causal=False, view=False),
        # Attention's training step, forward and backward, at the benchmark's shape.
        dict(name="attn_train", op="attn_train", b=4, h=32, hkv=32, sq=4096, sk=4096, d=128,
             causal=True, view=False),
        # Packed sequences of unequal length, forward and backward.
        dict(name="attn_varlen_train", op="varlen", lens="1024,3333,511,4096,77,2050", h=32,
             hkv=8, d=128, causal=True, train=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _round(x, to, lo):
    return max(lo, (x + to // 2) // to * to)


def draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "linear", "int4", "int4", "int4", "attn",
                     "attn", "attn_train", "varlen"])
    if op == "gemm":
        while True:
            m, n, k = _log(rng, 1, 4096), _log(rng, 256, 14336), _log(rng, 256, 14336)
            if rng.random() < 0.6:  # layer sizes are mostly round, rows are what they are
                n, k = _round(n, 128, 256), _round(k, 128, 256)
            if m * n * k <= MOST_GEMM:
                break
        return dict(op=op, m=m, n=n, k=k, layout=rng.choice(["nn", "nn", "nt"]),
                    out=rng.choice(["new", "new", "beta", "inplace"]))
    if op == "linear":
        while True:
            m, n, k = _log(rng, 64, 4096), _log(rng, 512, 8192), _log(rng, 512, 8192)
            if rng.random() < 0.7:
                n, k = _round(n, 128, 512), _round(k, 128, 512)
            if m * n * k <= MOST_GEMM // 2:
                break
        return dict(op=op, m=m, n=n, k=k)
    if op == "int4":
        while True:
            m = rng.randint(1, 4) if rng.random() < 0.3 else _log(rng, 1, 2048)
            n, k = _round(_log(rng, 1024, 14336), 32, 1024), _round(_log(rng, 1024, 14336), 128, 1024)
            if m * n * k <= MOST_INT4:
                break
        layouts = ["packed", "bytes", "sliced"] + (["fused", "fused"] if m <= 4 else [])
        layout = rng.choice(layouts)
        group = 128 if layout == "fused" else rng.choice([128, 128, 128, 64])
        return dict(op=op, m=m, n=n, k=k, group=group, layout=layout,
                    half_out=rng.random() < 0.5, act_order=rng.random() < 0.15)
    heads = rng.choice([(32, 32), (32, 8), (16, 16), (16, 2), (8, 8), (40, 8)])
    d = rng.choice([128, 128, 128, 64, 64, 80, 96, 256])
    causal = rng.random() < 0.5
    if op == "attn" and rng.random() < 0.5:  # decoding: a few queries against a cache
        return dict(op=op, b=_log(rng, 1, 32), h=heads[0], hkv=heads[1], sq=rng.choice([1, 1, 1, 2, 4]),
                    sk=_log(rng, 200, 16384), d=d, causal=False, view=False)
    if op in ("attn", "attn_train"):
        while True:
            b, s = _log(rng, 1, 8), _log(rng, 100, 4096)
            if b * heads[0] * s * s * d <= MOST_ATTN // 2:
                break
        return dict(op=op, b=b, h=heads[0], hkv=heads[1], sq=s, sk=s, d=d, causal=causal,
                    view=rng.random() < 0.5)
    while True:
        lens = [_log(rng, 16, 4096) for _ in range(rng.randint(1, 8))]
        if sum(s * s for s in lens) * heads[0] * d <= MOST_ATTN // 2:
            break
    return dict(op=op, lens=",".join(str(s) for s in lens), h=heads[0], hkv=heads[1], d=d,
                causal=causal, train=rng.random() < 0.5)


# ---- inputs -------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, std=1.0, dtype=torch.float16):
    return torch.randn(*shape, generator=g, device=DEVICE).mul_(std).to(dtype)


def _lens(case):
    return [int(s) for s in case["lens"].split(",")]


def _int4_raw(case, g):
    """q [K, N] of 0..15, scales [K/G, N], zero points [K/G, N] of 1..15."""
    n, k, ng = case["n"], case["k"], case["k"] // case["group"]
    q = torch.randint(0, 16, (k, n), generator=g, device=DEVICE, dtype=torch.int32)
    s = (torch.rand(ng, n, generator=g, device=DEVICE) * 0.009 + 0.001).half()
    z = torch.randint(1, 16, (ng, n), generator=g, device=DEVICE, dtype=torch.int32)
    return q, s, z


def _nibbles(x, dim):
    """Eight 4-bit values along `dim` to one int32, the first in the lowest bits."""
    x = x.unflatten(dim, (-1, 8)).movedim(dim + 1, 0)
    word = torch.zeros_like(x[0])
    for i in range(8):
        word |= x[i] << (4 * i)
    return word


def _inputs(case, seed):
    """Everything that the seed decides, before the package sees it."""
    g, op = _gen(seed), case["op"]
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        a = _randn(g, m, k)
        b = _randn(g, k, n, std=0.02) if case["layout"] == "nn" else _randn(g, n, k, std=0.02).t()
        c = _randn(g, m, n, dtype=torch.float32) if case["out"] != "new" else None
        return dict(a=a, b=b, c=c)
    if op == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(x=_randn(g, m, k), w=_randn(g, n, k, std=0.02), dy=_randn(g, m, n, std=0.1))
    if op == "int4":
        a = _randn(g, case["m"], case["k"])
        q, s, z = _int4_raw(case, g)
        perm = None
        if case["act_order"]:
            perm = torch.randperm(case["k"], generator=g, device=DEVICE)
        return dict(a=a, q=q, s=s, z=z, perm=perm)
    h, hkv, d = case["h"], case["hkv"], case["d"]
    if op == "varlen":
        total = sum(_lens(case))
        return dict(q=_randn(g, total, h, d), k=_randn(g, total, hkv, d), v=_randn(g, total, hkv, d),
                    do=_randn(g, total, h, d))
    b, sq, sk = case["b"], case["sq"], case["sk"]

    def heads(nh, s):
        if case["view"]:
            return _randn(g, b, s, nh, d).transpose(1, 2)
        return _randn(g, b, nh, s, d)

    return dict(q=heads(h, sq), k=heads(hkv, sk), v=heads(hkv, sk), do=heads(h, sq))


def prepare(case, seed):
    st, op = _inputs(case, seed), case["op"]
    st["case"] = case
    if op == "int4":
        qw = _nibbles(st.pop("q"), 0)
        s, z = st.pop("s"), st.pop("z")
        st["out"] = torch.float16 if case["half_out"] else torch.float32
        if case["layout"] == "fused":
            st["w"] = wo.prepack_int4_fused(qw, s, _nibbles(z, 1), case["group"])
        else:
            st["w"] = wo.prepack_int4(qw)
            zeros = z.to(torch.uint8) if case["layout"] == "bytes" else _nibbles(z, 1)
            st["params"] = (wo.prepack_int4_params(s, zeros) if case["layout"] == "sliced"
                            else (s, zeros))
    elif op == "varlen":
        lens = _lens(case)
        cu = torch.zeros(len(lens) + 1, dtype=torch.int32)
        cu[1:] = torch.tensor(lens).cumsum(0)
        st["cu"], st["max"] = cu.to(DEVICE), max(lens)
    if op == "attn_train" or case.get("train"):
        for name in ("q", "k", "v"):
            st[name].requires_grad_(True)
    return st


def run(st):
    case = st["case"]
    op = case["op"]
    if op == "gemm":
        if case["out"] == "new":
            return wo.matmul(st["a"], st["b"])
        if case["out"] == "beta":
            return wo.gemm(st["a"], st["b"], alpha=2.0, beta=0.5, C=st["c"])
        wo.gemm_inplace(st["a"], st["b"], st["c"], 2.0, 0.5)
        return st["c"]
    if op == "linear":
        x, w, dy = st["x"], st["w"], st["dy"]
        return {"y": wo.matmul(x, w.t()), "dx": wo.matmul(dy, w), "dw": wo.matmul(dy.t(), x)}
    if op == "int4":
        if case["layout"] == "fused":
            return wo.matmul_int4_fused(st["a"], st["w"], case["group"], out_dtype=st["out"],
                                        perm=st["perm"])
        return wo.matmul_int4(st["a"], st["w"], *st["params"], case["group"],
                              out_dtype=st["out"], perm=st["perm"])
    q, k, v = st["q"], st["k"], st["v"]
    if op == "varlen":
        o = wo.flash_attention_varlen(q, k, v, st["cu"], st["cu"], st["max"], st["max"],
                                      causal=case["causal"])
    else:
        o = wo.flash_attention(q, k, v, causal=case["causal"])
    if not o.requires_grad:
        return o
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), st["do"])
    return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}


# ---- the same in 64 bits --------------------------------------------------------------------

def _mm(a, b):
    return a.double() @ b.double()


def _attention(q, k, v, causal, do=None):
    """One head: q [Sq, d], k / v [Sk, d] in 64 bits -> o and, with do, dq, dk, dv."""
    scale = 1.0 / math.sqrt(q.shape[-1])
    s = (q @ k.t()).mul_(scale)
    if causal:
        s.masked_fill_(torch.ones_like(s, dtype=torch.bool).triu_(1), -math.inf)
    p = torch.softmax(s, dim=-1)
    o = p @ v
    if do is None:
        return (o,)
    dp = do @ v.t()
    ds = p * (dp - (do * o).sum(-1, keepdim=True))
    return o, (ds @ k).mul_(scale), (ds.t() @ q).mul_(scale), p.t() @ do


def _attention_all(q, k, v, causal, do):
    """Head by head: q [H, Sq, d], k / v [Hkv, Sk, d] of one sequence."""
    group = q.shape[0] // k.shape[0]
    outs = [torch.zeros(t.shape, dtype=torch.float64, device=DEVICE)
            for t in ((q,) if do is None else (q, q, k, v))]
    for i in range(q.shape[0]):
        j = i // group
        got = _attention(q[i].double(), k[j].double(), v[j].double(), causal,
                         None if do is None else do[i].double())
        outs[0][i] = got[0]
        if do is not None:
            outs[1][i] = got[1]
            outs[2][j] += got[2]
            outs[3][j] += got[3]
    return outs


def exact(case, seed):
    st, op = _inputs(case, seed), case["op"]
    if op == "gemm":
        y = _mm(st["a"], st["b"])
        return y if st["c"] is None else y.mul_(2.0).add_(st["c"].double(), alpha=0.5)
    if op == "linear":
        x, w, dy = st["x"], st["w"], st["dy"]
        return {"y": _mm(x, w.t()), "dx": _mm(dy, w), "dw": _mm(dy.t(), x)}
    if op == "int4":
        g = case["group"]
        # the weight is fp16((q - z) s) by definition: q - z is exact, the product rounded once
        w = (st["q"] - st["z"].repeat_interleave(g, 0)).float()
        w = (w * st["s"].float().repeat_interleave(g, 0)).half()
        a = st["a"] if st["perm"] is None else st["a"][:, st["perm"]]
        return _mm(a, w)
    q, k, v = st["q"], st["k"], st["v"]
    do = st["do"] if op == "attn_train" or case.get("train") else None
    if op == "varlen":
        outs = [torch.zeros(t.shape, dtype=torch.float64, device=DEVICE)
                for t in ((q,) if do is None else (q, q, k, v))]
        at = 0
        for s in _lens(case):
            rows = slice(at, at + s)
            part = [None if t is None else t[rows].transpose(0, 1) for t in (q, k, v, do)]
            for o, x in zip(outs, _attention_all(*part[:3], case["causal"], part[3])):
                o[rows] = x.transpose(0, 1)
            at += s
    else:
        per = [_attention_all(q[b], k[b], v[b], case["causal"], None if do is None else do[b])
               for b in range(case["b"])]
        outs = [torch.stack(x) for x in zip(*per)]
    return outs[0] if do is None else dict(zip(("o", "dq", "dk", "dv"), outs))


# ---- what a pass cannot do without ------------------------------------------------------------

def work(case):
    op = case["op"]
    if op in ("gemm", "linear", "int4"):
        m, n, k = case["m"], case["n"], case["k"]
        if op == "linear":  # three products; x, W, dy read once, y, dx, dW written once
            return dict(bytes=2 * (m * k + n * k + m * n) + 4 * (m * n + m * k + n * k),
                        flops=3 * 2 * m * n * k)
        if op == "gemm":
            return dict(bytes=2 * (m * k + k * n) + 4 * m * n * (1 if case["out"] == "new" else 2),
                        flops=2 * m * n * k)
        params = k // case["group"] * n * (3 if case["layout"] == "bytes" else 2.5)
        return dict(bytes=k * n / 2 + params + 2 * m * k + (2 if case["half_out"] else 4) * m * n,
                    flops=2 * m * n * k)
    h, hkv, d = case["h"], case["hkv"], case["d"]
    if op == "varlen":
        lens = _lens(case)
        rows_q = rows_k = sum(lens)
        pairs = sum(s * (s + 1) // 2 if case["causal"] else s * s for s in lens)
    else:
        rows_q, rows_k = case["b"] * case["sq"], case["b"] * case["sk"]
        s, t = case["sq"], case["sk"]
        pairs = case["b"] * (s * (s + 1) // 2 if case["causal"] else s * t)
    qo, kv = 2 * rows_q * h * d, 2 * rows_k * hkv * d
    train = op == "attn_train" or case.get("train")
    # forward: two products; backward: five.  Training reads dO and writes O, dQ, dK, dV.
    return dict(bytes=(2 * qo + 2 * kv) + ((2 * qo + 2 * kv) if train else 0),
                flops=2 * pairs * h * d * (7 if train else 2))


def tolerance(case):
    """About four times the error against 64 bits that the kernels show."""
    op = case["op"]
    if op in ("gemm", "linear"):
        return {"rel": 2e-6}  # fp32 sums of up to 14336 products: 4e-7 seen at 4096
    if op == "int4":
        # a weight with or without its rounding to fp16 (2e-4), the fp16 output (2e-4)
        return {"rel": 1e-3}
    if op == "attn_train" or case.get("train"):
        return {"rel": 1.2e-3}  # fp16 P and dS into the products, fp16 results: 3e-4 seen
    return {"rel": 1e-3}  # fp16 P into the product, fp16 result: 3e-4 seen
