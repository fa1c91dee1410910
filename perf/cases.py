"""The work that programs built on teenyformers_amd give it, as cases that can be timed and compared.

Six kinds of case, each one pass through public entry points:

  attn         flash attention forward and backward on [B, H, S, D] tensors (ops.flash_attn2_fwd / _bwd),
               bf16 and fp32, causal or not, MHA and GQA, with or without fp32 gradients
  layer        an attention layer's core through autograd, from projected activations [B, S, H*D] and back:
               head transposes, RoPE, flash attention, head merge
  norm_swiglu  a block's row-wise operations, forward and backward: residual add + RMSNorm, SwiGLU
  block        one decoder block on a prompt (llama.block_forward): every product and operation of a layer
  decode       one greedy decode step over a filled KV cache, replayed from its graph (llama.DecodeGraph)

Sizes are those of the configurations that the tests and the benchmark run, and ragged ones around them.
"""
from __future__ import annotations

import math

import torch

from teenyformers_amd import llama, ops

_DT = {"bf16": torch.bfloat16, "f32": torch.float32}
_EPS = 1e-5

# decoder shapes: the block configuration (hidden 2048) and the 8B-shaped model (hidden 4096)
_MODELS = {
    2048: dict(d_model=2048, n_heads=32, n_kv_heads_=8, intermediate_size=8192),
    4096: dict(d_model=4096, n_heads=32, n_kv_heads_=8, intermediate_size=14336),
}


def listed():
    return [
        # the headline training step: long causal MHA, compute-bound
        dict(name="attn_mha_4k", kind="attn", dtype="bf16", B=8, Hq=32, Hkv=32, Sq=4096, Sk=4096, D=128,
             causal=True, grad_f32=False),
        # fine-tuning on one ragged GQA sequence, gradients left in fp32 for the optimizer
        dict(name="attn_gqa_ragged", kind="attn", dtype="bf16", B=1, Hq=32, Hkv=8, Sq=1021, Sk=1021, D=64,
             causal=True, grad_f32=True),
        # encoder / cross attention: bidirectional, queries and keys of different odd lengths
        dict(name="attn_bidir_cross", kind="attn", dtype="bf16", B=4, Hq=16, Hkv=16, Sq=777, Sk=1023, D=64,
             causal=False, grad_f32=False),
        # the reference's own precision, a training step at its usual head size
        dict(name="attn_f32", kind="attn", dtype="f32", B=2, Hq=16, Hkv=16, Sq=1024, Sk=1024, D=64,
             causal=True, grad_f32=False),
        # a training step of the attention core at the prompt shape of the 8B-shaped model
        dict(name="layer_gqa_512", kind="layer", dtype="bf16", B=16, Hq=32, Hkv=8, S=512, D=128, base=5e5,
             train=True),
        # the smallest call: the reference's fp32 test shape, forward only; launches and host time count
        dict(name="layer_f32_small", kind="layer", dtype="f32", B=1, Hq=4, Hkv=4, S=128, D=64, base=1e4,
             train=False),
        # the memory-bound operations of a training step, 4 x 2048 tokens of the block configuration
        dict(name="norm_swiglu_8k", kind="norm_swiglu", dtype="bf16", M=8192, N=2048, F=8192, fused=False),
        # one block of a prompt of 4 x 2048 tokens
        dict(name="block_bf16", kind="block", dtype="bf16", hidden=2048, B=4, S=2048),
        # interactive decoding: one sequence, a long cache
        dict(name="decode_b1_4k", kind="decode", dtype="bf16", hidden=4096, layers=4, B=1, past=3900,
             capacity=4096),
        # the generation benchmark's batch and prompt
        dict(name="decode_b16", kind="decode", dtype="bf16", hidden=4096, layers=4, B=16, past=520,
             capacity=640),
        # serving: a larger batch of sequences per step
        dict(name="decode_b64", kind="decode", dtype="bf16", hidden=4096, layers=4, B=64, past=520,
             capacity=640),
        # the reference's generation example: one sequence in fp32
        dict(name="decode_f32", kind="decode", dtype="f32", hidden=2048, layers=2, B=1, past=520, capacity=640),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "layer", "norm_swiglu", "block", "decode"])
    f32 = rng.random() < 0.25
    dtype = "f32" if f32 else "bf16"
    if kind in ("attn", "layer"):
        D = rng.choice([32, 64, 128] if f32 else [64, 128])
        Hkv = rng.choice([1, 2, 4, 8, 16])
        Hq = min(64, Hkv * rng.choice([1, 2, 4, 8]))
        longest = 448 * Hkv // Hq if f32 and D == 128 else 1024 if f32 else 8192
        if kind == "layer":
            S = _log(rng, 32, min(longest, 4096))
            limit = _F32_FLOPS if f32 else _BF16_FLOPS / 4
            while _attn_flops(1, Hq, S, S, D, True, True) > limit:
                S = S * 2 // 3
            fit = int(limit / _attn_flops(1, Hq, S, S, D, True, True))
            return dict(kind=kind, dtype=dtype, B=_log(rng, 1, max(1, min(16, fit))), Hq=Hq, Hkv=Hkv, S=S, D=D,
                        base=rng.choice([1e4, 5e5]), train=rng.random() < 0.75)
        causal = rng.random() < 0.75
        Sq = _log(rng, 32, longest)
        Sk = Sq if causal or rng.random() < 0.5 else _log(rng, 32, min(longest, 4096))
        limit = _F32_FLOPS if f32 else _BF16_FLOPS
        while _attn_flops(1, Hq, Sq, Sk, D, causal, True) > limit:
            Sq, Sk = Sq * 2 // 3, Sk * 2 // 3
        fit = int(limit / _attn_flops(1, Hq, Sq, Sk, D, causal, True))
        return dict(kind=kind, dtype=dtype, B=_log(rng, 1, max(1, min(16, fit))), Hq=Hq, Hkv=Hkv, Sq=Sq, Sk=Sk,
                    D=D, causal=causal, grad_f32=not f32 and rng.random() < 0.25)
    if kind == "norm_swiglu":
        N = rng.choice([512, 1000, 2048, 3072, 4096])
        return dict(kind=kind, dtype=dtype, M=_log(rng, 1, 16384), N=N, F=rng.choice([2, 4]) * N,
                    fused=rng.random() < 0.5)
    hidden = rng.choice([2048, 4096])
    if kind == "block":
        return dict(kind=kind, dtype=dtype, hidden=hidden, B=rng.choice([1, 2, 4]),
                    S=_log(rng, 16, 256 if f32 else 2048))
    B = _log(rng, 1, 64)
    past = _log(rng, 64, 4000 if f32 else 12000)
    past = min(past, 65536 // B)
    return dict(kind=kind, dtype=dtype, hidden=2048 if f32 else hidden, layers=1 if f32 else rng.choice([2, 4]),
                B=min(B, 8) if f32 else B, past=past, capacity=past + rng.choice([32, 128, 200]))


# ---------------------------------------------------------------------------
# what a program has in hand
# ---------------------------------------------------------------------------
class _Random:
    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))
        self.dtype = dtype

    def __call__(self, *shape, std=1.0):
        return (torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32) * std).to(self.dtype)


def _config(case):
    return llama.LlamaConfig(n_layers=case.get("layers", 1), vocab_size=32000, max_seq_len=16384, eps=_EPS,
                             rope_base=5e5, **_MODELS[case["hidden"]])


def prepare(case, seed):
    c = case
    dt = _DT[c["dtype"]]
    rnd = _Random(seed, dt)
    s = dict(case=c)
    if c["kind"] == "attn":
        B, Hq, Hkv, Sq, Sk, D = (c[x] for x in ("B", "Hq", "Hkv", "Sq", "Sk", "D"))
        s.update(q=rnd(B, Hq, Sq, D), k=rnd(B, Hkv, Sk, D), v=rnd(B, Hkv, Sk, D), do=rnd(B, Hq, Sq, D))
    elif c["kind"] == "layer":
        B, Hq, Hkv, S, D = (c[x] for x in ("B", "Hq", "Hkv", "S", "D"))
        s.update(q=rnd(B, S, Hq * D), k=rnd(B, S, Hkv * D), v=rnd(B, S, Hkv * D), do=rnd(B, S, Hq * D))
        if c["train"]:
            for x in ("q", "k", "v"):
                s[x].requires_grad_(True)
    elif c["kind"] == "norm_swiglu":
        M, N, F = c["M"], c["N"], c["F"]
        s.update(x=rnd(M, N), res=rnd(M, N), w=1 + rnd(N, std=0.1), z=rnd(M, 2 * F), df=rnd(M, F), dy=rnd(M, N))
    elif c["kind"] == "block":
        cfg = _config(c)
        w = llama.init_weights(cfg, dtype=dt, seed=int(seed))
        s.update(cfg=cfg, w=w, x=rnd(c["B"], c["S"], cfg.d_model))
    else:
        # weights, a cache that a prompt has filled, and the captured step, as the generation program keeps them
        cfg = _config(c)
        model = llama.Llama(cfg, llama.init_weights(cfg, dtype=dt, seed=int(seed))).stream_layout()
        cache = llama.KVCache(cfg, c["B"], c["capacity"], dt)
        for t in cache.k + cache.v:
            t[:, :, :c["past"]] = rnd(c["B"], cfg.n_kv_heads(), c["past"], cfg.head_dim())
        cache.length = c["past"]
        ids = torch.randint(0, cfg.vocab_size, (c["B"], 1), generator=rnd.g, device="cuda")
        s.update(cfg=cfg, model=model, cache=cache, ids=ids, graph=llama.DecodeGraph(model, cache, ids))
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "attn":
        o, lse = ops.flash_attn2_fwd(s["q"], s["k"], s["v"], causal=c["causal"])
        dq, dk, dv = ops.flash_attn2_bwd(s["q"], s["k"], s["v"], o, lse, s["do"], causal=c["causal"],
                                         grad_f32=c["grad_f32"])
        return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv)
    if c["kind"] == "layer":
        with torch.set_grad_enabled(c["train"]):
            q = ops.RopeFunction.apply(ops.TransposeHeadsFunction.apply(s["q"], c["Hq"]), c["base"])
            k = ops.RopeFunction.apply(ops.TransposeHeadsFunction.apply(s["k"], c["Hkv"]), c["base"])
            v = ops.TransposeHeadsFunction.apply(s["v"], c["Hkv"])
            o = ops.MergeHeadsFunction.apply(ops.flash_attn2(q, k, v))
        if not c["train"]:
            return dict(o=o)
        dq, dk, dv = torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"])
        return dict(o=o.detach(), dq=dq, dk=dk, dv=dv)
    if c["kind"] == "norm_swiglu":
        y, h, rstd = ops.fused_add_rmsnorm(s["x"], s["res"], s["w"], _EPS)
        f = ops.swiglu(s["z"])
        dz = ops.swiglu_bwd(s["df"], s["z"])
        if c["fused"]:
            dx, dres, dw = ops.fused_add_rmsnorm_bwd(s["dy"], h, s["w"], rstd)
            return dict(y=y, h=h, rstd=rstd, f=f, dz=dz, dx=dx, dres=dres, dw=dw)
        dx, dw = ops.rmsnorm_bwd(s["dy"], h, s["w"], rstd)
        return dict(y=y, h=h, rstd=rstd, f=f, dz=dz, dx=dx, dw=dw)
    if c["kind"] == "block":
        return dict(y=llama.block_forward(s["cfg"], s["w"], s["x"]))
    # the step at the cache's filled length, as after a prompt
    g, cache = s["graph"], s["cache"]
    g.ids.copy_(s["ids"])
    g.pos.fill_(c["past"])
    cache.length = c["past"]
    g.replay()
    return dict(logits=g.logits, k=cache.k, v=cache.v)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _attn_flops(B, Hq, Sq, Sk, D, causal, train):
    if causal:
        n = min(Sq, Sk)
        pairs = n * (n + 1) / 2 + max(0, Sq - Sk) * Sk
    else:
        pairs = Sq * Sk
    return (14 if train else 4) * pairs * D * B * Hq


# a drawn attention case does no more than these: the headline case's work, and in fp32 a quarter of the listed one's
_BF16_FLOPS = _attn_flops(8, 32, 4096, 4096, 128, True, True)
_F32_FLOPS = _attn_flops(2, 16, 1024, 1024, 64, True, True) / 4


def work(case):
    c = case
    e = 2 if c["dtype"] == "bf16" else 4
    if c["kind"] == "attn":
        B, Hq, Hkv, Sq, Sk, D = (c[x] for x in ("B", "Hq", "Hkv", "Sq", "Sk", "D"))
        g = 4 if c["grad_f32"] else e
        nq, nk = B * Hq * Sq * D, B * Hkv * Sk * D
        return {"bytes": e * (3 * nq + 2 * nk) + 4 * B * Hq * Sq + g * (nq + 2 * nk),
                "flops": _attn_flops(B, Hq, Sq, Sk, D, c["causal"], True)}
    if c["kind"] == "layer":
        B, Hq, Hkv, S, D = (c[x] for x in ("B", "Hq", "Hkv", "S", "D"))
        nq, nk = B * Hq * S * D, B * Hkv * S * D
        return {"bytes": e * (2 * (nq + nk) + (2 * (nq + nk) if c["train"] else 0)),
                "flops": _attn_flops(B, Hq, S, S, D, True, c["train"])}
    if c["kind"] == "norm_swiglu":
        M, N, F = c["M"], c["N"], c["F"]
        return {"bytes": e * (M * N * (6 + c["fused"]) + 6 * M * F + 2 * N) + 4 * M, "flops": M * (20 * N + 30 * F)}
    cfg = _config(c)
    d, D, Hq, Hkv, F = cfg.d_model, cfg.head_dim(), cfg.n_heads, cfg.n_kv_heads(), cfg.d_ff()
    params = d * (Hq + 2 * Hkv) * D + Hq * D * d + 3 * d * F
    if c["kind"] == "block":
        T = c["B"] * c["S"]
        return {"bytes": e * (params + 2 * d + 2 * T * d),
                "flops": 2 * params * T + _attn_flops(c["B"], Hq, c["S"], c["S"], D, True, False)}
    B, L, n, V = c["B"], c["layers"], c["past"] + 1, cfg.vocab_size
    return {"bytes": e * (L * params + V * d + L * B * 2 * Hkv * n * D + B * (d + V)),
            "flops": 2 * B * (L * params + V * d) + L * 4 * B * Hq * n * D}


def tolerance(case):
    if case["dtype"] == "f32":
        # fp32 sums: 1e-7 to 2e-6 off 64 bits
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] == "decode":
        # a few layers in bf16: with the sums of the products in another order the logits are up to 8e-3 apart
        return {"rel": 3e-2, "max": 0.3}
    # operands and results of 8 bits: the start is 2e-3 to 4e-3 off 64 bits
    return {"rel": 1e-2, "max": 0.3}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _angles(S, D, base, pos0=0):
    """cos and sin of the angles that the rotation is defined by: fp32 position times fp32 inverse frequency."""
    ln = torch.tensor(base, dtype=torch.float32, device="cuda").log()
    k = torch.arange(D // 2, dtype=torch.float32, device="cuda")
    inv = (k * (-2.0 * ln / D)).double().exp().float()
    t = (torch.arange(pos0, pos0 + S, dtype=torch.float32, device="cuda")[:, None] * inv[None, :]).double()
    return t.cos(), t.sin()


def _rotate(x, cs, back=False):
    """x [..., S, D] by interleaved pairs."""
    cn, sn = cs
    sn = -sn if back else sn
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * cn - b * sn, a * sn + b * cn), -1).flatten(-2)


def _attention(q, k, v, do, causal):
    """Forward, and with do the backward, of [B, H, S, D] in 64 bits, a head at a time."""
    B, Hq, Sq, D = q.shape
    Hkv, Sk = k.shape[1], k.shape[2]
    o, lse = torch.empty_like(q), torch.empty(q.shape[:3], dtype=q.dtype, device=q.device)
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    scale = 1.0 / math.sqrt(D)
    mask = torch.ones(Sq, Sk, dtype=torch.bool, device=q.device).triu(1) if causal else None
    for b in range(B):
        for h in range(Hq):
            g = h // (Hq // Hkv)
            p = (q[b, h] @ k[b, g].t()).mul_(scale)
            if causal:
                p.masked_fill_(mask, -math.inf)
            lse[b, h] = torch.logsumexp(p, -1)
            p.sub_(lse[b, h][:, None]).exp_()
            o[b, h] = p @ v[b, g]
            if do is not None:
                dv[b, g] += p.t() @ do[b, h]
                ds = (do[b, h] @ v[b, g].t()).sub_((o[b, h] * do[b, h]).sum(-1, keepdim=True)).mul_(p).mul_(scale)
                dq[b, h] = ds @ k[b, g]
                dk[b, g] += ds.t() @ q[b, h]
    return o, lse, dq, dk, dv


def _norm(x, w):
    r = (x.square().mean(-1, keepdim=True) + _EPS).rsqrt()
    return x * r * w, r


def _layer(cfg, w, i, x, pos0, ck=None, cv=None):
    """One decoder block on x [B, S, d]; with a cache (ck, cv) the new rows are written at pos0 and attended after it."""
    B, S, d = x.shape
    Hq, Hkv, D = cfg.n_heads, cfg.n_kv_heads(), cfg.head_dim()
    get = lambda n: w["model.layers.%d.%s.weight" % (i, n)].double()  # noqa: E731
    n1, _ = _norm(x, get("input_layernorm"))
    qkv = (n1.reshape(B * S, d) @ get("self_attn.qkv_proj").t()).view(B, S, Hq + 2 * Hkv, D).transpose(1, 2)
    cs = _angles(S, D, cfg.rope_base, pos0)
    q, k, v = _rotate(qkv[:, :Hq], cs), _rotate(qkv[:, Hq:Hq + Hkv], cs), qkv[:, Hq + Hkv:]
    if ck is None:
        o = _attention(q, k, v.contiguous(), None, True)[0]
    else:
        ck[:, :, pos0:pos0 + 1], cv[:, :, pos0:pos0 + 1] = k, v
        o = _attention(q, ck[:, :, :pos0 + 1], cv[:, :, :pos0 + 1], None, False)[0]
    x = x + (o.transpose(1, 2).reshape(B * S, Hq * D) @ get("self_attn.o_proj").t()).view(B, S, d)
    n2, _ = _norm(x, get("post_attention_layernorm"))
    gu = n2.reshape(B * S, d) @ get("mlp.gate_up_proj").t()
    g, u = gu.chunk(2, -1)
    return x + ((torch.nn.functional.silu(g) * u) @ get("mlp.down_proj").t()).view(B, S, d)


@torch.no_grad()
def exact(case, seed):
    c = case
    if c["kind"] == "decode":
        # the captured step is not needed here: the same weights, cache and ids without it
        cfg, dt = _config(c), _DT[c["dtype"]]
        rnd = _Random(seed, dt)
        w = llama.init_weights(cfg, dtype=dt, seed=int(seed))
        shape = (c["B"], cfg.n_kv_heads(), c["capacity"], cfg.head_dim())
        ks = [torch.zeros(shape, dtype=torch.float64, device="cuda") for _ in range(cfg.n_layers)]
        vs = [torch.zeros(shape, dtype=torch.float64, device="cuda") for _ in range(cfg.n_layers)]
        for t in ks + vs:
            t[:, :, :c["past"]] = rnd(c["B"], cfg.n_kv_heads(), c["past"], cfg.head_dim()).double()
        ids = torch.randint(0, cfg.vocab_size, (c["B"], 1), generator=rnd.g, device="cuda")
        x = w["model.embed_tokens.weight"][ids].double()
        for i in range(cfg.n_layers):
            x = _layer(cfg, w, i, x, c["past"], ks[i], vs[i])
        y, _ = _norm(x[:, 0], w["model.norm.weight"].double())
        return dict(logits=y @ w["model.embed_tokens.weight"].double().t(), k=ks, v=vs)
    s = prepare(case, seed)
    if c["kind"] == "attn":
        o, lse, dq, dk, dv = _attention(*(s[x].double() for x in ("q", "k", "v", "do")), c["causal"])
        return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv)
    if c["kind"] == "layer":
        B, S, D = c["B"], c["S"], c["D"]
        cs = _angles(S, D, c["base"])
        split = lambda x: x.detach().double().view(B, S, -1, D).transpose(1, 2).contiguous()  # noqa: E731
        merge = lambda x: x.transpose(1, 2).reshape(B, S, -1)  # noqa: E731
        q, k = _rotate(split(s["q"]), cs), _rotate(split(s["k"]), cs)
        o, _, dq, dk, dv = _attention(q, k, split(s["v"]), split(s["do"]) if c["train"] else None, True)
        if not c["train"]:
            return dict(o=merge(o))
        return dict(o=merge(o), dq=merge(_rotate(dq, cs, True)), dk=merge(_rotate(dk, cs, True)), dv=merge(dv))
    if c["kind"] == "norm_swiglu":
        x, res, w, z, df, dy = (s[n].double() for n in ("x", "res", "w", "z", "df", "dy"))
        h = x + res
        y, r = _norm(h, w)
        g, u = z.chunk(2, -1)
        sg = torch.sigmoid(g)
        out = dict(y=y, h=h, rstd=r[:, 0], f=g * sg * u,
                   dz=torch.cat((df * u * sg * (1 + g * (1 - sg)), df * g * sg), -1))
        # the stored sum is what the gradient is taken at
        h = h.to(s["x"].dtype).double()
        dot = (dy * w * h).mean(-1, keepdim=True)
        out["dw"] = (dy * h * r).sum(0)
        if c["fused"]:
            out["dx"] = out["dres"] = r * w * (dy - h * r * r * dot)
        else:
            out["dx"] = r * (w * dy - h * r * r * dot)
        return out
    return dict(y=_layer(s["cfg"], s["w"], 0, s["x"].double(), 0))
