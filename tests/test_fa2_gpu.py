"""GPU parity of flash-attention 2 (forward and backward) against the oracle.

fp32 path: max abs <= 1e-5 against the oracle's fp32 restatement of the
reference kernels, for O, LSE and the gradients alike.  bf16 path: rel-L2 <= 5e-3 and max abs <= 2e-2 against
the fp32 oracle run on the same bf16-rounded inputs, for O and for the fp32
gradients of the bf16 backward (TEENY_GRAD_F32); gradients stored as bf16
get the same bar with the max-abs part scaled by the tensor's magnitude
above 4 (check_bf16); LSE (fp32) within 2e-2.  Each op is compared on its
own inputs: the backward's oracle receives the same O and LSE the GPU
backward received.  At the full benchmark shapes the GPU runs the whole
problem and the oracle checks every row and key of whole (batch, kv head)
groups.
"""
import math

import numpy as np
import pytest
import torch

from oracle import oracle as O
from teenyformers_amd import _lib, ops

pytestmark = pytest.mark.gpu

F32_TOL = 1e-5
BF16_MAX_ABS = 2e-2
BF16_REL_L2 = 5e-3


def randn(seed, *shape):
    return np.random.default_rng(seed).standard_normal(shape).astype(np.float32)


def dev(a, dtype):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda").to(dtype)


def host(t):
    return t.float().cpu().numpy()


def rel_l2(got, want):
    """||got - want|| / ||want||, or None when the reference is exactly zero:
    there the relative error is undefined and the max-abs bar alone applies
    (one query row and one key: O = V, so dP = Delta and dS, dQ and dK are
    exactly zero, and the kernels return rounding noise of ~1e-8)."""
    n = np.linalg.norm(want.ravel())
    return None if n == 0 else float(np.linalg.norm((got - want).ravel()) / n)


def bf16_bar(m):
    """The max-abs bar of a bf16-stored tensor whose largest value is m:
    2e-2 * max(1, 2^(floor(log2 m) - 1)).  2e-2 is 2.56 half-ulps of the
    bf16 binade [2, 4) (half-ulp 2^-7).  A bf16 value in the binade
    [2^e, 2^(e+1)) cannot sit closer than its half-ulp 2^(e-8) to the fp32
    value it stores, so a tensor whose largest values exceed 4 (GQA-summed
    dK/dV, dQ of the 8x-spiked keys: up to ~36) gets the same 2.56 half-ulps
    of its top binade; unit-scale tensors, such as every output at the B8 H32
    S4096 D128 shape, get the flat 2e-2."""
    return BF16_MAX_ABS * max(1.0, 2.0 ** (math.floor(math.log2(m)) - 1)) if m > 0 else BF16_MAX_ABS


def check_bf16(name, got, want):
    """bf16 bar: rel-L2 <= 5e-3 and max abs <= bf16_bar(max|want|)."""
    err = float(np.abs(got - want).max())
    r = rel_l2(got, want)
    bar = bf16_bar(float(np.abs(want).max()))
    assert err <= bar and (r is None or r <= BF16_REL_L2), \
        f"{name}: max abs {err:.3e} (bar {bar:.3e}), rel-L2 {r}"


def check_flat(name, got, want):
    """The stated bf16 bar without scaling: rel-L2 <= 5e-3, max abs <= 2e-2
    (for outputs that are not rounded to bf16: O's error is the bf16
    rounding of its own storage, but the fp32 gradients carry only the
    kernels' bf16 operand rounding)."""
    err = float(np.abs(got - want).max())
    r = rel_l2(got, want)
    assert err <= BF16_MAX_ABS and (r is None or r <= BF16_REL_L2), \
        f"{name}: max abs {err:.3e}, rel-L2 {r}"


def launched(f):
    """f's result and the names of the library's kernels that it launched."""
    _lib.profile_enable(True)
    try:
        out = f()
        return out, sorted(_lib.profile_stats())
    finally:
        _lib.profile_enable(False)


def inputs(seed, B, Hq, Hkv, Sq, Sk, D, bf16, spike=False):
    q, k, v, do = (randn(seed, B, Hq, Sq, D), randn(seed + 1, B, Hkv, Sk, D),
                   randn(seed + 2, B, Hkv, Sk, D), randn(seed + 3, B, Hq, Sq, D))
    if spike:  # 1% of K rows x8 stresses the running max
        rows = np.random.default_rng(seed + 4).choice(Sk, max(1, Sk // 100), replace=False)
        k[:, :, rows] *= 8
    if bf16:
        q, k, v, do = (O.bf16_round(t) for t in (q, k, v, do))
    return q, k, v, do


# ---------------------------------------------------------------------------
# fp32: the reference's precision
# ---------------------------------------------------------------------------

def test_c1_rope_transpose_fa2_f32(cuda):
    """B1 H4 S128 D64: RoPE (theta 1e4) + [B,S,H,D]->[B,H,S,D] + causal FA2."""
    B, S, H, D = 1, 128, 4, 64
    qs, ks, vs = randn(100, B, S, H * D), randn(101, B, S, H * D), randn(102, B, S, H * D)
    lnb = float(np.log(np.float32(1e4)).astype(np.float32))
    q = ops.rope(ops.transpose_heads(dev(qs, torch.float32), H), 1e4)
    k = ops.rope(ops.transpose_heads(dev(ks, torch.float32), H), 1e4)
    v = ops.transpose_heads(dev(vs, torch.float32), H)
    o, lse = ops.flash_attn2_fwd(q, k, v, 1.0 / math.sqrt(D), causal=True)
    qe = O.rope(O.transpose_heads(qs, B, S, H, D), lnb)
    ke = O.rope(O.transpose_heads(ks, B, S, H, D), lnb)
    ve = O.transpose_heads(vs, B, S, H, D)
    oe, le = O.fa2_fwd(qe, ke, ve, 1.0 / math.sqrt(D), True)
    assert np.abs(host(o) - oe).max() <= F32_TOL
    assert np.abs(host(lse) - le).max() <= F32_TOL


F32_SHAPES = [  # B, Hq, Hkv, Sq, Sk, D
    (1, 4, 4, 128, 128, 64),
    (2, 4, 2, 77, 77, 32),
    (1, 2, 1, 40, 90, 16),
    (1, 2, 2, 90, 40, 128),
    (1, 3, 3, 65, 65, 8),
]


@pytest.mark.parametrize("shape", F32_SHAPES)
@pytest.mark.parametrize("causal", [True, False])
def test_fa2_f32_fwd_bwd(cuda, shape, causal):
    B, Hq, Hkv, Sq, Sk, D = shape
    q, k, v, do = inputs(10, *shape, bf16=False)
    scale = 1.0 / math.sqrt(D)
    qd, kd, vd, dod = (dev(t, torch.float32) for t in (q, k, v, do))
    o, lse = ops.flash_attn2_fwd(qd, kd, vd, scale, causal)
    oe, le = O.fa2_fwd(q, k, v, scale, causal)
    assert np.abs(host(o) - oe).max() <= F32_TOL
    assert np.abs(host(lse) - le).max() <= F32_TOL
    dq, dk, dv = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, causal)
    dqe, dke, dve = O.fa2_bwd(q, k, v, oe, do, le, scale, causal)
    for name, got, want in (("dq", dq, dqe), ("dk", dk, dke), ("dv", dv, dve)):
        err = float(np.abs(host(got) - want).max())
        print(f"fa2 f32 {shape} causal={causal} {name}: max abs {err:.2e} "
              f"(max |want| {np.abs(want).max():.2f})", flush=True)
        assert err <= F32_TOL, f"{name} {err}"


F32_EDGES = [  # B, Hq, Hkv, Sq, Sk, D: 16-row wavefronts, 32-row tiles, 64-row workgroups
    (1, 1, 1, 1, 1, 64),
    (2, 2, 2, 15, 17, 128),
    (1, 2, 1, 16, 31, 32),
    (1, 2, 2, 33, 32, 16),
    (1, 4, 2, 63, 65, 64),
    (1, 1, 1, 97, 128, 8),
    (1, 8, 1, 200, 70, 64),     # the dK/dV walk shared out over workgroups
    (2, 4, 1, 161, 161, 128),   # ... unevenly
]


@pytest.mark.parametrize("shape", F32_EDGES)
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("aligned", [True, False])
def test_fa2_f32_edges(cuda, shape, causal, aligned):
    """Tile and wavefront edges against the oracle; tensors that start 4 bytes
    past a 16-byte boundary take the kernels' register copy.  The gradients
    sum up to group * Sq fp32 terms: the flat bar scaled by the largest one."""
    B, Hq, Hkv, Sq, Sk, D = shape

    def put(a):
        t = torch.empty(a.size + 1, dtype=torch.float32, device="cuda")[0 if aligned else 1:]
        t = t[:a.size].view(a.shape)
        t.copy_(torch.from_numpy(a))
        return t

    q, k, v, do = inputs(30, *shape, bf16=False)
    scale = 1.0 / math.sqrt(D)
    qd, kd, vd, dod = (put(t) for t in (q, k, v, do))
    o, lse = ops.flash_attn2_fwd(qd, kd, vd, scale, causal, out=put(np.zeros_like(q)))
    oe, le = O.fa2_fwd(q, k, v, scale, causal)
    assert np.abs(host(o) - oe).max() <= F32_TOL
    assert np.abs(host(lse) - le).max() <= F32_TOL
    grads, names = launched(lambda: ops.flash_attn2_bwd(
        qd, kd, vd, put(oe), lse, dod, scale, causal, dq=put(np.zeros_like(q)),
        dk=put(np.zeros_like(k)), dv=put(np.zeros_like(v))))
    # walks of at least two shares of four q tiles are shared out (their merge
    # stores whole vectors)
    shared = Hq // Hkv * math.ceil(Sq / 32) >= 8
    assert ("teeny_fa2_dkdv_merge_bf16_g32" in names) == (shared and aligned)
    for name, got, want in zip(("dq", "dk", "dv"), grads, O.fa2_bwd(q, k, v, oe, do, le, scale, causal)):
        err = float(np.abs(host(got) - want).max())
        assert err <= F32_TOL * max(1.0, float(np.abs(want).max())), f"{name} {err}"


@pytest.mark.parametrize("shape", [  # B, Hq, Hkv, Sq, Sk, D
    (1, 1, 1, 40, 40, 64), (2, 4, 2, 100, 100, 128), (1, 2, 1, 70, 70, 32), (1, 2, 2, 37, 37, 16),
    (1, 1, 1, 65, 65, 8),
    (1, 2, 1, 50, 90, 64),     # keys past every query row
    (1, 8, 1, 200, 70, 64),    # the dK/dV walk shared out over workgroups
])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_fa2_f32_causal_masked_rows_are_inert(cuda, shape, bad):
    """A causally masked (query, key) pair has no influence, whatever its rows
    hold: with K and V not finite from key n on, query rows before n keep the
    O, LSE and dQ of finite K and V; with Q, dO and LSE not finite before
    query n, keys from n on keep their dK and dV.  n falls inside the 32-row
    tiles, at their edges and at the 16-row wavefronts'."""
    B, Hq, Hkv, Sq, Sk, D = shape
    q, k, v, do = inputs(40, *shape, bf16=False)
    scale = 1.0 / math.sqrt(D)
    oe, le = O.fa2_fwd(q, k, v, scale, True)
    want = O.fa2_bwd(q, k, v, oe, do, le, scale, True)

    def same(name, n, got, exact):
        got = host(got)
        assert np.isfinite(got).all(), f"{name} n={n}"
        bar = F32_TOL * max(1.0, float(np.abs(exact).max()))
        assert np.abs(got - exact).max() <= bar, f"{name} n={n}"

    put = lambda t: dev(t, torch.float32)  # noqa: E731
    qd, kd, vd, dod, od, lsed = (put(t) for t in (q, k, v, do, oe, le))
    for n in (1, 7, 16, 31, 32, 33, min(Sq, Sk) - 1, min(Sq, Sk)):
        kb, vb = kd.clone(), vd.clone()
        kb[:, :, n:] = vb[:, :, n:] = bad
        o, lse = ops.flash_attn2_fwd(qd, kb, vb, scale, True)
        dq, _, _ = ops.flash_attn2_bwd(qd, kb, vb, od, lsed, dod, scale, True)
        same("o", n, o[:, :, :n], oe[:, :, :n])
        same("lse", n, lse.view(B, Hq, Sq)[:, :, :n], le.reshape(B, Hq, Sq)[:, :, :n])
        same("dq", n, dq[:, :, :n], want[0][:, :, :n])
        qb, dob, lb = qd.clone(), dod.clone(), lsed.clone()
        qb[:, :, :n] = dob[:, :, :n] = bad
        lb.view(B, Hq, Sq)[:, :, :n] = bad
        _, dk, dv = ops.flash_attn2_bwd(qb, kd, vd, od, lb, dob, scale, True)
        if n < Sk:
            same("dk", n, dk[:, :, n:], want[1][:, :, n:])
            same("dv", n, dv[:, :, n:], want[2][:, :, n:])


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_fa2_f32_visible_infinities(cuda, causal, D):
    """One infinite V element reaches its own column of the rows that see it
    and nothing else, in a tile on the diagonal as elsewhere; a key whose
    score is -inf for every query (an infinite K element against queries of
    one sign) has dK = dV = 0, also where the last query tile is ragged."""
    B, H, S, r, d = 1, 2, 77, 41, 5
    q, k, v, do = inputs(44, B, H, H, S, S, D, bf16=False)
    scale = 1.0 / math.sqrt(D)
    oe, le = O.fa2_fwd(q, k, v, scale, causal)
    vb = v.copy()
    vb[:, :, r, d] = np.inf
    o, lse = ops.flash_attn2_fwd(*(dev(t, torch.float32) for t in (q, k, vb)), scale, causal)
    o = host(o)
    sees = np.arange(S) >= (r if causal else 0)
    assert np.isposinf(o[:, :, sees, d]).all()
    o[:, :, sees, d] = oe[:, :, sees, d]
    assert np.abs(o - oe).max() <= F32_TOL
    assert np.abs(host(lse).reshape(le.shape) - le).max() <= F32_TOL
    q[..., 0] = np.abs(q[..., 0]) + 0.125
    kb = k.copy()
    kb[:, :, r, 0] = -np.inf
    keep = np.arange(S) != r
    qd, kd, vd, dod = (dev(t, torch.float32) for t in (q, kb, v, do))
    o, lse = ops.flash_attn2_fwd(qd, kd, vd, scale, causal)
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    _, dk, dv = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, causal)
    assert not dk[:, :, r].any() and not dv[:, :, r].any()
    assert torch.isfinite(dk[:, :, keep]).all() and torch.isfinite(dv[:, :, keep]).all()


# ---------------------------------------------------------------------------
# bf16 MFMA path
# ---------------------------------------------------------------------------

BF16_SHAPES = [  # B, Hq, Hkv, Sq, Sk, D
    (1, 4, 4, 128, 128, 64),
    (2, 8, 2, 300, 300, 128),   # GQA 4, ragged
    (1, 8, 1, 513, 513, 128),   # GQA 8 (MQA), ragged past a tile
    (2, 4, 4, 256, 256, 64),
    (1, 4, 2, 100, 300, 128),   # Sq < Sk
    (1, 4, 2, 300, 100, 64),    # Sq > Sk
    (1, 2, 2, 1, 1, 64),        # one row
    (1, 2, 2, 1024, 1024, 128),
    (2, 8, 2, 200, 260, 64),    # causal: GQA 4 packed (a wavefront per q head), Sq < Sk
    (1, 8, 2, 300, 100, 64),    # GQA 4 packed, Sq > Sk
    (1, 16, 2, 333, 333, 128),  # GQA 8 packed
    (1, 4, 1, 1, 100, 64),      # GQA 4 packed, one query row
    (2, 8, 2, 33, 70, 128),     # GQA 4 packed, one row past a 32-row block
]


@pytest.mark.parametrize("shape", BF16_SHAPES)
@pytest.mark.parametrize("causal", [True, False])
def test_fa2_bf16_fwd(cuda, shape, causal):
    B, Hq, Hkv, Sq, Sk, D = shape
    q, k, v, _ = inputs(20, *shape, bf16=True, spike=True)
    scale = 1.0 / math.sqrt(D)
    o, lse = ops.flash_attn2_fwd(dev(q, torch.bfloat16), dev(k, torch.bfloat16),
                                 dev(v, torch.bfloat16), scale, causal)
    oe, le = O.fa2_fwd(q, k, v, scale, causal)
    check_bf16("O", host(o), oe)
    assert np.abs(host(lse) - le).max() <= 2e-2


MERGED_SHAPES = BF16_SHAPES + [
    (16, 32, 8, 512, 512, 128),    # the Llama-3-8B prefill's attention
    (1, 8, 8, 2048, 2048, 128),    # plain, several row blocks
    (1, 8, 2, 5000, 5000, 128),    # GQA 4 packed, long
]


@pytest.mark.parametrize("shape", MERGED_SHAPES)
@pytest.mark.parametrize("causal", [True, False])
def test_fa2_bf16_fwd_merged(cuda, shape, causal):
    """The merged-heads forward writes [B, Sq, Hq*D]: bit for bit
    merge_heads of the [B, Hq, Sq, D] forward, LSE bit for bit the same."""
    B, Hq, Hkv, Sq, Sk, D = shape
    g = torch.Generator(device="cuda").manual_seed(Sq * 7 + Hq)
    q = torch.randn((B, Hq, Sq, D), generator=g, device="cuda").to(torch.bfloat16)
    k = torch.randn((B, Hkv, Sk, D), generator=g, device="cuda").to(torch.bfloat16)
    v = torch.randn((B, Hkv, Sk, D), generator=g, device="cuda").to(torch.bfloat16)
    scale = 1.0 / math.sqrt(D)
    o, lse = ops.flash_attn2_fwd(q, k, v, scale, causal)
    om, lm = ops.flash_attn2_fwd_merged(q, k, v, scale, causal)
    torch.cuda.synchronize()
    assert om.shape == (B, Sq, Hq * D)
    assert torch.equal(om.view(torch.int16), ops.merge_heads(o).view(torch.int16))
    assert torch.equal(lm.view(torch.int32), lse.view(torch.int32))


QKV_SHAPES = [  # B, Hq, Hkv, S, cache length, D
    (16, 32, 8, 512, 640, 128),   # the Llama-3-8B prefill (GQA 4 packed)
    (4, 32, 8, 2048, 2048, 64),   # the Llama block
    (2, 8, 8, 300, 320, 128),     # MHA: the 4-wavefront form, ragged
    (1, 16, 2, 333, 400, 128),    # GQA 8 packed
    (1, 8, 2, 8200, 8200, 128),   # the 8-wavefront form (8000+ rows)
    (3, 4, 1, 1, 64, 64),         # one prompt row
]


@pytest.mark.parametrize("shape", QKV_SHAPES)
@pytest.mark.parametrize("causal", [True, False])
def test_fa2_bf16_fwd_qkv(cuda, shape, causal):
    """The prompt attention from the fused QKV projection (its q heads
    rotated as they load, with the RoPE table's (cos, sin)) gives the bits of
    the split into a Q buffer followed by the merged-heads forward; the split
    without q_out writes the same cache rows and nothing else."""
    B, Hq, Hkv, S, L, D = shape
    base = 5e5
    g = torch.Generator(device="cuda").manual_seed(S + Hq + D)
    qkv = torch.randn((B, S, (Hq + 2 * Hkv) * D), generator=g, device="cuda").to(torch.bfloat16)
    kc1 = torch.zeros((B, Hkv, L, D), dtype=torch.bfloat16, device="cuda")
    vc1, kc2, vc2 = torch.zeros_like(kc1), torch.zeros_like(kc1), torch.zeros_like(kc1)
    q = torch.empty((B, Hq, S, D), dtype=torch.bfloat16, device="cuda")
    ops.qkv_rope_split(qkv, q, kc1, vc1, 0, Hq, Hkv, base)
    ops.qkv_rope_split(qkv, None, kc2, vc2, 0, Hq, Hkv, base)
    scale = 1.0 / math.sqrt(D)
    o1, l1 = ops.flash_attn2_fwd_merged(q, kc1, vc1, scale, causal)
    cs = ops.rope_table(S + 3, D, base, "cuda")
    o2, l2 = ops.flash_attn2_fwd_qkv(qkv, cs, kc2, vc2, Hq, scale, causal)
    torch.cuda.synchronize()
    assert torch.equal(kc1.view(torch.int16), kc2.view(torch.int16))
    assert torch.equal(vc1.view(torch.int16), vc2.view(torch.int16))
    assert torch.equal(o2.view(torch.int16), o1.view(torch.int16))
    assert torch.equal(l2.view(torch.int32), l1.view(torch.int32))


def test_rope_table_values(cuda):
    """teeny_rope_table against the angle of rope.rs:86-88 formed as the
    oracle forms it (fp32 theta = fp32(pos) * fp32(exp(fp32(k * c)))), its
    cos and sin taken in float64: within a few fp32 ulps of 1."""
    n, D, base = 4100, 128, 5e5
    cs = ops.rope_table_pairs(ops.rope_table(n, D, base, "cuda"), D).cpu().numpy()
    assert cs.shape == (4128, D // 2, 2)
    cs = cs[:n].astype(np.float64)
    c = np.float32(np.float32(-2.0) * np.float32(ops._ln(base))) / np.float32(D)
    kc = (np.arange(D // 2, dtype=np.float32) * c).astype(np.float64)
    inv = np.exp(kc).astype(np.float32)
    theta = (np.arange(n, dtype=np.float32)[:, None] * inv[None, :]).astype(np.float64)
    err = np.maximum(np.abs(cs[..., 0] - np.cos(theta)), np.abs(cs[..., 1] - np.sin(theta)))
    assert float(err.max()) <= 2.5e-7, float(err.max())


def test_fa2_fwd_merged_rejects_f32(cuda):
    q = torch.zeros((1, 2, 8, 64), device="cuda")
    with pytest.raises(TypeError):
        ops.flash_attn2_fwd_merged(q, q, q)


@pytest.mark.parametrize("B,Hq,Hkv,S,D", [(1, 8, 2, 8300, 64), (1, 8, 2, 5000, 128)])
def test_fa2_bf16_fwd_packed_long(cuda, B, Hq, Hkv, S, D):
    """The GQA-packed causal forward (a wavefront per q head of a group of
    4) on long sequences: D = 64 takes it at any length, D = 128 below 8000
    rows.  The first, a middle and the last 128 query rows of every head
    against the oracle (q_offset gives the slice its causal positions)."""
    q, k, v, _ = inputs(80 + S, B, Hq, Hkv, S, S, D, bf16=True, spike=True)
    scale = 1.0 / math.sqrt(D)
    o, lse = ops.flash_attn2_fwd(dev(q, torch.bfloat16), dev(k, torch.bfloat16),
                                 dev(v, torch.bfloat16), scale, True)
    o, lse = host(o), host(lse)
    for r0 in (0, S // 2 + 5, S - 128):
        oe, le = O.fa2_fwd(q[:, :, r0:r0 + 128], k, v, scale, True, q_offset=r0)
        check_bf16(f"O rows {r0}+", o[:, :, r0:r0 + 128], oe)
        assert np.abs(lse[:, :, r0:r0 + 128] - le).max() <= 2e-2


@pytest.mark.parametrize("causal", [True, False])
def test_fa2_bf16_fwd_late_maximum(cuda, causal):
    """Rows whose maximum score lies far past their first 64-key tile: keys
    150-159 scaled x30 and key 300 x60 put P = 2^(t - m) of the first tile's
    maximum m beyond 2^31 (and beyond fp32 for key 300), so the forward must
    redo those tiles with their own maximum and rescale O and l; O and LSE
    as the oracle's."""
    B, Hq, Hkv, S, D = 1, 4, 2, 384, 128
    q, k, v, _ = inputs(31, B, Hq, Hkv, S, S, D, bf16=True)
    k[:, :, 150:160] *= 30
    k[:, :, 300] *= 60
    k = O.bf16_round(k)
    scale = 1.0 / math.sqrt(D)
    o, lse = ops.flash_attn2_fwd(dev(q, torch.bfloat16), dev(k, torch.bfloat16),
                                 dev(v, torch.bfloat16), scale, causal)
    oe, le = O.fa2_fwd(q, k, v, scale, causal)
    assert np.isfinite(host(o)).all() and np.isfinite(host(lse)).all()
    check_bf16("O", host(o), oe)
    assert np.abs(host(lse) - le).max() <= 2e-2 * max(1.0, float(np.abs(le).max()) / 64)


@pytest.mark.parametrize("shape", BF16_SHAPES)
@pytest.mark.parametrize("causal", [True, False])
def test_fa2_bf16_bwd(cuda, shape, causal):
    B, Hq, Hkv, Sq, Sk, D = shape
    q, k, v, do = inputs(30, *shape, bf16=True)
    scale = 1.0 / math.sqrt(D)
    qd, kd, vd, dod = (dev(t, torch.bfloat16) for t in (q, k, v, do))
    o, lse = ops.flash_attn2_fwd(qd, kd, vd, scale, causal)
    dq, dk, dv = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, causal)
    # the backward op's inputs include O and LSE: the oracle gets the same ones
    dqe, dke, dve = O.fa2_bwd(q, k, v, host(o), do, host(lse), scale, causal)
    check_bf16("dQ", host(dq), dqe)
    check_bf16("dK", host(dk), dke)
    check_bf16("dV", host(dv), dve)
    # fp32 gradients from the same kernels: the flat bar
    g32 = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, causal, grad_f32=True)
    assert all(t.dtype == torch.float32 for t in g32)
    for name, got, want in zip(("dQ", "dK", "dV"), g32, (dqe, dke, dve)):
        check_flat(name + " (fp32)", host(got), want)
    # the hi + lo operands leave the fp32 gradients closer to the oracle
    for a, b, w in zip(g32, (dq, dk, dv), (dqe, dke, dve)):
        ra, rb = rel_l2(host(a), w), rel_l2(host(b), w)
        assert ra is None or ra <= rb


@pytest.mark.parametrize("shape", [(1, 4, 2, 2048, 2048, 64), (1, 2, 1, 2100, 2050, 128),
                                   (2, 4, 2, 2200, 2200, 64)])
def test_fa2_bf16_bwd_gqa_two_groups(cuda, shape):
    """Causal GQA with an even group and 2048+ query rows: dK/dV in two
    wavefront groups per workgroup, each walking half of the q heads of the
    same keys, their sums added through LDS; no partial sums, so the larger
    workspace equals the base one.  bf16 and fp32 gradients against the
    oracle."""
    B, Hq, Hkv, Sq, Sk, D = shape
    q, k, v, do = inputs(50, *shape, bf16=True)
    scale = 1.0 / math.sqrt(D)
    qd, kd, vd, dod = (dev(t, torch.bfloat16) for t in (q, k, v, do))
    o, lse = ops.flash_attn2_fwd(qd, kd, vd, scale, True)
    assert ops.flash_attn2_bwd_workspace_bytes(qd, kd) == ops.flash_attn2_bwd_workspace_bytes(qd)
    dq, dk, dv = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, True)
    g32 = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, True, grad_f32=True)
    dqe, dke, dve = O.fa2_bwd(q, k, v, host(o), do, host(lse), scale, True)
    for name, got, w in zip(("dQ", "dK", "dV"), (dq, dk, dv), (dqe, dke, dve)):
        check_bf16(name, host(got), w)
    for name, got, w in zip(("dQ", "dK", "dV"), g32, (dqe, dke, dve)):
        check_flat(name + " (fp32)", host(got), w)


@pytest.mark.parametrize("grad_f32", [False, True])
def test_fa2_bf16_bwd_gqa_split(cuda, grad_f32):
    """B1 Hq2 Hkv1 S12288 D64 causal (a group of 2, 96 key blocks): with the
    workspace of teeny_flash_attn2_bwd_workspace_bytes_gqa each group's q
    heads split over 2 dK/dV workgroups (fp32 partials merged in a fixed
    order); with the base workspace the two-group kernel runs instead.  dQ
    is the same kernel either way; dK and dV agree to the bf16 rounding of
    the summation order (or closer, for fp32 gradients).  The split against
    the oracle: the B1 Hq64 Hkv8 S16384 whole-group test (4 splits)."""
    B, Hq, Hkv, S, D = 1, 2, 1, 12288, 64
    gen = torch.Generator(device="cuda").manual_seed(51)
    q, do = (torch.randn(B, Hq, S, D, generator=gen, device="cuda").to(torch.bfloat16)
             for _ in range(2))
    k, v = (torch.randn(B, Hkv, S, D, generator=gen, device="cuda").to(torch.bfloat16)
            for _ in range(2))
    scale = 1.0 / math.sqrt(D)
    o, lse = ops.flash_attn2_fwd(q, k, v, scale, True)
    small = ops.flash_attn2_bwd_workspace_bytes(q)
    big = ops.flash_attn2_bwd_workspace_bytes(q, k)
    assert big == small + 2 * 2 * B * Hkv * S * D * 4
    outs = []
    for n in (small, big):
        print(f"  workspace {n} bytes, grad_f32={grad_f32}", flush=True)
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        outs.append(ops.flash_attn2_bwd(q, k, v, o, lse, do, scale, True, workspace=ws,
                                        grad_f32=grad_f32))
    torch.cuda.synchronize()
    assert torch.equal(outs[0][0], outs[1][0])
    tol = 2.0 ** -20 if grad_f32 else 2.0 ** -7
    for a, b in ((outs[0][1], outs[1][1]), (outs[0][2], outs[1][2])):
        a, b = host(a), host(b)
        assert np.isfinite(a).all() and np.isfinite(b).all()
        assert np.all(np.abs(a - b) <= np.abs(a) * tol + 1e-6)


@pytest.mark.parametrize("grad_f32", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal", [
    (1, 8, 2, 421, 421, 128, True),    # GQA: shares of 56 items cross head boundaries
    (1, 2, 2, 2000, 130, 64, False),    # MHA, bidirectional, two key blocks
    (1, 8, 1, 200, 300, 64, True),     # causal blocks past the last query row: empty shares
    (1, 4, 1, 2050, 2050, 64, True),   # instead of the two-group kernel, 16 shares
])
def test_fa2_bf16_bwd_shared_walk(cuda, B, Hq, Hkv, Sq, Sk, D, causal, grad_f32):
    """dK/dV walks shared by several workgroups (the default workspace) against
    the unshared kernels (the smaller workspace) and the oracle.  Both sum the
    same fp32 products in another order: fp32 gradients within 2^-16 of the
    tensor's largest value, bf16 ones within one rounding more."""
    q, k, v, do = inputs(61, B, Hq, Hkv, Sq, Sk, D, bf16=True)
    scale = 1.0 / math.sqrt(D)
    qd, kd, vd, dod = (dev(t, torch.bfloat16) for t in (q, k, v, do))
    o, lse = ops.flash_attn2_fwd(qd, kd, vd, scale, causal)
    n = ops.flash_attn2_bwd_workspace_bytes(qd)
    shared = ops._lib.lib().teeny_flash_attn2_bwd_workspace_bytes_shared(
        Sq, Sk, B, Hq, Hkv, D, ops.TEENY_BF16)
    assert shared > ops.flash_attn2_bwd_workspace_bytes(qd, kd)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    a = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, causal, workspace=ws, grad_f32=grad_f32)
    b = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, causal, grad_f32=grad_f32)
    c = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, causal, grad_f32=grad_f32)
    assert all(torch.equal(x, y) for x, y in zip(b, c))  # deterministic
    assert torch.equal(a[0], b[0])
    for x, y in zip(a[1:], b[1:]):
        x, y = host(x), host(y)
        tol = 2.0 ** -16 * np.abs(x).max() + (0.0 if grad_f32 else 2.0 ** -7 * np.abs(x))
        assert np.all(np.abs(x - y) <= tol)
    want = O.fa2_bwd(q, k, v, host(o), do, host(lse), scale, causal)
    for name, got, w in zip(("dq", "dk", "dv"), b, want):
        check_bf16(name, host(got), w)


@pytest.mark.parametrize("grad_f32", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal", [
    (1, 2, 2, 1000, 1000, 64, True),   # blocks of 2 to 16 tiles of 64 keys
    (1, 4, 1, 1025, 1025, 64, True),   # GQA groups of 4: blocks of one tile (none for group 1) to 17
    (1, 1, 1, 33, 960, 64, False),     # 15 tiles, the shortest walk taken
    (2, 2, 1, 1, 1023, 64, False),     # one row, a last tile of 63 keys
    (1, 4, 1, 64, 1985, 128, True),    # keys past every row: a short walk after all
    (1, 2, 2, 970, 1100, 64, True),    # keys past every row beside a long walk
    (1, 1, 1, 1930, 1930, 128, True),
    (1, 2, 2, 130, 1921, 128, False),  # 31 tiles, the last of one key
])
def test_fa2_bf16_bwd_dq_two_key_groups(cuda, B, Hq, Hkv, Sq, Sk, D, causal, grad_f32):
    """dQ whose keys two wavefront groups of a workgroup share (few rows, long
    walks), against the oracle, twice with the same bits.  bf16 gradients at
    the bf16 bar; fp32 ones at the flat bar, and dQ's error, 2^-17 of dS's
    operand rounding (hi + lo) against the stored bf16's 2^-9, at most a
    sixteenth of the bf16 gradient's."""
    q, k, v, do = inputs(67, B, Hq, Hkv, Sq, Sk, D, bf16=True)
    scale = 1.0 / math.sqrt(D)
    qd, kd, vd, dod = (dev(t, torch.bfloat16) for t in (q, k, v, do))
    o, lse = ops.flash_attn2_fwd(qd, kd, vd, scale, causal)
    run = lambda g32: ops.flash_attn2_bwd(  # noqa: E731
        qd, kd, vd, o, lse, dod, scale, causal, grad_f32=g32)
    a, names = launched(lambda: run(grad_f32))
    dq_names = [n for n in names if "_bwd_dq_" in n]
    walk = min(Sq, Sk) if causal else Sk
    assert len(dq_names) == 1 and ("_k2" in dq_names[0]) == (walk >= 15 * D), names
    b = run(grad_f32)
    assert all(torch.equal(x, y) for x, y in zip(a, b))
    want = O.fa2_bwd(q, k, v, host(o), do, host(lse), scale, causal)
    for name, got, w in zip(("dq", "dk", "dv"), a, want):
        (check_flat if grad_f32 else check_bf16)(name, host(got), w)
    if grad_f32:
        assert rel_l2(host(a[0]), want[0]) <= rel_l2(host(run(False)[0]), want[0]) / 16


def _random_shapes(n, seed=2026):
    """Seeded random shapes off the tile grid: ragged lengths, Sq != Sk, GQA
    groups 1-8, both head dims."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        hkv = int(rng.choice([1, 2, 4]))
        group = int(rng.choice([1, 2, 4, 8]))
        sq = int(rng.integers(1, 700))
        sk = sq if rng.random() < 0.5 else int(rng.integers(1, 700))
        out.append((int(rng.integers(1, 4)), hkv * group, hkv, sq, sk, int(rng.choice([64, 128])),
                    bool(rng.random() < 0.6)))
    return out


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal", _random_shapes(12))
def test_fa2_bf16_random_shapes(cuda, B, Hq, Hkv, Sq, Sk, D, causal):
    """Forward and backward at seeded random shapes against the oracle."""
    q, k, v, do = inputs(60 + Sq, B, Hq, Hkv, Sq, Sk, D, bf16=True, spike=Sk >= 100)
    scale = 1.0 / math.sqrt(D)
    qd, kd, vd, dod = (dev(t, torch.bfloat16) for t in (q, k, v, do))
    o, lse = ops.flash_attn2_fwd(qd, kd, vd, scale, causal)
    oe, le = O.fa2_fwd(q, k, v, scale, causal)
    check_bf16("O", host(o), oe)
    finite = np.isfinite(le)  # causal rows with no visible key (Sq > Sk) have no LSE
    assert np.abs(host(lse)[finite] - le[finite]).max(initial=0.0) <= 2e-2
    dq, dk, dv = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, causal)
    dqe, dke, dve = O.fa2_bwd(q, k, v, host(o), do, host(lse), scale, causal)
    check_bf16("dQ", host(dq), dqe)
    check_bf16("dK", host(dk), dke)
    check_bf16("dV", host(dv), dve)
    # fp32 gradients from the same kernels (hi + lo bf16 P and dS): the flat bar
    g32 = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, scale, causal, grad_f32=True)
    for name, got, want in zip(("dQ", "dK", "dV"), g32, (dqe, dke, dve)):
        check_flat(name + " (fp32)", host(got), want)


@pytest.mark.parametrize("B,Hq,Hkv,S,D", [(1, 8, 2, 700, 128), (3, 8, 2, 777, 128),
                                         (16, 32, 8, 512, 128), (2, 8, 8, 1000, 64)])
def test_fa2_bf16_deterministic(cuda, B, Hq, Hkv, S, D):
    """Every output bit-identical across calls: O, LSE, dQ, dK, dV (and
    the fp32-gradient option).  A row maximum that read a matrix product's
    result too early once made whole rows of O and LSE differ by an ulp
    from call to call at D = 128."""
    q, k, v, do = inputs(40 + S, B, Hq, Hkv, S, S, D, bf16=True)
    qd, kd, vd, dod = (dev(t, torch.bfloat16) for t in (q, k, v, do))
    runs = []
    for _ in range(3):
        o, lse = ops.flash_attn2_fwd(qd, kd, vd)
        g = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod)
        g32 = ops.flash_attn2_bwd(qd, kd, vd, o, lse, dod, grad_f32=True)
        runs.append((o, lse) + tuple(g) + tuple(g32))
    for other in runs[1:]:
        for name, x, y in zip(("O", "LSE", "dQ", "dK", "dV", "dQ32", "dK32", "dV32"),
                              runs[0], other):
            assert torch.equal(x, y), name


# ---------------------------------------------------------------------------
# Full benchmark shapes: whole (batch, kv head) groups against the oracle
# ---------------------------------------------------------------------------

def _group_check(B, Hq, Hkv, S, D, seed, spike, groups):
    """Run fwd+bwd at full size on the GPU, with bf16 and with fp32
    gradients; the oracle then evaluates every query row of each listed
    (b, kv head) group's q heads and every key of its kv head: O, LSE, dQ
    and the GQA-summed dK/dV, key block 0 (which accumulates every query
    row of every q head of the group) included."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shape_q, shape_kv = (B, Hq, S, D), (B, Hkv, S, D)
    q = torch.randn(shape_q, generator=gen, device="cuda").to(torch.bfloat16)
    k = torch.randn(shape_kv, generator=gen, device="cuda")
    if spike:
        idx = torch.randperm(S, generator=gen, device="cuda")[: max(1, S // 100)]
        k[:, :, idx] *= 8
    k = k.to(torch.bfloat16)
    v = torch.randn(shape_kv, generator=gen, device="cuda").to(torch.bfloat16)
    do = torch.randn(shape_q, generator=gen, device="cuda").to(torch.bfloat16)
    scale = 1.0 / math.sqrt(D)
    o, lse = ops.flash_attn2_fwd(q, k, v, scale, True)
    dq, dk, dv = ops.flash_attn2_bwd(q, k, v, o, lse, do, scale, True)
    g32 = ops.flash_attn2_bwd(q, k, v, o, lse, do, scale, True, grad_f32=True)
    torch.cuda.synchronize()
    group = Hq // Hkv
    for b, hk in groups:
        print(f"  group b={b} kv head {hk}", flush=True)
        hs = slice(hk * group, (hk + 1) * group)
        qq, dd = host(q[b:b + 1, hs]), host(do[b:b + 1, hs])
        kk, vv = host(k[b:b + 1, hk:hk + 1]), host(v[b:b + 1, hk:hk + 1])
        oe, le = O.fa2_fwd(qq, kk, vv, scale, True)
        check_bf16(f"O[{b},{hk}]", host(o[b:b + 1, hs]), oe)
        assert np.abs(host(lse[b:b + 1, hs]) - le).max() <= 2e-2
        # the backward's inputs include O and LSE: give the oracle the same ones
        og, lg = host(o[b:b + 1, hs]), host(lse[b:b + 1, hs])
        want = O.fa2_bwd(qq, kk, vv, og, dd, lg, scale, True)
        got16 = (dq[b:b + 1, hs], dk[b:b + 1, hk:hk + 1], dv[b:b + 1, hk:hk + 1])
        got32 = (g32[0][b:b + 1, hs], g32[1][b:b + 1, hk:hk + 1], g32[2][b:b + 1, hk:hk + 1])
        for name, a, c, w in zip(("dQ", "dK", "dV"), got16, got32, want):
            check_bf16(f"{name}[{b},{hk}]", host(a), w)
            check_flat(f"{name}[{b},{hk}] (fp32)", host(c), w)
    assert torch.isfinite(dq.float()).all() and torch.isfinite(dk.float()).all()
    assert torch.isfinite(dv.float()).all()


def test_fa2_bf16_c3_full_size(cuda):
    """B8 H32 S4096 D128 causal, the headline shape: two whole heads."""
    _group_check(8, 32, 32, 4096, 128, seed=7, spike=False, groups=[(0, 0), (7, 31)])


@pytest.mark.parametrize("S", [16384, 8191])
def test_fa2_bf16_c5_long_gqa(cuda, S):
    """B1 Hq64 Hkv8 D128 causal, 1% of K rows x8; S = 16384 (each group's q
    heads split over 4 dK/dV workgroups, fp32 partials and their merge) and
    ragged 8191 (dK/dV in two wavefront groups per workgroup): one whole
    GQA group of 8 q heads."""
    _group_check(1, 64, 8, S, 128, seed=8, spike=True, groups=[(0, 5)])


@pytest.mark.parametrize("B,S,groups", [(2, 4096, [(1, 7)]), (16, 512, [(15, 3)]),
                                         (8, 1024, [(0, 0), (7, 5)])])
def test_fa2_bf16_gqa4_packed_group(cuda, B, S, groups):
    """Causal GQA groups of 4 (Hq32 Hkv8 D128), which run the GQA-packed
    forward and dQ: B2 S4096 (its dK/dV runs in two wavefront groups per
    workgroup), the Llama-3-8B prefill's B16 S512 and B8 S1024 (below 2048
    rows, all 512 dK/dV workgroups resident at once, heavy and light key
    blocks paired on each CU); whole groups, 1% of K rows x8."""
    _group_check(B, 32, 8, S, 128, seed=9 + S, spike=True, groups=groups)


@pytest.mark.parametrize("B,Hq,Hkv,S,D,groups", [(8, 32, 8, 1024, 64, [(3, 2)]),
                                                 (2, 32, 32, 1024, 128, [(1, 31), (0, 0)])])
def test_fa2_bf16_dkdv_cu_pairs(cuda, B, Hq, Hkv, S, D, groups):
    """Causal shapes whose 512 dK/dV workgroups are all resident at once, so
    the kernel pairs heavy and light key blocks on each CU: GQA 4 at D = 64
    and MHA at D = 128; whole groups against the oracle."""
    _group_check(B, Hq, Hkv, S, D, seed=11 + S + D, spike=True, groups=groups)
