"""Fused GQA forward parity on the GPU vs the CPU oracle (gqa_naive of
pytorch_reference.py:51-74, plus the causal mask).  Bound: normwise
<= 2e-2 for bf16/f16 outputs; the reference's own f16 allclose gate
(atol = rtol = 5e-3, cutile-attn-gqa/main.py:258-265) on its correctness shape."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce, from_bits, import_submodule, load_golden
from oracle import gqa as ogqa
from oracle.metrics import normwise_rel_err

pytestmark = pytest.mark.gpu
TOL = 2e-2

shapes = import_submodule("shapes")
inputs = import_submodule("inputs")


def run(ops, q, k, v, causal):
    o = ops.gqa_fwd(q.cuda(), k.cuda(), v.cuda(), causal=causal)
    torch.cuda.synchronize()
    return o.cpu()


def test_golden_reference_correctness_shape(ops):
    """Reference SHAPE_CORRECTNESS (1,128,4,2,64), f16, non-causal, reference inputs."""
    announce("gqa golden correctness f16")
    g = load_golden("gqa_correctness_f16")
    q, k, v = (from_bits(g[x], torch.float16) for x in "qkv")
    o = run(ops, q, k, v, causal=False).float().numpy()
    assert np.allclose(o, g["o"], atol=5e-3, rtol=5e-3)
    assert normwise_rel_err(o, g["o"]) <= 5e-3


def test_golden_causal_bf16(ops):
    announce("gqa golden causal bf16 S=80 D=128")
    g = load_golden("gqa_causal_bf16_s80")
    q, k, v = (from_bits(g[x], torch.bfloat16) for x in "qkv")
    o = run(ops, q, k, v, causal=True)
    assert normwise_rel_err(o, g["o"]) <= TOL


CASES = [
    # (B, S, Hq, Hkv, D, causal, dtype)
    (1, 128, 4, 2, 64, False, torch.bfloat16),
    (1, 128, 4, 2, 64, True, torch.float16),
    (2, 200, 8, 2, 128, True, torch.bfloat16),   # ragged S, G = 4
    (1, 257, 8, 8, 128, True, torch.bfloat16),   # MHA (G = 1), ragged
    (1, 190, 8, 1, 64, False, torch.bfloat16),   # MQA (G = 8)
    (1, 64, 6, 3, 128, True, torch.float16),     # G = 2
    (1, 1, 4, 1, 128, True, torch.bfloat16),     # single token
    (1, 1024, 32, 8, 128, True, torch.bfloat16),
    (1, 2048, 32, 8, 128, False, torch.float16),  # reference bench shape (llama3_8b)
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"B{c[0]}S{c[1]}H{c[2]}/{c[3]}D{c[4]}{'c' if c[5] else 'n'}")
def test_parity_vs_oracle(ops, case):
    B, S, Hq, Hkv, D, causal, dt = case
    announce(f"gqa B{B} S{S} Hq{Hq} Hkv{Hkv} D{D} causal={causal} {dt}")
    s = shapes.GQAShape("t", B, S, Hq, Hkv, D, causal)
    q, k, v = inputs.gqa_inputs(s, dtype=dt)
    o = run(ops, q, k, v, causal)
    heads = list(range(Hq)) if Hq * S <= 8192 else [0, Hq // 2 + 1, Hq - 1]
    ref = ogqa.gqa_naive(q, k, v, causal=causal, heads=heads)
    err = normwise_rel_err(o[:, heads], ref[:, heads])
    assert err <= TOL, f"normwise rel err {err:.3e}"


def test_baseline_config(ops):
    """BASELINE config: B1 Hq32 Hkv8 S4096 D128 bf16 causal, N(0,1) inputs;
    three heads (one per distinct position in its KV group) against the oracle."""
    announce("gqa BASELINE causal S4096")
    s = shapes.GQA_BASELINE
    q, k, v = inputs.gqa_inputs(s)
    o = run(ops, q, k, v, True)
    heads = [0, 13, 31]
    ref = ogqa.gqa_naive(q, k, v, causal=True, heads=heads)
    err = normwise_rel_err(o[:, heads], ref[:, heads])
    assert err <= TOL, f"normwise rel err {err:.3e}"
    assert torch.isfinite(o.float()).all()


def test_constant_value_gives_constant_output(ops):
    announce("gqa V=1 -> O=1")
    s = shapes.GQAShape("t", 1, 300, 8, 2, 128, True)
    q, k, _ = inputs.gqa_inputs(s)
    v = torch.ones_like(k)
    o = run(ops, q, k, v, True).float()
    assert torch.all((o - 1.0).abs() <= 1e-2)


def test_causal_first_row_is_first_value(ops):
    """Causal query 0 sees only key 0: O[:, h, 0] = V[:, h // G, 0]."""
    announce("gqa causal row 0")
    s = shapes.GQAShape("t", 1, 128, 4, 2, 128, True)
    q, k, v = inputs.gqa_inputs(s)
    o = run(ops, q, k, v, True).float()
    for h in range(4):
        assert torch.allclose(o[0, h, 0], v[0, h // 2, 0].float(), atol=1e-2, rtol=1e-2)


# Every tile mx_gqa_fwd_tile accepts at these head groupings: (B, S, Hq, Hkv, D, BLOCK_M, wave_m).
# G = 4 covers the 8-wave kernel at 1, 2, 4 heads per workgroup, the 4-wave kernel at 32-row blocks and
# the one-wave-per-SIMD kernel (wave_m 64); G = 2 the 4-wave kernel at 64-row blocks; G = 1 whole-workgroup
# blocks; G = 8 eight heads per workgroup.  Ragged S everywhere.
TILES = [
    (1, 300, 8, 2, 128, 32, 32), (1, 300, 8, 2, 128, 64, 32), (1, 300, 8, 2, 128, 128, 32),
    (1, 300, 8, 2, 128, 256, 32), (1, 300, 8, 2, 128, 64, 64), (2, 300, 8, 2, 128, 128, 64),
    (1, 300, 8, 2, 128, 256, 64),
    (1, 200, 4, 2, 64, 64, 32), (1, 200, 4, 2, 64, 128, 32), (1, 200, 4, 2, 64, 256, 32),
    (1, 200, 4, 2, 64, 128, 64), (1, 200, 4, 2, 64, 256, 64),
    (1, 170, 4, 4, 64, 128, 32), (1, 170, 4, 4, 64, 256, 32), (1, 170, 4, 4, 128, 256, 64),
    (1, 130, 8, 1, 64, 32, 32), (1, 130, 8, 1, 128, 64, 64),
]


@pytest.mark.parametrize("causal", [True, False], ids=["c", "n"])
@pytest.mark.parametrize("case", TILES, ids=lambda c: f"B{c[0]}S{c[1]}H{c[2]}/{c[3]}D{c[4]}bm{c[5]}wm{c[6]}")
def test_tile_parity_vs_oracle(ops, case, causal):
    """Each explicit tile (the reference's --block-m override,
    cutile-attn-gqa/main.py:202-230) against gqa_naive, both dtypes."""
    B, S, Hq, Hkv, D, bm, wm = case
    for dt in (torch.bfloat16, torch.float16):
        announce(f"gqa tile BLOCK_M={bm} wave_m={wm} B{B} S{S} Hq{Hq} Hkv{Hkv} D{D} causal={causal} {dt}")
        assert ops.gqa_tile_supported(Hq, Hkv, D, bm, 64, wm)
        s = shapes.GQAShape("t", B, S, Hq, Hkv, D, causal)
        q, k, v = inputs.gqa_inputs(s, dtype=dt, seed=inputs.SEED + bm + wm)
        o = ops.gqa_fwd(q.cuda(), k.cuda(), v.cuda(), causal=causal, block_m=bm, block_n=64, wave_m=wm)
        torch.cuda.synchronize()
        ref = ogqa.gqa_naive(q, k, v, causal=causal)
        err = normwise_rel_err(o.cpu(), ref)
        assert err <= TOL, f"normwise rel err {err:.3e}"


@pytest.mark.parametrize("bm,wm", [(64, 32), (128, 32), (256, 32), (64, 64), (128, 64), (256, 64)])
def test_tile_baseline_config(ops, bm, wm):
    """The BASELINE shape (B1 Hq32 Hkv8 S4096 D128 bf16 causal) on every
    tile of the reference's BLOCK_M sweep: three heads against the oracle,
    and the tile's output equal to the default tile's up to rounding."""
    announce(f"gqa BASELINE tile BLOCK_M={bm} wave_m={wm}")
    s = shapes.GQA_BASELINE
    q, k, v = (t.cuda() for t in inputs.gqa_inputs(s))
    o = ops.gqa_fwd(q, k, v, causal=True, block_m=bm, block_n=64, wave_m=wm)
    torch.cuda.synchronize()
    heads = [0, 13, 31]
    qc, kc, vc = q.cpu(), k.cpu(), v.cpu()
    ref = ogqa.gqa_naive(qc, kc, vc, causal=True, heads=heads)
    err = normwise_rel_err(o.cpu()[:, heads], ref[:, heads])
    assert err <= TOL, f"normwise rel err {err:.3e}"
    assert torch.isfinite(o.float()).all()


def test_tile_rejections_enqueue_nothing(ops):
    """A tile no kernel has raises before any launch, and leaves out untouched."""
    import importlib

    _lib = importlib.import_module("cuda-oxide-bench_amd._lib")
    s = shapes.GQAShape("t", 1, 128, 8, 2, 128, True)
    q, k, v = (t.cuda() for t in inputs.gqa_inputs(s))
    out = torch.full_like(q, float("nan"))
    for bm, bn, wm in ((64, 32, 32), (16, 64, 32), (32, 64, 64)):
        with pytest.raises(_lib.MXError):
            ops.gqa_fwd(q, k, v, causal=True, out=out, block_m=bm, block_n=bn, wave_m=wm)
    torch.cuda.synchronize()
    assert torch.isnan(out.float()).all()


# Sizes at which the default launch splits the keys between 2 or 4 groups of waves: last tiles of 1, 2 and 63
# keys, a group whose only tile has one key (S 129 and 193), query rows whose group's first tile is masked, one head
# and several per workgroup; and sizes that one group takes, the shortest and one where the choice turns.
ONE_GROUP = [(1, 1, 8, 8, 64), (1, 63, 8, 2, 64), (1, 65, 8, 1, 64), (2, 129, 8, 8, 128), (4, 640, 16, 16, 64)]
KEY_GROUPS = ONE_GROUP + [(1, 191, 16, 4, 64), (1, 257, 8, 4, 64), (1, 320, 8, 1, 128), (2, 447, 8, 8, 64),
                          (1, 1000, 8, 2, 64), (1, 1025, 8, 4, 128), (2, 1001, 16, 4, 64), (1, 577, 32, 8, 128),
                          (1, 129, 8, 8, 64), (1, 130, 8, 2, 64), (1, 193, 8, 1, 64), (1, 193, 8, 8, 128),
                          (1, 257, 8, 2, 128)]


@pytest.mark.parametrize("causal", [True, False], ids=["c", "n"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["b", "h"])
@pytest.mark.parametrize("case", KEY_GROUPS, ids=lambda c: f"B{c[0]}S{c[1]}H{c[2]}/{c[3]}D{c[4]}")
def test_key_groups(ops, case, dt, causal):
    """Every output row against 64-bit attention.  Roundings on the way, each at
    most u = 2^-9 (bf16) or 2^-12 (f16): Q with the scale folded in (moves a
    score by u |s|, so a weight by about u log2-range; scores here stay below
    12), the probabilities, the output; the bound allows 12 u per row's norm of
    the values it mixes.  Scores drift along the keys so that the groups'
    maxima differ, and K and V are followed by NaN in memory."""
    B, S, Hq, Hkv, D = case
    announce(f"gqa key groups B{B} S{S} Hq{Hq} Hkv{Hkv} D{D} causal={causal} {dt}")
    g = torch.Generator().manual_seed(S * 7 + Hq + D)
    q = torch.randn((B, Hq, S, D), generator=g).to(dt)
    k = (torch.randn((B, Hkv, S, D), generator=g) * torch.linspace(1.0, 2.0, S)[:, None]).to(dt)
    v = torch.randn((B, Hkv, S, D), generator=g).to(dt)

    def padded(t):
        buf = torch.full((t.numel() + 8192,), float("nan"), dtype=dt, device="cuda")
        buf[:t.numel()].view(t.shape).copy_(t)
        return buf[:t.numel()].view(t.shape)

    o = ops.gqa_fwd(padded(q), padded(k), padded(v), causal=causal)
    torch.cuda.synchronize()
    kd, vd = (t.double().repeat_interleave(Hq // Hkv, 1) for t in (k, v))
    s = q.double() @ kd.transpose(-1, -2).contiguous() / D ** 0.5
    if causal:
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool).triu(1), float("-inf"))
    p = torch.softmax(s, dim=-1)
    ref = p @ vd
    u = 2.0 ** -9 if dt == torch.bfloat16 else 2.0 ** -12
    err = (o.cpu().double() - ref).norm(dim=-1)
    mixed = torch.sqrt((p ** 2) @ (vd.norm(dim=-1, keepdim=True) ** 2)).squeeze(-1) + ref.norm(dim=-1)
    assert (err <= 12 * u * mixed).all(), (err / (u * mixed)).max()


def _assert_rows(o, q, k, v, causal):
    """Every output row within test_key_groups' bound of 64-bit attention."""
    S, G = q.shape[2], q.shape[1] // k.shape[1]
    kd, vd = (t.double().repeat_interleave(G, 1) for t in (k, v))
    s = q.double() @ kd.transpose(-1, -2).contiguous() / q.shape[3] ** 0.5
    if causal:
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool).triu(1), float("-inf"))
    p = torch.softmax(s, dim=-1)
    ref = p @ vd
    u = 2.0 ** -9 if q.dtype == torch.bfloat16 else 2.0 ** -12
    err = (o.double() - ref).norm(dim=-1)
    mixed = torch.sqrt((p ** 2) @ (vd.norm(dim=-1, keepdim=True) ** 2)).squeeze(-1) + ref.norm(dim=-1)
    assert (err <= 12 * u * mixed).all(), (err / (u * mixed)).max()


# (S, Hq, Hkv, d_qk, d_v, tile): 4 and 2 key groups, one group, the explicit tiles of both kernels, MLA prefill
FAR_BELOW = [(129, 8, 8, 64, 64, None), (193, 8, 2, 64, 64, None), (257, 8, 2, 64, 64, None),
             (193, 8, 8, 128, 128, None), (321, 8, 2, 128, 128, None), (65, 8, 2, 128, 128, None),
             (193, 8, 2, 64, 64, (256, 32)), (193, 8, 2, 128, 128, (256, 64)), (193, 8, 2, 64, 64, (128, 64)),
             (193, 4, 4, 192, 128, None), (193, 4, 4, 96, 64, None)]


@pytest.mark.parametrize("causal", [True, False], ids=["c", "n"])
@pytest.mark.parametrize("low", ["last", "first tile", "tile starts", "all"])
@pytest.mark.parametrize("case", FAR_BELOW, ids=lambda c: f"S{c[0]}H{c[1]}/{c[2]}D{c[3]}-{c[4]}{'t%d-%d' % c[5] if c[5] else ''}")
def test_scores_far_below_the_rest(ops, case, low, causal):
    """Keys that score 240 to 420 powers of two below the others, where a tile
    of them is all that a row has met so far: the last key alone in a key
    group's tile, the whole first tile, the first key of every tile (a causal
    row's only key there), every key."""
    S, Hq, Hkv, dqk, dv, tile = case
    announce(f"gqa far below: {low} S{S} Hq{Hq} Hkv{Hkv} D{dqk}/{dv} tile={tile} causal={causal}")
    g = torch.Generator().manual_seed(S + dqk)
    dt = torch.bfloat16
    q = torch.randn((1, Hq, S, dqk), generator=g).to(dt)
    k = torch.randn((1, Hkv, S, dqk), generator=g).to(dt)
    v = torch.randn((1, Hkv, S, dv), generator=g).to(dt)
    rows = {"last": slice(S - 1, S), "first tile": slice(0, 64), "tile starts": slice(0, S, 64), "all": slice(0, S)}[low]
    q[..., 0], k[..., 0] = 32.0, 0.0
    k[:, :, rows, 0] = -72.0
    args = [t.cuda() for t in (q, k, v)]
    if dqk != dv:
        o = ops.mla_prefill_fwd(*args, causal=causal)
    elif tile is None:
        o = ops.gqa_fwd(*args, causal=causal)
    else:
        o = ops.gqa_fwd(*args, causal=causal, block_m=tile[0], wave_m=tile[1])
    torch.cuda.synchronize()
    _assert_rows(o.cpu(), q, k, v, causal)


@pytest.mark.parametrize("causal", [True, False], ids=["c", "n"])
@pytest.mark.parametrize("low", [0.0, -72.0], ids=["", "low"])
@pytest.mark.parametrize("hidden", ["first tile", "all but last", "first half", "last half", "all"])
@pytest.mark.parametrize("case", FAR_BELOW, ids=lambda c: f"S{c[0]}H{c[1]}/{c[2]}D{c[3]}-{c[4]}{'t%d-%d' % c[5] if c[5] else ''}")
def test_scores_of_minus_infinity(ops, case, hidden, low, causal):
    """Keys hidden by a component of -inf (q > 0 there): the same rows as
    softmax, NaN where a row sees hidden keys only, whether or not the keys are
    split between groups; with the visible keys at the others' level or 240 to
    420 powers of two below zero."""
    S, Hq, Hkv, dqk, dv, tile = case
    announce(f"gqa -inf: {hidden} {low} S{S} Hq{Hq} Hkv{Hkv} D{dqk}/{dv} tile={tile} causal={causal}")
    g = torch.Generator().manual_seed(S + dqk)
    dt = torch.bfloat16
    q = torch.randn((1, Hq, S, dqk), generator=g).to(dt)
    k = torch.randn((1, Hkv, S, dqk), generator=g).to(dt)
    v = torch.randn((1, Hkv, S, dv), generator=g).to(dt)
    rows = {"first tile": slice(0, 64), "all but last": slice(0, S - 1), "first half": slice(0, S // 2),
            "last half": slice(S // 2, S), "all": slice(0, S)}[hidden]
    q[..., 0], k[..., 0] = 32.0, low
    k[:, :, rows, 0] = float("-inf")
    args = [t.cuda() for t in (q, k, v)]
    if dqk != dv:
        o = ops.mla_prefill_fwd(*args, causal=causal)
    elif tile is None:
        o = ops.gqa_fwd(*args, causal=causal)
    else:
        o = ops.gqa_fwd(*args, causal=causal, block_m=tile[0], wave_m=tile[1])
    torch.cuda.synchronize()
    o = o.cpu()
    visible = torch.ones(S, dtype=torch.bool)
    visible[rows] = False
    seen = visible.cumsum(0) > 0 if causal else visible.any().expand(S)  # rows that see a key
    assert torch.isnan(o[:, :, ~seen]).all()
    # the rows that see a key, over the visible keys alone
    S1, G = int(seen.sum()), Hq // Hkv
    if S1 == 0:
        return
    kd, vd = (t.double().repeat_interleave(G, 1) for t in (k[:, :, visible], v[:, :, visible]))
    s = q[:, :, seen].double() @ kd.transpose(-1, -2).contiguous() / dqk ** 0.5
    if causal:
        at = torch.arange(S)
        s = s.masked_fill(at[visible][None, :] > at[seen][:, None], float("-inf"))
    p = torch.softmax(s, dim=-1)
    ref = p @ vd
    err = (o[:, :, seen].double() - ref).norm(dim=-1)
    mixed = torch.sqrt((p ** 2) @ (vd.norm(dim=-1, keepdim=True) ** 2)).squeeze(-1) + ref.norm(dim=-1)
    assert (err <= 12 * 2.0 ** -9 * mixed).all(), (err / (2.0 ** -9 * mixed)).max()
