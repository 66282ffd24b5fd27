"""The workloads this framework is timed on, each through its public operators.

A case is a plain dict naming an operator path ("kind") and its sizes.  The
listed cases and draw() cover one range per kind:

  gemm         bf16 linear layer, C = A @ B: from decode batches against a
               weight matrix to 8192^3, M any, N and K multiples of 8
  fp8_linear   fp8 linear layer: activation quantisation (1x128 scales)
               followed by the block-scaled e4m3 GEMM
  gqa          fused grouped-query attention of a prompt, causal or not,
               bf16 or f16, head dims 64 and 128
  mla_prefill  multi-head attention of a prompt on up-projected MLA heads
               (qk 192 / v 128)
  mla_step     one weight-absorbed MLA decode step over a latent cache, all
               128 heads or the 16 to 64 a tensor-parallel rank holds
  gdn, kda     one recurrent decode step, the fp32 state updated in place

Every state holds what a serving or benchmark program has in hand before the
call: activations, weights (quantised once for fp8), the latent cache, the
recurrent state and, for the MLA step, the workspace it keeps.
"""
import importlib
import math

import torch

_pkg = importlib.import_module("cuda-oxide-bench_amd")
ops = _pkg.load_ops()
quant = _pkg.quant

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
_D_C, _D_ROPE, _D_NOPE, _D_V = 512, 64, 128, 128  # MLA widths: latent, rope, nope and value head dims


def listed():
    return [
        # one token through one recurrent layer at batch 1: the smallest call
        {"name": "kda_b1_h32", "kind": "kda", "batch": 1, "heads": 32, "dk": 128, "dv": 128, "dtype": "f16"},
        # the recurrent layer of a decode batch of 64, two value heads per key head
        {"name": "gdn_b64_h32", "kind": "gdn", "batch": 64, "heads": 32, "key_heads": 16, "dk": 128, "dv": 128,
         "dtype": "bf16"},
        # decode batch of 32 at a context of 4096, all 128 heads on one GPU
        {"name": "mla_step_b32_h128_t4096", "kind": "mla_step", "batch": 32, "heads": 128, "ctx": 4096},
        # the 16 heads of one of eight tensor-parallel ranks, a larger batch, a context that is no multiple of a stage
        {"name": "mla_step_b48_h16_t6001", "kind": "mla_step", "batch": 48, "heads": 16, "ctx": 6001},
        # prompt of 4096 tokens, 32 query and 8 key/value heads, causal
        {"name": "gqa_s4096_causal", "kind": "gqa", "batch": 1, "heads": 32, "kv_heads": 8, "seq": 4096, "d": 128,
         "causal": True, "dtype": "bf16"},
        # two shorter prompts of an odd length, the smaller head dim, f16, no mask (an encoder's layer)
        {"name": "gqa_b2_s1001_d64_f16", "kind": "gqa", "batch": 2, "heads": 16, "kv_heads": 4, "seq": 1001, "d": 64,
         "causal": False, "dtype": "f16"},
        # prompt of about 2000 tokens on 128 up-projected MLA heads
        {"name": "mla_prefill_h128_s1900", "kind": "mla_prefill", "batch": 1, "heads": 128, "seq": 1900,
         "causal": True, "dtype": "bf16"},
        # a decode batch of 16 against one weight matrix
        {"name": "gemm_16x7168x4096", "kind": "gemm", "m": 16, "n": 7168, "k": 4096},
        # a mid-size product with every dimension off the tiles
        {"name": "gemm_2000x2040x2056", "kind": "gemm", "m": 2000, "n": 2040, "k": 2056},
        # the largest product
        {"name": "gemm_8192", "kind": "gemm", "m": 8192, "n": 8192, "k": 8192},
        # a decode batch of 64 through an fp8 linear layer
        {"name": "fp8_linear_64x4096x7168", "kind": "fp8_linear", "m": 64, "n": 4096, "k": 7168},
        # a prompt of 3000 tokens through an fp8 linear layer
        {"name": "fp8_linear_3000x7168x2048", "kind": "fp8_linear", "m": 3000, "n": 7168, "k": 2048},
    ]


def _log(rng, lo, hi, step=1):
    """A size between lo and hi, spread over its logarithm, a multiple of step."""
    x = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(-(-lo // step) * step, x // step * step)


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "fp8_linear", "fp8_linear", "gqa", "gqa", "mla_prefill", "mla_step",
                       "mla_step", "gdn", "kda"])
    if kind == "gemm":
        return {"kind": kind, "m": _log(rng, 1, 8192), "n": _log(rng, 512, 8192, 8), "k": _log(rng, 512, 8192, 8)}
    if kind == "fp8_linear":
        return {"kind": kind, "m": _log(rng, 1, 8192), "n": _log(rng, 512, 8192, 16), "k": _log(rng, 512, 8192, 128)}
    if kind == "gqa":
        batch, heads = rng.choice([1, 1, 2, 4]), rng.choice([8, 16, 32])
        return {"kind": kind, "batch": batch, "heads": heads, "kv_heads": heads // rng.choice([1, 2, 4, 8]),
                "seq": _log(rng, 128, 8400 // max(2, batch)), "d": rng.choice([64, 128]),
                "causal": rng.random() < 0.7, "dtype": rng.choice(["bf16", "f16"])}
    if kind == "mla_prefill":
        heads = rng.choice([16, 32, 64, 128])
        return {"kind": kind, "batch": 1, "heads": heads, "seq": _log(rng, 128, 2500), "causal": rng.random() < 0.7,
                "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if kind == "mla_step":
        batch = _log(rng, 1, 64)
        return {"kind": kind, "batch": batch, "heads": rng.choice([16, 32, 64, 128]),
                "ctx": _log(rng, 500, min(32768, 280000 // batch))}
    dk, dv = rng.choice([(64, 64), (128, 128), (128, 128), (256, 256), (512, 512)])
    heads = rng.choice([4, 8, 16, 32, 64])
    most = max(1, (64 << 20) // (heads * dk * dv * 2))  # state of at most 128 MiB in fp32
    case = {"kind": kind, "batch": _log(rng, 1, min(64, most)), "heads": heads, "dk": dk, "dv": dv,
            "dtype": rng.choice(["bf16", "f16"])}
    if kind == "gdn":
        case["key_heads"] = heads // rng.choice([1, 2])
    return case


def _randn(g, shape, dtype, scale=1.0):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (x if scale == 1.0 else x * scale).to(dtype)


def _inputs(case, seed):
    """The values of inputs.py (uniform[-1,1] GEMM operands, N(0,1) attention
    inputs, normalised GDN keys and gated decays), made on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "gemm":
        a = torch.rand((case["m"], case["k"]), generator=g, device="cuda") * 2 - 1
        b = torch.rand((case["k"], case["n"]), generator=g, device="cuda") * 2 - 1
        return {"a": a.to(torch.bfloat16), "b": b.to(torch.bfloat16)}
    if kind == "fp8_linear":
        x = _randn(g, (case["m"], case["k"]), torch.bfloat16)
        w = _randn(g, (case["k"], case["n"]), torch.float32)
        w8, sw = quant.quantize_fp8_blockwise(w, (128, 128))
        return {"x": x, "w8": w8, "sw": sw}
    if kind == "gqa":
        dt, s, d = _DTYPES[case["dtype"]], case["seq"], case["d"]
        q = _randn(g, (case["batch"], case["heads"], s, d), dt)
        k = _randn(g, (case["batch"], case["kv_heads"], s, d), dt)
        v = _randn(g, (case["batch"], case["kv_heads"], s, d), dt)
        return {"q": q, "k": k, "v": v}
    if kind == "mla_prefill":
        dt, hs = _DTYPES[case["dtype"]], (case["batch"], case["heads"], case["seq"])
        return {"q": _randn(g, hs + (_D_NOPE + _D_ROPE,), dt), "k": _randn(g, hs + (_D_NOPE + _D_ROPE,), dt),
                "v": _randn(g, hs + (_D_V,), dt)}
    if kind == "mla_step":
        b, h, bf = case["batch"], case["heads"], torch.bfloat16
        return {"q_nope": _randn(g, (b, h, _D_NOPE), bf), "q_rope": _randn(g, (b, h, _D_ROPE), bf),
                "kv": _randn(g, (b, case["ctx"], _D_C + _D_ROPE), bf),
                "w_uk": _randn(g, (h, _D_NOPE, _D_C), bf, 1.0 / math.sqrt(_D_NOPE)),
                "w_uv": _randn(g, (h, _D_C, _D_V), bf, 1.0 / math.sqrt(_D_C))}
    dt, b, h, dk, dv = _DTYPES[case["dtype"]], case["batch"], case["heads"], case["dk"], case["dv"]
    hk = case.get("key_heads", h)
    q = torch.randn((b, hk, dk), generator=g, device="cuda")
    k = torch.randn((b, hk, dk), generator=g, device="cuda")
    x = {"q": (q / q.norm(dim=-1, keepdim=True)).to(dt), "k": (k / k.norm(dim=-1, keepdim=True)).to(dt),
         "v": _randn(g, (b, h, dv), dt), "S": _randn(g, (b, h, dk, dv), torch.float32, 0.1)}
    if kind == "gdn":
        x["alpha"] = torch.exp(-torch.nn.functional.softplus(torch.randn((b, h), generator=g, device="cuda")))
        x["beta"] = torch.sigmoid(torch.randn((b, h), generator=g, device="cuda"))
    else:
        x["g"] = (-0.5 * torch.randn((b, h, dk), generator=g, device="cuda").abs()).to(dt)
        x["beta"] = (0.1 + 0.8 * torch.rand((b, h), generator=g, device="cuda")).to(dt)
    return x


def _mla_scale():
    return (_D_NOPE + _D_ROPE) ** -0.5


def prepare(case, seed):
    x = _inputs(case, seed)
    if case["kind"] == "mla_step":
        need = ops.mla_decode_absorbed_workspace_bytes(case["batch"], case["heads"], case["ctx"])
        x["workspace"] = torch.empty(need + 256, dtype=torch.uint8, device="cuda")
    return {"case": case, "x": x}


def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind == "gemm":
        return ops.gemm_bf16(x["a"], x["b"])
    if kind == "fp8_linear":
        x8, sx = ops.quant_fp8_act(x["x"])
        return {"y": ops.gemm_fp8_bs(x8, sx, x["w8"], x["sw"]), "codes": x8, "scales": sx}
    if kind == "gqa":
        return ops.gqa_fwd(x["q"], x["k"], x["v"], causal=case["causal"])
    if kind == "mla_prefill":
        return ops.mla_prefill_fwd(x["q"], x["k"], x["v"], causal=case["causal"])
    if kind == "mla_step":
        return ops.mla_decode_absorbed(x["q_nope"], x["q_rope"], x["kv"], x["w_uk"], x["w_uv"], _mla_scale(),
                                       workspace=x["workspace"])
    if kind == "gdn":
        o, s = ops.gdn_decode(x["q"], x["k"], x["v"], x["alpha"], x["beta"], x["S"], S_out=x["S"])
        return {"o": o, "S": s}
    o, s = ops.kda_decode(x["q"], x["k"], x["v"], x["g"], x["beta"], x["S"], S_out=x["S"])
    return {"o": o, "S": s}


def work(case):
    """Each input read once, each output written once; 2 flops per
    multiply-add of the products (the masked half of causal scores left out)."""
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "fp8_linear":
        m, n, k = case["m"], case["n"], case["k"]
        quantise = 2 * m * k + m * k + 4 * m * (k // 128)
        return {"bytes": quantise + k * n + 4 * (k // 128) * -(-n // 128) + 2 * m * n, "flops": 2 * m * n * k}
    if kind in ("gqa", "mla_prefill"):
        b, h, s = case["batch"], case["heads"], case["seq"]
        dq, dv = (case["d"], case["d"]) if kind == "gqa" else (_D_NOPE + _D_ROPE, _D_V)
        kv = case.get("kv_heads", h)
        pairs = s * (s + 1) // 2 if case["causal"] else s * s
        return {"bytes": 2 * b * s * (h + kv) * (dq + dv), "flops": 2 * b * h * pairs * (dq + dv)}
    if kind == "mla_step":
        b, h, t = case["batch"], case["heads"], case["ctx"]
        weights = h * _D_C * (_D_NOPE + _D_V)
        io = b * h * (_D_NOPE + _D_ROPE + _D_V)
        return {"bytes": 2 * (b * t * (_D_C + _D_ROPE) + weights + io),
                "flops": 2 * b * h * (t * (2 * _D_C + _D_ROPE) + _D_C * (_D_NOPE + _D_V))}
    b, h, dk, dv = case["batch"], case["heads"], case["dk"], case["dv"]
    hk = case.get("key_heads", h)
    gates = 8 * b * h if kind == "gdn" else 2 * b * h * (dk + 1)
    return {"bytes": 8 * b * h * dk * dv + 4 * b * hk * dk + 4 * b * h * dv + gates, "flops": 6 * b * h * dk * dv}


def tolerance(case):
    """About four times the measured 2-norm distance from the 64-bit result
    (bf16 outputs 1.7e-3 from the output's own rounding, more where inner
    values are rounded to 16 bits as well; f16 outputs 2.1e-4)."""
    f16 = case.get("dtype") == "f16"
    if case["kind"] in ("gemm", "fp8_linear"):
        return {"rel": 7e-3}
    if case["kind"] in ("gqa", "mla_prefill"):
        return {"rel": 1.5e-3 if f16 else 1e-2}
    if case["kind"] == "mla_step":
        return {"rel": 1.6e-2}
    return {"rel": 1e-3 if f16 else 7e-3}


def _attention(q, k, v, scale, causal):
    """softmax(scale q k^T) v in float64, one (batch, head) at a time."""
    b, h, s, _ = q.shape
    group = h // k.shape[1]
    out = torch.empty((b, h, s, v.shape[3]), dtype=torch.float64, device=q.device)
    for i in range(b):
        for j in range(h):
            kk, vv = k[i, j // group].double(), v[i, j // group].double()
            for r0 in range(0, s, 2048):
                r1 = min(s, r0 + 2048)
                score = (q[i, j, r0:r1].double() @ kk.t().contiguous()) * scale
                if causal:
                    rows = torch.arange(r0, r1, device=q.device)[:, None]
                    score.masked_fill_(torch.arange(s, device=q.device)[None, :] > rows, -math.inf)
                out[i, j, r0:r1] = torch.softmax(score, dim=-1) @ vv
    return out


def exact(case, seed):
    """What run() returns for these inputs, in 64 bits, from plain torch.  The
    fp8 codes have no such value, and the product takes the codes of the
    stated recipe (scale = amax / 448 in fp32, round to nearest even)."""
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "gemm":
        return x["a"].double() @ x["b"].double()
    if kind == "fp8_linear":
        m, k, n = case["m"], case["k"], case["n"]
        xb = x["x"].float().reshape(m, k // 128, 128)
        amax = xb.abs().amax(-1)
        # scale and quotient rounded to fp32 from 64 bits (a device division by a constant multiplies by its reciprocal)
        sx = torch.where(amax > 0, (amax.double() / 448.0).float(), torch.ones_like(amax))
        codes = (xb.double() / sx.double()[..., None]).float().clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
        xd = (codes.double() * sx.double()[..., None]).reshape(m, k)
        sw = x["sw"].double().repeat_interleave(128, 0).repeat_interleave(128, 1)[:k, :n]
        return {"y": xd @ (x["w8"].double() * sw), "codes": None, "scales": sx.double()}
    if kind == "gqa":
        return _attention(x["q"], x["k"], x["v"], 1.0 / math.sqrt(case["d"]), case["causal"])
    if kind == "mla_prefill":
        return _attention(x["q"], x["k"], x["v"], _mla_scale(), case["causal"])
    if kind == "mla_step":
        b, h = case["batch"], case["heads"]
        wk, wv = x["w_uk"].double(), x["w_uv"].double()
        q = torch.stack([x["q_nope"][:, j].double() @ wk[j] for j in range(h)], dim=1)
        q = torch.cat([q, x["q_rope"].double()], dim=-1)
        lat = []
        for i in range(b):
            kv = x["kv"][i].double()
            lat.append(torch.softmax((q[i] @ kv.t().contiguous()) * _mla_scale(), dim=-1) @ kv[:, :_D_C])
        lat = torch.stack(lat)
        return torch.stack([lat[:, j] @ wv[j] for j in range(h)], dim=1)
    group = case["heads"] // case.get("key_heads", case["heads"])
    q, k = (x[n].double().repeat_interleave(group, 1) for n in ("q", "k"))
    v, s = x["v"].double(), x["S"].double()
    if kind == "gdn":
        s = s * x["alpha"].double()[..., None, None]
    else:
        s = s * torch.exp(x["g"].double())[..., None]
    r = v - (k[..., None] * s).sum(-2)
    s = s + x["beta"].double()[..., None, None] * k[..., None] * r[..., None, :]
    return {"o": (q[..., None] * s).sum(-2), "S": s}
