"""Benchmark of the quant-inference kernel path on one MI355X.

Headline (the `value` of the JSON line): the fused causal GQA forward at
BASELINE configs[1] — B=1, Hq=32, Hkv=8, S=4096, D=128, bf16, N(0,1)
inputs, scale 1/sqrt(128) — in algorithmic TFLOP/s (causal work
2*B*Hq*D*S*(S+1)).  A "step" is one forward pass over that batch with the
inputs already resident in HBM.

Every other BASELINE config is measured the same way and reported under
"others" with its own `roofline` and `cpu_baseline` blocks:
  gemm_bf16_1024   bf16 GEMM 1024^3 (configs[0], U[-1,1] inputs)
  gemm_bf16_8192   bf16 GEMM 8192^3 (the north star's GEMM target size)
  gemm_fp8_8192    fp8 1x128/128x128 block-scaled GEMM 8192^3
  mla_decode       MLA absorbed decode B32 H128 T4096 576/512
  gdn_decode       GDN decode B64 Hk16 Hv32 d128
and the widened rows with theirs (absorbed MLA step, KDA decode, fp8
activation quantiser on its first 256 rows for the CPU, MLA prefill on 16
of 128 heads for the CPU), plus hipblaslt_8192: the
vendor library's bf16 and per-tensor fp8 GEMMs at 8192^3 on the same GPU,
a labelled reference line.

Timing: W untimed warm-up launches, then exactly K launches between
torch.cuda.synchronize() calls with one HIP event pair on the launching
stream.  The headline launches are issued eagerly from Python (each
~150 us kernel hides the host cost); the other kernels' K launches are
captured once into a HIP graph and replayed, so few-microsecond kernels
are timed on the device, not as Python launch overhead.  Before each
case's warm-up (for graph-timed cases, before the untimed replay) the GPU
runs --settle-ms (default 300) of a plain device GEMM, so the timed steps
start at load clocks rather than at the clocks of an idle GPU; the JSON
line reports it under "settle".

Rotated inputs (the HBM-bound cases mla_decode, gdn_decode, kda_decode,
quant_fp8_act, mla_absorbed): MI355X has a 256 MB Infinity Cache (MALL)
in front of HBM, and these working sets (67-270 MB) fit in it or sit at
its edge, so replaying one input set measures partly cache bandwidth.
Each such case is therefore also timed with R copies of its inputs (and
outputs), step j of the graph using copy j % R, so that between two
touches of one copy more than 256 MB of other copies stream through.
The case's `value` and `roofline` are the rotated figures; the same-buffer
figure is kept as `hot`.

Parity gate (the reference's rule: a kernel that fails its correctness
check reports no numbers, analysis/wave15-attention-architecture/reference/
README.md:47-58): every case's GPU output is compared against the CPU
oracle, on the whole workload in the CPU leg, or with --no-cpu-baseline on
a bounded sample (listed under `parity.check`).  Bounds: normwise
max|got-ref|/max|ref| <= 2e-2 for bf16/fp8 outputs, <= 1e-3 for the fp32
GDN/KDA state, codes and scales bit-exact for the fp8 quantiser.  If any
case misses its bound, no JSON line is printed and the exit status is 3.

CPU baseline (BASELINE.md's plan): this repository's CPU oracle (the
restatement of the reference's CPU implementation, "port") on the same
seeded inputs, torch fp32 on the host's cores, 1 warm-up + 3 timed runs,
median; the GPU output is compared against it on the same sample.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu-baseline] [--settle-ms MS]
       [--only NAME[,NAME...]] [--only-headline] [--calibrate-copy]
Prints exactly one JSON line on stdout (progress goes to stderr).
"""
from __future__ import annotations

import argparse
import importlib
import json
import os
import platform
import statistics
import sys
import time
from pathlib import Path

REPO_ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(REPO_ROOT))

METRIC = "TFLOPS & %MFMA peak (GEMM, GQA fwd); GB/s & %HBM peak (MLA/GDN decode)"
TRAFFIC_FILE = REPO_ROOT / "profiles" / "hbm_traffic.json"


def log(msg: str) -> None:
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


# ---------------------------------------------------------------- timing
# Device settle.  An MI355X coming out of idle runs at low clocks for a few
# hundred milliseconds of load (measured: the headline kernel takes 151 us
# per launch right after idle, 141 us after 100 ms of load and 127 us after
# 300 ms).  Before each case's warm-up steps the GPU is therefore kept busy
# for SETTLE_MS with a plain device GEMM (torch.matmul, 8192^2 bf16; not
# the measured kernel), so that the warm-up and timed steps run at load
# clocks.  The W warm-up and K timed steps themselves are unchanged.
SETTLE_MS = 300.0
_SETTLE: dict = {}


def settle() -> None:
    import torch

    if SETTLE_MS <= 0:
        return
    if "a" not in _SETTLE:
        g = torch.Generator(device="cuda").manual_seed(1)
        _SETTLE["a"] = torch.randn(8192, 8192, device="cuda", generator=g).to(torch.bfloat16)
        _SETTLE["c"] = torch.empty_like(_SETTLE["a"])
    a, c = _SETTLE["a"], _SETTLE["c"]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    while (time.perf_counter() - t0) * 1e3 < SETTLE_MS:
        for _ in range(8):
            torch.matmul(a, a, out=c)
        torch.cuda.synchronize()


def time_eager(fn, steps: int, warmup: int):
    """`warmup` calls, then exactly `steps` back-to-back calls bracketed by
    synchronize() and one event pair on the current stream.  Returns (event
    ms per launch, wall ms per step)."""
    import torch

    settle()
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    for _ in range(steps):
        fn()
    end.record()
    torch.cuda.synchronize()
    wall_ms = (time.perf_counter() - t0) * 1e3 / steps
    return start.elapsed_time(end) / steps, wall_ms


def time_graph(fn, steps: int, warmup: int):
    """`warmup` eager calls, then `steps` calls captured into one HIP graph;
    the graph is replayed once untimed and once timed (one event pair on
    the replay stream).  The operators launch kernels only (no memset or
    copy nodes), so the replayed graph is the same work as the eager calls."""
    import torch

    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(steps):
            fn()
    torch.cuda.synchronize()
    settle()
    g.replay()
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    g.replay()
    end.record()
    torch.cuda.synchronize()
    wall_ms = (time.perf_counter() - t0) * 1e3 / steps
    ms = start.elapsed_time(end) / steps
    del g
    return ms, wall_ms


def time_graph_rotated(fns, steps: int, warmup: int):
    """As time_graph, with step j of the captured graph calling fns[j % R]
    (R input/output copies), so each copy is touched once every R steps."""
    import torch

    r = len(fns)
    for j in range(max(warmup, r)):
        fns[j % r]()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for f in fns:
            f()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for j in range(steps):
            fns[j % r]()
    torch.cuda.synchronize()
    settle()
    g.replay()
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    g.replay()
    end.record()
    torch.cuda.synchronize()
    wall_ms = (time.perf_counter() - t0) * 1e3 / steps
    ms = start.elapsed_time(end) / steps
    del g
    return ms, wall_ms


MALL_BYTES = 256 << 20  # MI355X Infinity Cache


def rotation_count(bytes_per_set: int) -> int:
    """Copies R such that the other R-1 copies streamed between two touches
    of one copy exceed the Infinity Cache at least 1.5 times over."""
    r = 2
    while (r - 1) * bytes_per_set < 1.5 * MALL_BYTES:
        r += 1
    return r


def rotate(rec: dict, fns, set_bytes: int, work: float, c, wl: str, kernel: str) -> None:
    """Time the case again over rotated copies; the rotated figure becomes the
    case's value and roofline, the same-buffer one moves to rec["hot"]."""
    ms, wall = time_graph_rotated(fns, c.steps, c.warmup)
    rec["hot"] = {"value": rec["value"], "mean_ms": rec["mean_ms"], "wall_ms": rec["wall_ms"],
                  "roofline": rec["roofline"],
                  "note": "one input/output set replayed every step (working set can sit in the 256 MB MALL)"}
    rec["value"] = c.F.gbps(work, ms)
    rec["mean_ms"], rec["wall_ms"] = ms, wall
    rec["roofline"] = roofline("hbm", work, ms, c.F.PEAK_HBM_GBPS, "GB/s", wl, kernel)
    rec["rotated"] = {"sets": len(fns), "bytes_per_set": set_bytes,
                      "bytes_between_reuse": (len(fns) - 1) * set_bytes,
                      "note": f"step j reads and writes copy j % {len(fns)}; value and roofline are this figure"}


# ---------------------------------------------------------------- parity gate
OUT_BOUND = 2e-2     # normwise, bf16/fp8 outputs
STATE_BOUND = 1e-3   # normwise, fp32 GDN/KDA state


def parity_record(c, rec: dict, sample_check) -> None:
    """rec["parity"]: the CPU leg's whole-workload comparison when it ran,
    else `sample_check()` -> dict of measured errors on a bounded sample."""
    leg = rec.get("cpu_baseline")
    if leg is not None:
        par = {"check": "cpu_baseline sample: " + leg["sample"].split(";")[0]}
        if "parity_normwise_on_sample" in leg:
            par["output_normwise"] = leg["parity_normwise_on_sample"]
        if "parity_normwise_state_on_sample" in leg:
            par["state_normwise"] = leg["parity_normwise_state_on_sample"]
        if "codes_bit_exact_on_sample" in leg:
            par["bit_exact"] = bool(leg["codes_bit_exact_on_sample"] and leg["scales_bit_exact_on_sample"])
    else:
        par = sample_check()
    par["bounds"] = {"output_normwise": OUT_BOUND, "state_normwise": STATE_BOUND}
    rec["parity"] = par


def parity_failures(results: dict) -> list[str]:
    """Cases whose GPU output misses its bound (or was never checked)."""
    bad = []
    for name, rec in results.items():
        par = rec.get("parity")
        if par is None:
            if name not in REFERENCE_LINES:
                bad.append(f"{name}: no parity check")
            continue
        e = par.get("output_normwise")
        if e is not None and not e <= OUT_BOUND:
            bad.append(f"{name}: output normwise {e:.3e} > {OUT_BOUND}")
        e = par.get("state_normwise")
        if e is not None and not e <= STATE_BOUND:
            bad.append(f"{name}: state normwise {e:.3e} > {STATE_BOUND}")
        if par.get("bit_exact") is False:
            bad.append(f"{name}: quantised codes/scales not bit-exact")
        if all(par.get(k) is None for k in ("output_normwise", "state_normwise", "bit_exact")):
            bad.append(f"{name}: parity check measured nothing")
    return bad


def _nw(got, ref) -> float:
    from oracle.metrics import normwise_rel_err

    return float(normwise_rel_err(got, ref))


# ---------------------------------------------------------------- CPU leg
def cpu_info() -> str:
    try:
        for line in Path("/proc/cpuinfo").read_text().splitlines():
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or "unknown"


def host_threads() -> int:
    """The cores this process may use: its CPU affinity, capped by
    OMP_NUM_THREADS when that is set (the GPU box gives a job a share of the
    host's cores and says so there)."""
    try:
        n = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        n = os.cpu_count() or 1
    env = os.environ.get("OMP_NUM_THREADS")
    if env and env.isdigit() and int(env) > 0:
        n = min(n, int(env))
    return max(1, n)


def cpu_leg(run, work: float, unit: str, sample: str, got=None, ref_of=None) -> dict:
    """Time `run()` (the oracle on the sample): 1 warm-up + 3 timed runs,
    median.  `work` is the algorithmic FLOPs (unit TFLOPS) or bytes (GB/s)
    of one run.  With `got`/`ref_of`, the GPU output is compared against
    the oracle's on the same sample (normwise max|got-ref|/max|ref|)."""
    import torch

    from oracle.metrics import normwise_rel_err

    torch.set_num_threads(host_threads())
    threads = torch.get_num_threads()
    ref = run()  # warm-up
    times = []
    for _ in range(3):
        t0 = time.perf_counter()
        ref = run()
        times.append(time.perf_counter() - t0)
    med = statistics.median(times)
    value = work / med / (1e12 if unit == "TFLOPS" else 1e9)
    out = {
        "value": value,
        "unit": unit,
        "cores": threads,
        "kind": "port",
        "sample": f"{sample}; fp32 torch CPU oracle, 1 warm-up + 3 runs, median {med:.3f} s "
                  f"(runs {', '.join(f'{t:.3f}' for t in times)} s), {threads} threads ({cpu_info()})",
        "median_s": med,
    }
    if got is not None:
        r = ref_of(ref) if ref_of else ref
        out["parity_normwise_on_sample"] = normwise_rel_err(got, r)
    return out


# ---------------------------------------------------------------- traffic
def load_traffic(workload: str):
    """HBM bytes per launch of a workload's kernel(s) from the committed
    rocprofv3 FETCH_SIZE / WRITE_SIZE summary (calibrated against a device
    copy of known size), or None when the summary does not cover it."""
    try:
        d = json.loads(TRAFFIC_FILE.read_text())
    except (OSError, ValueError):
        return None
    e = d.get("workloads", {}).get(workload)
    return None if e is None else e.get("hbm_bytes_per_launch")


def roofline(bound: str, work: float, ms: float, peak: float, unit: str, workload: str, kernel: str) -> dict:
    achieved = work / (ms * 1e-3) / (1e12 if unit == "TFLOP/s" else 1e9)
    return {
        "bound": bound,
        "achieved": round(achieved, 3),
        "peak": peak,
        "unit": unit,
        "frac": round(achieved / peak, 5),
        "traffic": load_traffic(workload),
        "kernel": kernel,
        "launch_mean_ms": round(ms, 6),
        "algorithmic_work_per_launch": work,
    }


# ---------------------------------------------------------------- cases
class Ctx:
    def __init__(self, pkg, ops, steps, warmup, cpu):
        self.pkg, self.ops, self.steps, self.warmup, self.cpu = pkg, ops, steps, warmup, cpu
        self.S, self.F, self.I = pkg.shapes, pkg.flops, pkg.inputs


def case_gqa(c: Ctx) -> dict:
    import torch

    shape = c.S.GQA_BASELINE
    q, k, v = c.I.gqa_inputs(shape)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    out = torch.empty_like(qd)
    ms, wall = time_eager(lambda: c.ops.gqa_fwd(qd, kd, vd, causal=True, out=out), c.steps, c.warmup)
    flops = c.F.gqa_causal_flops(shape)
    wl = (f"gqa_fwd causal B{shape.batch} Hq{shape.n_q} Hkv{shape.n_kv} S{shape.seq} D{shape.d_head} bf16")
    rec = {
        "workload": wl, "unit": "TFLOPS", "mean_ms": ms, "wall_ms": wall, "flops": flops,
        "value": c.F.tflops(flops, ms),
        "tflops_reference_convention": c.F.tflops(c.F.gqa_attention_flops(shape), ms),
        "roofline": roofline("mfma", flops, ms, c.F.PEAK_BF16_TFLOPS, "TFLOP/s", wl,
                             "gqa_fwd_kernel<128, 128, BF16, true, 1, 8, 1>"),
        "shape": shape,
    }
    if c.cpu:
        from oracle import gqa as ogqa

        got = out.cpu()
        rec["cpu_baseline"] = cpu_leg(lambda: ogqa.gqa_naive(q, k, v, causal=True), flops, "TFLOPS",
                                      f"the whole workload (all {shape.n_q} query heads, causal S={shape.seq})",
                                      got=got)

    def sample():
        from oracle import gqa as ogqa

        hs = [0, 13, shape.n_q - 1]
        return {"check": f"query heads {hs} of {shape.n_q}, full causal S={shape.seq}",
                "output_normwise": _nw(out.cpu()[:, hs], ogqa.gqa_naive(q, k, v, causal=True, heads=hs)[:, hs])}

    parity_record(c, rec, sample)
    return rec


def _gemm_bf16(c: Ctx, shape, name: str) -> dict:
    import torch

    a, b = c.I.gemm_inputs(shape)
    ad, bd = a.cuda(), b.cuda()
    out = torch.empty((shape.m, shape.n), dtype=torch.bfloat16, device="cuda")
    ms, wall = time_graph(lambda: c.ops.gemm_bf16(ad, bd, out=out), c.steps, c.warmup)
    flops = c.F.gemm_flops(shape)
    wl = f"gemm_bf16 M{shape.m} N{shape.n} K{shape.k} U[-1,1]"
    kernel = ("gemm_bf16_dma16s_kernel (256x256 tiles, A and B rings)" if shape.m >= 4096
              else "gemm_bf16_dma64_kernel (64x64 tiles)")
    rec = {"workload": wl, "unit": "TFLOPS", "mean_ms": ms, "wall_ms": wall, "value": c.F.tflops(flops, ms),
           "roofline": roofline("mfma", flops, ms, c.F.PEAK_BF16_TFLOPS, "TFLOP/s", wl, kernel)}
    if c.cpu:
        from oracle import gemm as ogemm

        got = out.cpu()
        rec["cpu_baseline"] = cpu_leg(lambda: ogemm.gemm_ref(a, b), flops, "TFLOPS",
                                      f"the whole {shape.m}x{shape.n}x{shape.k} product", got=got)

    def sample():
        from oracle import gemm as ogemm

        rows = sorted(set(list(range(32)) + list(range(shape.m - 32, shape.m))))
        return {"check": f"rows {{0..31, {shape.m - 32}..{shape.m - 1}}} of C, every column",
                "output_normwise": _nw(out.cpu()[rows], ogemm.gemm_ref(a[rows], b))}

    parity_record(c, rec, sample)
    del ad, bd, out
    return rec


def case_gemm_bf16_1024(c: Ctx) -> dict:
    return _gemm_bf16(c, c.S.GEMM_PARITY, "gemm_bf16_1024")


def case_gemm_bf16_8192(c: Ctx) -> dict:
    return _gemm_bf16(c, c.S.GEMM_TARGET, "gemm_bf16_8192")


def case_gemm_fp8_8192(c: Ctx) -> dict:
    import torch

    shape = c.S.FP8_TARGET
    a8, sa, b8, sb = c.I.fp8_gemm_inputs(shape)
    a8d, sad, b8d, sbd = a8.cuda(), sa.cuda(), b8.cuda(), sb.cuda()
    out = torch.empty((shape.m, shape.n), dtype=torch.bfloat16, device="cuda")
    ms, wall = time_graph(lambda: c.ops.gemm_fp8_bs(a8d, sad, b8d, sbd, out=out), c.steps, c.warmup)
    flops = c.F.gemm_flops(shape)
    wl = f"gemm_fp8_bs M{shape.m} N{shape.n} K{shape.k} e4m3 1x128/128x128 scales"
    rec = {"workload": wl, "unit": "TFLOPS", "mean_ms": ms, "wall_ms": wall, "value": c.F.tflops(flops, ms),
           "bytes_per_launch": c.F.gemm_fp8_bytes(shape),
           "roofline": roofline("mfma", flops, ms, c.F.PEAK_FP8_TFLOPS, "TFLOP/s", wl, "gemm_fp8_bs_kernel")}
    if c.cpu:
        from oracle import fp8 as ofp8

        got = out.cpu()
        rec["cpu_baseline"] = cpu_leg(lambda: ofp8.gemm_fp8_bs_ref_torch(a8, sa, b8, sb), flops, "TFLOPS",
                                      f"the whole {shape.m}^3 product of the dequantised operands", got=got)

    def sample():
        from oracle import fp8 as ofp8

        rows = list(range(32)) + list(range(shape.m - 32, shape.m))
        return {"check": f"rows {{0..31, {shape.m - 32}..{shape.m - 1}}} of C, every column",
                "output_normwise": _nw(out.cpu()[rows], ofp8.gemm_fp8_bs_ref_torch(a8[rows], sa[rows], b8, sb))}

    parity_record(c, rec, sample)
    del a8d, sad, b8d, sbd, out
    return rec


def case_hipblaslt_8192(c: Ctx) -> dict:
    """The vendor library beside this repo's GEMMs, same box and run: torch.matmul
    (hipBLASLt) on the bf16 8192^3 inputs of gemm_bf16_8192 and on the
    1024^3 ones of gemm_bf16_1024, and
    torch._scaled_mm (hipBLASLt fp8, one per-tensor scale each, column-major
    B) at 8192^3.  A reference line, not this repository's kernels: the
    library has no 1x128/128x128 block-scaled fp8 GEMM to compare against."""
    import torch

    shape = c.S.GEMM_TARGET
    a, b = c.I.gemm_inputs(shape)
    ad, bd = a.cuda(), b.cuda()
    out = torch.empty((shape.m, shape.n), dtype=torch.bfloat16, device="cuda")
    ms_bf16, _ = time_graph(lambda: torch.matmul(ad, bd, out=out), c.steps, c.warmup)
    del ad, bd
    # the same at configs[0] (1024^3), beside gemm_bf16_1024
    s0 = c.S.GEMM_PARITY
    a0, b0 = (t.cuda() for t in c.I.gemm_inputs(s0))
    out0 = torch.empty((s0.m, s0.n), dtype=torch.bfloat16, device="cuda")
    ms_1024, _ = time_graph(lambda: torch.matmul(a0, b0, out=out0), c.steps, c.warmup)
    del a0, b0, out0
    g = torch.Generator().manual_seed(c.I.SEED)
    a8 = torch.randn((shape.m, shape.k), generator=g).to(torch.float8_e4m3fn).cuda()
    b8 = torch.randn((shape.n, shape.k), generator=g).to(torch.float8_e4m3fn).cuda().t()  # column-major [K, N]
    one = torch.ones((), dtype=torch.float32, device="cuda")
    ms_fp8, _ = time_graph(lambda: torch._scaled_mm(a8, b8, scale_a=one, scale_b=one, out_dtype=torch.bfloat16),
                           c.steps, c.warmup)
    fl = c.F.gemm_flops(shape)
    return {"workload": "hipBLASLt reference: bf16 torch.matmul and fp8 per-tensor torch._scaled_mm, 8192^3",
            "unit": "TFLOPS", "mean_ms": ms_bf16, "wall_ms": ms_bf16, "value": c.F.tflops(fl, ms_bf16),
            "bf16_tflops": c.F.tflops(fl, ms_bf16), "fp8_per_tensor_tflops": c.F.tflops(fl, ms_fp8),
            "fp8_per_tensor_mean_ms": ms_fp8,
            "bf16_1024_tflops": c.F.tflops(c.F.gemm_flops(s0), ms_1024), "bf16_1024_mean_ms": ms_1024,
            "note": "vendor library on the same GPU for comparison; not part of this repository's path"}


def case_hbm_copy(c: Ctx) -> dict:
    """A plain device copy (torch's copy kernel, 128 MiB read + 128 MiB
    written per step) over rotated buffers, timed like the HBM-bound cases:
    the streaming bandwidth this GPU delivers with caches defeated, as a
    reference line for the decode kernels' rotated figures."""
    import torch

    n = 128 << 20
    per_set = 2 * n
    sets = [(torch.ones(n, dtype=torch.uint8, device="cuda"), torch.empty(n, dtype=torch.uint8, device="cuda"))
            for _ in range(rotation_count(per_set))]
    ms, wall = time_graph_rotated([lambda t=t: t[1].copy_(t[0]) for t in sets], c.steps, c.warmup)
    del sets
    return {"workload": f"device copy {n >> 20} MiB -> {n >> 20} MiB, rotated buffers", "unit": "GB/s",
            "mean_ms": ms, "wall_ms": wall, "value": c.F.gbps(per_set, ms),
            "frac_hbm_peak": c.F.gbps(per_set, ms) / c.F.PEAK_HBM_GBPS,
            "note": "reference line: torch's device copy, not this repository's path"}


def case_mla_decode(c: Ctx) -> dict:
    import torch

    shape = c.S.MLA_BASELINE
    q, kv = c.I.mla_inputs(shape)
    qd, kvd = q.cuda(), kv.cuda()
    o = torch.empty((shape.batch, shape.n_h, shape.d_latent), dtype=torch.bfloat16, device="cuda")
    ws = torch.empty(max(1, c.ops.mla_decode_workspace_bytes(shape.batch, shape.n_h, shape.ctx)),
                     dtype=torch.uint8, device="cuda")
    ms, wall = time_graph(lambda: c.ops.mla_decode(qd, kvd, shape.scale, out=o, workspace=ws), c.steps, c.warmup)
    nb, fl = c.F.mla_decode_bytes(shape), c.F.mla_decode_flops(shape)
    wl = f"mla_decode absorbed B{shape.batch} H{shape.n_h} T{shape.ctx} 576/512 bf16"
    kern = "mla_decode_kernel + mla_combine_kernel (one call)"
    rec = {"workload": wl, "unit": "GB/s", "mean_ms": ms, "wall_ms": wall, "value": c.F.gbps(nb, ms),
           "tflops": c.F.tflops(fl, ms), "flops": fl,
           "roofline": roofline("hbm", nb, ms, c.F.PEAK_HBM_GBPS, "GB/s", wl, kern)}
    set_b = (kvd.numel() + qd.numel() + o.numel()) * 2
    sets = [(qd, kvd, o)] + [(qd.clone(), kvd.clone(), torch.empty_like(o))
                             for _ in range(rotation_count(set_b) - 1)]
    rotate(rec, [lambda t=t: c.ops.mla_decode(t[0], t[1], shape.scale, out=t[2], workspace=ws) for t in sets],
           set_b, nb, c, wl, kern)
    rec["tflops"] = c.F.tflops(fl, rec["mean_ms"])
    o = sets[(c.steps - 1) % len(sets)][2]  # the last step's output
    del sets
    if c.cpu:
        from oracle import mla as omla

        got = o.cpu()
        rec["cpu_baseline"] = cpu_leg(lambda: omla.mla_decode_ref(q, kv, shape.scale), nb, "GB/s",
                                      f"the whole workload ({shape.batch} sequences x {shape.n_h} heads, "
                                      f"T={shape.ctx})", got=got)

    def sample():
        from oracle import mla as omla

        bs = [0, shape.batch - 1]
        return {"check": f"sequences {bs} of {shape.batch}, all heads, T={shape.ctx}",
                "output_normwise": _nw(o.cpu()[bs], omla.mla_decode_ref(q, kv, shape.scale, batches=bs)[bs])}

    parity_record(c, rec, sample)
    del qd, kvd, o, ws
    return rec


def case_gdn_decode(c: Ctx) -> dict:
    import torch

    shape = c.S.GDN_BASELINE
    x = c.I.gdn_inputs(shape)
    xd = {n: t.cuda() for n, t in x.items()}
    so = torch.empty_like(xd["S_in"])
    od = torch.empty((shape.batch, shape.n_heads, shape.d_v), dtype=torch.bfloat16, device="cuda")
    ms, wall = time_graph(lambda: c.ops.gdn_decode(xd["q"], xd["k"], xd["v"], xd["alpha"], xd["beta"], xd["S_in"],
                                                   S_out=so, o=od), c.steps, c.warmup)
    nb = c.F.gdn_decode_bytes(shape)
    wl = (f"gdn_decode B{shape.batch} Hk{shape.hk} Hv{shape.n_heads} dk{shape.d_k} dv{shape.d_v} "
          f"bf16 q/k/v, fp32 state")
    rec = {"workload": wl, "unit": "GB/s", "mean_ms": ms, "wall_ms": wall, "value": c.F.gbps(nb, ms),
           "roofline": roofline("hbm", nb, ms, c.F.PEAK_HBM_GBPS, "GB/s", wl, "gdn_decode_kernel")}
    sets = [(xd, so, od)] + [({n: t.clone() for n, t in xd.items()}, torch.empty_like(so), torch.empty_like(od))
                             for _ in range(rotation_count(nb) - 1)]
    rotate(rec, [lambda t=t: c.ops.gdn_decode(t[0]["q"], t[0]["k"], t[0]["v"], t[0]["alpha"], t[0]["beta"],
                                              t[0]["S_in"], S_out=t[1], o=t[2]) for t in sets],
           nb, nb, c, wl, "gdn_decode_kernel")
    _, so, od = sets[(c.steps - 1) % len(sets)]
    del sets
    if c.cpu:
        from oracle import gdn as ogdn
        from oracle.metrics import normwise_rel_err

        o_gpu, s_gpu = od.cpu(), so.cpu()
        leg = cpu_leg(lambda: ogdn.gdn_decode_ref(**x), nb, "GB/s",
                      f"the whole workload ({shape.batch}x{shape.n_heads} value heads, "
                      f"{shape.d_k}x{shape.d_v} fp32 state)", got=o_gpu, ref_of=lambda r: r[0])
        ro, rs = ogdn.gdn_decode_ref(**x)
        leg["parity_normwise_state_on_sample"] = normwise_rel_err(s_gpu, rs)
        rec["cpu_baseline"] = leg

    def sample():
        from oracle import gdn as ogdn

        ro, rs = ogdn.gdn_decode_ref(**x)
        return {"check": "the whole workload (output and state)", "output_normwise": _nw(od.cpu(), ro),
                "state_normwise": _nw(so.cpu(), rs)}

    parity_record(c, rec, sample)
    del xd, so, od
    return rec


def case_mla_absorbed(c: Ctx) -> dict:
    import torch

    shape = c.S.MLA_BASELINE
    q, kv = c.I.mla_inputs(shape)
    kvd = kv.cuda()
    xh = c.I.mla_projection_inputs(shape)
    x = {n: t.cuda() for n, t in xh.items()}
    od = torch.empty((shape.batch, shape.n_h, 128), dtype=torch.bfloat16, device="cuda")
    wsa = torch.empty(c.ops.mla_decode_absorbed_workspace_bytes(shape.batch, shape.n_h, shape.ctx) + 256,
                      dtype=torch.uint8, device="cuda")
    ms, wall = time_graph(lambda: c.ops.mla_decode_absorbed(x["q_nope"], x["q_rope"], kvd, x["w_uk"], x["w_uv"],
                                                            shape.scale, out=od, workspace=wsa),
                          c.steps, c.warmup)
    # cache + both weights + q_nope/q_rope read once, O written once
    nb = kv.numel() * 2 + sum(x[n].numel() * 2 for n in ("w_uk", "w_uv", "q_nope", "q_rope")) + od.numel() * 2
    wl = f"mla_decode_absorbed step B{shape.batch} H{shape.n_h} T{shape.ctx} d_nope128 d_v128"
    kern = "mla_decode_kernel (+ two batched bf16 GEMMs and mla_combine_kernel, one call)"
    rec = {"workload": wl, "unit": "GB/s", "mean_ms": ms, "wall_ms": wall, "value": c.F.gbps(nb, ms),
           "roofline": roofline("hbm", nb, ms, c.F.PEAK_HBM_GBPS, "GB/s", wl, kern),
           "note": "one mx_mla_decode_absorbed call: q_nope W_UK, latent decode + combine, o_lat W_UV; "
                   "bytes: cache, weights, q_nope/q_rope in, O out"}
    sets = [(x, kvd, od)] + [({n: t.clone() for n, t in x.items()}, kvd.clone(), torch.empty_like(od))
                             for _ in range(rotation_count(nb) - 1)]
    rotate(rec, [lambda t=t: c.ops.mla_decode_absorbed(t[0]["q_nope"], t[0]["q_rope"], t[1], t[0]["w_uk"],
                                                       t[0]["w_uv"], shape.scale, out=t[2], workspace=wsa)
                 for t in sets], nb, nb, c, wl, kern)
    od = sets[(c.steps - 1) % len(sets)][2]
    del sets
    if c.cpu:
        from oracle import mla as omla

        got = od.cpu()
        rec["cpu_baseline"] = cpu_leg(lambda: omla.mla_absorbed_ref(xh["q_nope"], xh["q_rope"], kv, xh["w_uk"],
                                                                    xh["w_uv"], shape.scale), nb, "GB/s",
                                      f"the whole workload ({shape.batch} sequences x {shape.n_h} heads, "
                                      f"T={shape.ctx}, both projections)", got=got)

    def sample():
        from oracle import mla as omla

        r = omla.mla_absorbed_ref(xh["q_nope"][:2], xh["q_rope"][:2], kv[:2], xh["w_uk"], xh["w_uv"], shape.scale)
        return {"check": f"sequences [0, 1] of {shape.batch}, all heads, both projections",
                "output_normwise": _nw(od.cpu()[:2], r)}

    parity_record(c, rec, sample)
    del kvd, x, od, wsa
    return rec


def case_kda_decode(c: Ctx) -> dict:
    import torch

    shape = c.S.KDA_LARGE
    xh = c.I.kda_inputs(shape)
    x = {n: t.cuda() for n, t in xh.items()}
    so = torch.empty_like(x["S_in"])
    od = torch.empty((shape.batch, shape.n_heads, shape.d_v), dtype=torch.float16, device="cuda")
    ms, wall = time_graph(lambda: c.ops.kda_decode(x["q"], x["k"], x["v"], x["g"], x["beta"], x["S_in"],
                                                   S_out=so, o=od), c.steps, c.warmup)
    nb = c.F.kda_decode_bytes(shape)
    wl = f"kda_decode B{shape.batch} H{shape.n_heads} d{shape.d_k} f16"
    rec = {"workload": wl, "unit": "GB/s", "mean_ms": ms, "wall_ms": wall, "value": c.F.gbps(nb, ms),
           "roofline": roofline("hbm", nb, ms, c.F.PEAK_HBM_GBPS, "GB/s", wl, "gdn_decode_kernel (KDA gate)")}
    sets = [(x, so, od)] + [({n: t.clone() for n, t in x.items()}, torch.empty_like(so), torch.empty_like(od))
                            for _ in range(rotation_count(nb) - 1)]
    rotate(rec, [lambda t=t: c.ops.kda_decode(t[0]["q"], t[0]["k"], t[0]["v"], t[0]["g"], t[0]["beta"],
                                              t[0]["S_in"], S_out=t[1], o=t[2]) for t in sets],
           nb, nb, c, wl, "gdn_decode_kernel (KDA gate)")
    rec["frac_hbm_peak"] = rec["value"] / c.F.PEAK_HBM_GBPS
    _, so, od = sets[(c.steps - 1) % len(sets)]
    del sets
    if c.cpu:
        from oracle import kda as okda
        from oracle.metrics import normwise_rel_err

        o_gpu, s_gpu = od.cpu(), so.cpu()
        leg = cpu_leg(lambda: okda.kda_decode_ref(**xh), nb, "GB/s",
                      f"the whole workload ({shape.batch}x{shape.n_heads} heads, {shape.d_k}x{shape.d_v} state; "
                      f"float64 numpy oracle)", got=o_gpu, ref_of=lambda r: r[0])
        leg["sample"] = leg["sample"].replace("fp32 torch CPU oracle", "float64 numpy CPU oracle")
        leg["parity_normwise_state_on_sample"] = normwise_rel_err(s_gpu, okda.kda_decode_ref(**xh)[1])
        rec["cpu_baseline"] = leg

    def sample():
        import torch as _t

        from oracle import kda as okda

        ro, rs = okda.kda_decode_ref(**xh)
        return {"check": "the whole workload (output and state), float64 numpy oracle",
                "output_normwise": _nw(od.float().cpu(), _t.from_numpy(ro).float()),
                "state_normwise": _nw(so.cpu(), _t.from_numpy(rs).float())}

    parity_record(c, rec, sample)
    del x, so, od
    return rec


QUANT_CPU_ROWS = 256  # rows of the 8192-wide activation the CPU leg quantises


def case_quant_fp8_act(c: Ctx) -> dict:
    import numpy as np
    import torch

    m = k = 8192
    xh = torch.randn((m, k), generator=torch.Generator().manual_seed(c.I.SEED)).to(torch.bfloat16)
    xa = xh.cuda()
    qa = torch.empty((m, k), dtype=torch.float8_e4m3fn, device="cuda")
    sa = torch.empty((m, k // 128), dtype=torch.float32, device="cuda")
    ms, wall = time_graph(lambda: c.ops.quant_fp8_act(xa, q=qa, scales=sa), c.steps, c.warmup)
    nb = c.F.quant_fp8_act_bytes(m, k)
    wl = f"quant_fp8_act {m}x{k} bf16 -> e4m3 + 1x128 scales"
    rec = {"workload": wl, "unit": "GB/s", "mean_ms": ms, "wall_ms": wall, "value": c.F.gbps(nb, ms),
           "roofline": roofline("hbm", nb, ms, c.F.PEAK_HBM_GBPS, "GB/s", wl, "quant_fp8_act_kernel<BF16>")}
    sets = [(xa, qa, sa)] + [(xa.clone(), torch.empty_like(qa), torch.empty_like(sa))
                             for _ in range(rotation_count(nb) - 1)]
    rotate(rec, [lambda t=t: c.ops.quant_fp8_act(t[0], q=t[1], scales=t[2]) for t in sets], nb, nb, c, wl,
           "quant_fp8_act_kernel<BF16>")
    rec["frac_hbm_peak"] = rec["value"] / c.F.PEAK_HBM_GBPS
    _, qa, sa = sets[(c.steps - 1) % len(sets)]
    del sets
    if c.cpu:
        from oracle import fp8 as ofp8

        r = QUANT_CPU_ROWS
        xs = xh[:r].float().numpy()
        leg = cpu_leg(lambda: ofp8.quantize_blockwise(xs, (1, 128)), c.F.quant_fp8_act_bytes(r, k), "GB/s",
                      f"the first {r} of {m} rows ({r}x{k}); numpy oracle")
        leg["sample"] = leg["sample"].replace("fp32 torch CPU oracle", "numpy CPU oracle")
        codes, scales = ofp8.quantize_blockwise(xs, (1, 128))
        leg["codes_bit_exact_on_sample"] = bool(np.array_equal(ofp8.fp8_tensor_codes(qa[:r].cpu()), codes))
        leg["scales_bit_exact_on_sample"] = bool(np.array_equal(sa[:r].cpu().numpy(), scales))
        rec["cpu_baseline"] = leg

    def sample():
        from oracle import fp8 as ofp8

        r = QUANT_CPU_ROWS
        codes, scales = ofp8.quantize_blockwise(xh[:r].float().numpy(), (1, 128))
        exact = (np.array_equal(ofp8.fp8_tensor_codes(qa[:r].cpu()), codes)
                 and np.array_equal(sa[:r].cpu().numpy(), scales))
        return {"check": f"the first {r} of {m} rows, codes and scales", "bit_exact": bool(exact)}

    parity_record(c, rec, sample)
    del xa, qa, sa
    return rec


MLA_PREFILL_CPU_HEADS = 16  # heads of 128 the CPU leg computes


def case_mla_prefill(c: Ctx) -> dict:
    import torch

    shape = c.S.MLA_PREFILL_BENCH
    qh, kh, vh = c.I.mla_prefill_inputs(shape, dtype=torch.bfloat16)
    q, k, v = qh.cuda(), kh.cuda(), vh.cuda()
    o = torch.empty((shape.batch, shape.n_h, shape.seq, shape.d_v), dtype=torch.bfloat16, device="cuda")
    ms, wall = time_graph(lambda: c.ops.mla_prefill_fwd(q, k, v, out=o), c.steps, c.warmup)
    fl = c.F.mla_attention_flops(shape)
    wl = f"mla_prefill B{shape.batch} S{shape.seq} H{shape.n_h} qk{shape.qk_head_dim} v{shape.d_v} bf16 non-causal"
    rec = {"workload": wl, "unit": "TFLOPS", "mean_ms": ms, "wall_ms": wall,
           "value": c.F.tflops(fl, ms), "frac_mfma_peak": c.F.tflops(fl, ms) / c.F.PEAK_BF16_TFLOPS,
           "roofline": roofline("mfma", fl, ms, c.F.PEAK_BF16_TFLOPS, "TFLOP/s", wl,
                                "gqa_fwd_kernel<192, 128, BF16, false, 1, 8, 1>")}
    if c.cpu:
        from oracle import mla as omla

        hs = list(range(MLA_PREFILL_CPU_HEADS))
        got = o[:, :len(hs)].cpu()
        rec["cpu_baseline"] = cpu_leg(lambda: omla.mla_prefill_ref(qh, kh, vh, heads=hs)[:, :len(hs)],
                                      fl * len(hs) // shape.n_h, "TFLOPS",
                                      f"{len(hs)} of {shape.n_h} heads (S={shape.seq}, full S x S)", got=got)

    def sample():
        from oracle import mla as omla

        hs = [0, 1]
        return {"check": f"heads {hs} of {shape.n_h} (S={shape.seq}, full S x S)",
                "output_normwise": _nw(o[:, hs].cpu(), omla.mla_prefill_ref(qh, kh, vh, heads=hs)[:, hs])}

    parity_record(c, rec, sample)
    del q, k, v, o
    return rec


CASES = {
    "gqa": case_gqa,
    "gemm_bf16_1024": case_gemm_bf16_1024,
    "gemm_bf16_8192": case_gemm_bf16_8192,
    "gemm_fp8_8192": case_gemm_fp8_8192,
    "mla_decode": case_mla_decode,
    "gdn_decode": case_gdn_decode,
    "mla_absorbed": case_mla_absorbed,
    "kda_decode": case_kda_decode,
    "quant_fp8_act": case_quant_fp8_act,
    "mla_prefill": case_mla_prefill,
    "hipblaslt_8192": case_hipblaslt_8192,
    "hbm_copy": case_hbm_copy,
}
# vendor / runtime reference lines: they compute nothing of this path
REFERENCE_LINES = ("hipblaslt_8192", "hbm_copy")
# the BASELINE.json configs; these and the absorbed step, KDA, the
# quantiser and the prefill carry a roofline block and a CPU leg
BASELINE_CASES = ("gqa", "gemm_bf16_1024", "gemm_bf16_8192", "gemm_fp8_8192", "mla_decode", "gdn_decode")


def calibrate_copy(steps: int) -> int:
    """A plain device-to-device copy of a known size (1 GiB read + 1 GiB
    written per launch), for scaling rocprofv3 FETCH_SIZE / WRITE_SIZE
    readings of the kernels above to bytes."""
    import torch

    n = 1 << 30
    src = torch.empty(n, dtype=torch.uint8, device="cuda").fill_(1)
    dst = torch.empty_like(src)
    for _ in range(2):
        dst.copy_(src)
    torch.cuda.synchronize()
    for _ in range(steps):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"calibration": "device copy", "bytes_read_per_launch": n, "bytes_written_per_launch": n,
                      "launches": steps}), flush=True)
    return 0


def settle_note() -> dict:
    return {"ms_before_each_case": SETTLE_MS,
            "work": "torch.matmul 8192x8192 bf16 (a device GEMM, not the measured kernel)",
            "why": "the GPU leaves idle clocks only after a few hundred ms of load; warm-up and timed steps "
                   "(exactly --warmup and --steps) then run at load clocks"}


def _clean(rec: dict) -> dict:
    return {k: v for k, v in rec.items() if k not in ("shape",)}


def main() -> int:
    global SETTLE_MS
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--settle-ms", type=float, default=SETTLE_MS,
                    help="device GEMM load before each case's warm-up (ms; 0 disables)")
    ap.add_argument("--only-headline", action="store_true", help="run only the headline GQA case")
    ap.add_argument("--only", default="", help=f"comma-separated cases to run (of {', '.join(CASES)})")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="run only a 1 GiB device copy (profiler calibration of byte counters)")
    args = ap.parse_args()

    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path "
              "(every kernel is single-device; sharding is described in DESIGN.md). "
              "Run with --gpus 1.", file=sys.stderr)
        return 2
    SETTLE_MS = max(0.0, args.settle_ms)
    if args.steps < 1 or args.warmup < 0:
        print("--steps must be >= 1 and --warmup >= 0", file=sys.stderr)
        return 2
    only = [s for s in args.only.split(",") if s]
    unknown = [s for s in only if s not in CASES]
    if unknown:
        print(f"unknown case(s) {unknown}; known: {', '.join(CASES)}", file=sys.stderr)
        return 2

    import torch

    if args.calibrate_copy:
        return calibrate_copy(args.steps)
    pkg = importlib.import_module("cuda-oxide-bench_amd")
    ops = pkg.load_ops()
    log(f"device: {torch.cuda.get_device_name(0)}")
    ctx = Ctx(pkg, ops, args.steps, args.warmup, cpu=not args.no_cpu_baseline)

    names = only or (["gqa"] if args.only_headline else list(CASES))
    results = {}
    for name in names:
        log(f"case {name} ...")
        rec = CASES[name](ctx)
        extra = f", CPU {rec['cpu_baseline']['value']:.4g} {rec['cpu_baseline']['unit']}" \
            if "cpu_baseline" in rec else ""
        log(f"case {name}: {rec['value']:.1f} {rec['unit']} (event mean {rec['mean_ms'] * 1e3:.2f} us){extra}")
        results[name] = rec

    return emit(results, names, args.steps, args.warmup, pkg.flops.tflops)


def emit(results: dict, names: list, steps: int, warmup: int, tflops) -> int:
    """Print the one JSON line, or nothing and status 3 when a case failed its parity check."""
    bad = parity_failures(results)
    if bad:
        for b in bad:
            log(f"PARITY FAILURE {b}")
        log("no numbers reported: a kernel that fails its correctness check is not published")
        return 3
    head = results.get("gqa")
    if head is None:  # a profiling run of other cases: report the first one as the line's value
        first = results[names[0]]
        print(json.dumps({"metric": METRIC, "value": round(first["value"], 3), "unit": first["unit"], "n_gpus": 1,
                          "steps": steps, "warmup": warmup, "ms_per_step": round(first["wall_ms"], 5),
                          "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
                          "dtype": "bf16", "data": "synthetic", "config": {"workload": first["workload"]},
                          "partial_run": names, "settle": settle_note(),
                          "others": {n: _clean(r) for n, r in results.items()}},
                         default=float), flush=True)
        return 0

    shape = head["shape"]
    line = {
        "metric": METRIC,
        "value": round(tflops(head["flops"], head["wall_ms"]), 3),
        "unit": "TFLOPS",
        "n_gpus": 1,
        "steps": steps,
        "warmup": warmup,
        "ms_per_step": round(head["wall_ms"], 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded N(0,1) bf16 Q/K/V, seed 0xC0FFEE)",
        "config": {
            "workload": head["workload"],
            "batch": shape.batch, "seq": shape.seq, "n_q": shape.n_q, "n_kv": shape.n_kv,
            "d_head": shape.d_head, "causal": True, "softmax_scale": shape.d_head ** -0.5,
            "flops_per_step": head["flops"], "flops_convention": "causal algorithmic 2*B*Hq*D*S*(S+1)",
        },
        "roofline": head["roofline"],
        "cpu_baseline": head.get("cpu_baseline"),
        "parity": head.get("parity"),
        "settle": settle_note(),
        "tflops_reference_convention": round(head["tflops_reference_convention"], 3),
        "others": {n: _clean(r) for n, r in results.items() if n != "gqa"},
    }
    print(json.dumps(line, default=float), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
