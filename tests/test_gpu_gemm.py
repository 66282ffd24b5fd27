"""bf16 GEMM parity on the GPU: HIP kernel vs the CPU oracle (fp32 matmul of
the bf16 operands, cutile-matmul-tc-bf16/main.py:98-107).  Bound: normwise
max|got-ref|/max|ref| <= 2e-2 (bf16 output), plus the reference harness's
own sampled gate |err| <= 0.2 + 0.05|ref| (:129-135) and exact KATs."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import announce, from_bits, import_submodule, load_golden
from oracle import gemm as ogemm
from oracle.metrics import normwise_rel_err

pytestmark = pytest.mark.gpu
TOL = 2e-2

shapes = import_submodule("shapes")
inputs = import_submodule("inputs")


def run(ops, a, b):
    c = ops.gemm_bf16(a.cuda(), b.cuda())
    torch.cuda.synchronize()
    return c.cpu()


def test_golden_fixture(ops):
    announce("gemm_bf16 golden 72x136x96")
    g = load_golden("gemm_bf16_72x136x96")
    a, b = from_bits(g["a"], torch.bfloat16), from_bits(g["b"], torch.bfloat16)
    c = run(ops, a, b)
    assert normwise_rel_err(c, g["c"]) <= 1e-2


@pytest.mark.parametrize("mnk", [(1, 8, 8), (16, 16, 32), (100, 136, 72), (257, 264, 520), (512, 512, 512),
                                 (1024, 1024, 1024), (2048, 1024, 512), (4096, 8192, 256)])
def test_parity_vs_oracle(ops, mnk):
    m, n, k = mnk
    announce(f"gemm_bf16 {m}x{n}x{k}")
    a, b = inputs.gemm_inputs(shapes.GemmShape("t", m, n, k))
    c = run(ops, a, b)
    ref = ogemm.gemm_ref(a, b)
    err = normwise_rel_err(c, ref)
    assert err <= TOL, f"normwise rel err {err:.3e}"
    # bf16 output: every element within a few bf16 ulps of the fp32 result
    assert torch.all((c.float() - ref).abs() <= 0.2 + 0.05 * ref.abs())


@pytest.mark.parametrize("mnk,path", [((64, 64, 4096), "32-column streams"),
                                      ((256, 1024, 2048), "32-column streams"),
                                      ((1024, 1024, 1024), "256 tiles, 16 K tiles"),
                                      ((1024, 1024, 576), "9 K tiles"),
                                      ((960, 1024, 512), "240 tiles, 8 K tiles"),
                                      ((1024, 1024, 512), "256 tiles, 8 K tiles"),
                                      ((768, 1024, 640), "192 tiles, 10 K tiles"),
                                      ((1024, 960, 768), "240 tiles, 12 K tiles"),
                                      ((512, 2048, 896), "256 tiles, 14 K tiles"),
                                      ((1024, 1024, 1536), "256 tiles, 24 K tiles"),
                                      ((512, 1024, 4096), "64-column streams")])
def test_small_grid_paths(ops, mnk, path):
    """Grids of at most one 64x64 tile per CU with K >= 512: streams of B for
    the fewest tiles, else 64x64 tiles through a ring of four K tiles, with
    K tile counts around whole periods of the ring."""
    m, n, k = mnk
    announce(f"gemm_bf16 {m}x{n}x{k} ({path})")
    a, b = inputs.gemm_inputs(shapes.GemmShape("t", m, n, k))
    c = run(ops, a, b)
    ref = ogemm.gemm_ref(a, b)
    err = normwise_rel_err(c, ref)
    assert err <= TOL, f"normwise rel err {err:.3e}"
    assert torch.all((c.float() - ref).abs() <= 0.2 + 0.05 * ref.abs())


@pytest.mark.parametrize("mnk", [(1024, 1024, 1024), (768, 1024, 640), (1024, 1024, 1536)])
def test_small_grid_strided(ops, mnk):
    """Leading dimensions beyond the row lengths (lda > K, ldb > N,
    ldc > N) on 64x64 tiles; C's padding columns are left untouched."""
    m, n, k = mnk
    announce(f"gemm_bf16 {m}x{n}x{k} strided")
    lib = import_submodule("_lib")
    a, b = inputs.gemm_inputs(shapes.GemmShape("t", m, n, k))
    pad = 72
    a_full = torch.zeros((m, k + pad), dtype=torch.bfloat16, device="cuda")
    b_full = torch.zeros((k, n + pad), dtype=torch.bfloat16, device="cuda")
    c_full = torch.full((m, n + pad), 7.0, dtype=torch.bfloat16, device="cuda")
    a_full[:, :k] = a.cuda()
    b_full[:, :n] = b.cuda()
    lib.call("mx_gemm_bf16", a_full.data_ptr(), b_full.data_ptr(), c_full.data_ptr(), m, n, k, k + pad, n + pad,
             n + pad, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    c = c_full.cpu()
    ref = ogemm.gemm_ref(a, b)
    err = normwise_rel_err(c[:, :n], ref)
    assert err <= TOL, f"normwise rel err {err:.3e}"
    assert torch.all((c[:, :n].float() - ref).abs() <= 0.2 + 0.05 * ref.abs())
    assert torch.all(c[:, n:] == 7.0)


def test_reference_distribution_sampled_gate(ops):
    """The reference harness's own check at its smoke size: U[0,1) inputs,
    200 sampled cells, |err| <= 0.2 + 0.05|ref| (cutile-matmul-tc-bf16/main.py:110-135)."""
    announce("gemm_bf16 reference-dist 512 sampled")
    s = shapes.GEMM_SMOKE
    a, b = inputs.gemm_inputs(s, dist="reference")
    c = run(ops, a, b).float().numpy()
    rng = np.random.default_rng(inputs.SAMPLE_SEED)
    rows = rng.integers(0, s.m, size=200)
    cols = rng.integers(0, s.n, size=200)
    refs = ogemm.sample_reference(a, b, rows, cols)
    got = c[rows, cols]
    assert np.all(np.abs(got - refs) <= 0.2 + 0.05 * np.abs(refs))


@pytest.mark.parametrize("k", [64, 1024])
def test_kat_constant(ops, k):
    """A=1, B=1 -> K; A=2, B=3 -> 6K (oxide-gemm-sol/bench/cublas_correctness_test.py:8-11)."""
    announce(f"gemm_bf16 KAT constant K={k}")
    m = n = 256
    for av, bv, want in ((1.0, 1.0, k), (2.0, 3.0, 6 * k)):
        a = torch.full((m, k), av, dtype=torch.bfloat16)
        b = torch.full((k, n), bv, dtype=torch.bfloat16)
        c = run(ops, a, b)
        assert torch.all(c.float() == want)


def test_kat_pattern(ops):
    """A[i,:]=(i%8+1), B[:,j]=(j%8+1) -> (i%8+1)(j%8+1)K, exactly representable."""
    announce("gemm_bf16 KAT pattern")
    m, n, k = 384, 264, 128
    a = (torch.arange(m) % 8 + 1).float()[:, None].expand(m, k).to(torch.bfloat16).contiguous()
    b = (torch.arange(n) % 8 + 1).float()[None, :].expand(k, n).to(torch.bfloat16).contiguous()
    c = run(ops, a, b).float()
    want = ((torch.arange(m) % 8 + 1)[:, None] * (torch.arange(n) % 8 + 1)[None, :] * k).float()
    assert torch.equal(c, want)


@pytest.mark.parametrize("mnk", [(4096, 4096, 32), (4096, 4096, 96), (4000, 4040, 4128), (4096, 4352, 2048),
                                 (4096, 4096, 64), (4096, 4096, 192), (4000, 4040, 4096), (4096, 4096, 1600)])
def test_direct_load_path(ops, mnk):
    """About one 256x256 tile per CU and more: 256x256 tiles (A and B rings of
    their own) from K 192 on, 128x192 where their rounds fill the CUs better,
    128x128 with the whole K at once below K 128.  Fewer K tiles than ring
    slots, a K tail of 32, ragged M and N, and K-tile counts that are no
    multiple of either ring's period."""
    m, n, k = mnk
    announce(f"gemm_bf16 direct-load {m}x{n}x{k}")
    a, b = inputs.gemm_inputs(shapes.GemmShape("t", m, n, k))
    c = run(ops, a, b)
    ref = ogemm.gemm_ref(a, b)
    err = normwise_rel_err(c, ref)
    assert err <= TOL, f"normwise rel err {err:.3e}"
    assert torch.all((c.float() - ref).abs() <= 0.2 + 0.05 * ref.abs())


def test_target_size_sampled(ops):
    """8192^3 (the roofline target): 256 cells against fp64 dot products."""
    announce("gemm_bf16 8192^3 sampled")
    s = shapes.GEMM_TARGET
    a, b = inputs.gemm_inputs(s)
    c = ops.gemm_bf16(a.cuda(), b.cuda())
    torch.cuda.synchronize()
    rng = np.random.default_rng(inputs.SAMPLE_SEED)
    rows = rng.integers(0, s.m, size=256)
    cols = rng.integers(0, s.n, size=256)
    got = c[torch.from_numpy(rows).cuda(), torch.from_numpy(cols).cuda()].float().cpu().numpy()
    a32, b32 = a.float().numpy(), b.float().numpy()
    ref = np.array([ogemm.ref_elem(a32, b32, r, cc) for r, cc in zip(rows, cols)])
    scale = np.abs(ref).max()
    assert np.abs(got - ref).max() / scale <= TOL


@pytest.mark.parametrize("mnk,path", [((2048, 2048, 2048), "128x128 tiles, 64 K tiles"),
                                      ((2000, 2040, 2048), "ragged M and N"),
                                      ((2560, 2560, 1024), "400 tiles: two rounds of workgroups"),
                                      ((2048, 2048, 32), "half a K tile, the whole K at once"),
                                      ((2048, 2048, 160), "two K tiles and a tail of 32, fewer than the ring's stages"),
                                      ((2048, 4096, 1056), "16 K tiles and a tail of 32: three ring periods and one"),
                                      ((4080, 2056, 256), "ragged, 544 tiles")])
def test_direct_load_128_paths(ops, mnk, path):
    """Mid-size GEMMs: 128x128 tiles through a ring of five K tiles, or the
    whole K at once (K 32); 256x256 tiles for the last shape.  2048^3 is a size of the reference's
    mixed-dtype harness sweep (cutile-matmul-tiled-mixed/main.py:60)."""
    m, n, k = mnk
    announce(f"gemm_bf16 {m}x{n}x{k} direct-load 128x128 ({path})")
    a, b = inputs.gemm_inputs(shapes.GemmShape("t", m, n, k))
    c = run(ops, a, b)
    ref = ogemm.gemm_ref(a, b)
    err = normwise_rel_err(c, ref)
    assert err <= TOL, f"normwise rel err {err:.3e}"
    assert torch.all((c.float() - ref).abs() <= 0.2 + 0.05 * ref.abs())


@pytest.mark.parametrize("mnk", [(1, 7168, 4096), (16, 4096, 7168), (32, 256, 64), (33, 1000, 192), (64, 2048, 7168),
                                 (7, 296, 640), (48, 3000, 1344), (256, 512, 4096), (130, 1024, 2048),
                                 (1000, 96, 1024), (2048, 128, 4096), (96, 512, 8192)])
def test_weight_streaming_small_m(ops, mnk):
    """Few rows or few tiles run the streams of B, here the 32x32 one: single
    rows, one K block (fewer than the waves), a last chunk of 1, 2 or 8 rows, a
    last column block 8 or 24 wide, block counts that do not divide by the
    wave count, more rows than columns."""
    m, n, k = mnk
    announce(f"gemm_bf16 {m}x{n}x{k} weight streaming")
    a, b = inputs.gemm_inputs(shapes.GemmShape("t", m, n, k))
    c = run(ops, a, b)
    ref = ogemm.gemm_ref(a, b)
    err = normwise_rel_err(c, ref)
    assert err <= TOL, f"normwise rel err {err:.3e}"
    assert torch.all((c.float() - ref).abs() <= 0.2 + 0.05 * ref.abs())


@pytest.mark.parametrize("mnk,path", [((3072, 3072, 1024), "144 tiles of 256x256 against 576 of 128x128"),
                                      ((3000, 3064, 512), "ragged, 144 tiles"),
                                      ((3584, 3584, 2048), "196 tiles against 784")])
def test_direct_load_256_below_one_tile_per_cu(ops, mnk, path):
    """Fewer than one 256x256 tile per CU still runs 256x256 tiles where the
    rounds of 128x128 ones would cost more."""
    m, n, k = mnk
    announce(f"gemm_bf16 {m}x{n}x{k} direct-load 256x256 ({path})")
    a, b = inputs.gemm_inputs(shapes.GemmShape("t", m, n, k))
    c = run(ops, a, b)
    ref = ogemm.gemm_ref(a, b)
    err = normwise_rel_err(c, ref)
    assert err <= TOL, f"normwise rel err {err:.3e}"
    assert torch.all((c.float() - ref).abs() <= 0.2 + 0.05 * ref.abs())


@pytest.mark.parametrize("mnk,path", [((2048, 2048, 2056), "128x128 tiles, K tail of 8"),
                                      ((4096, 8192, 264), "256x256 tiles, K tail of 8"),
                                      ((2048, 2048, 72), "128x128 tiles, whole K at once")])
def test_k_tail_of_eight(ops, mnk, path):
    """Large products whose K is 8 past a multiple of 64."""
    m, n, k = mnk
    announce(f"gemm_bf16 {m}x{n}x{k} {path}")
    a, b = inputs.gemm_inputs(shapes.GemmShape("t", m, n, k))
    c = run(ops, a, b)
    ref = ogemm.gemm_ref(a, b)
    err = normwise_rel_err(c, ref)
    assert err <= TOL, f"normwise rel err {err:.3e}"
    assert torch.all((c.float() - ref).abs() <= 0.2 + 0.05 * ref.abs())


def test_rejects_bad_arguments(ops):
    a = torch.zeros((64, 60), dtype=torch.bfloat16, device="cuda")  # K % 8 != 0
    b = torch.zeros((60, 64), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(Exception):
        ops.gemm_bf16(a, b)


@pytest.mark.parametrize("bmnk", [(1, 64, 64, 64), (7, 100, 136, 72), (128, 32, 512, 128), (128, 32, 128, 512), (16, 5, 40, 192),
                                  (3, 300, 264, 520), (4, 1024, 1024, 256),
                                  # K split among the waves: 4, 8 and 12 chunks of K, 32 x 64 and 32 x 32
                                  # tiles, ragged M and N
                                  (8, 17, 72, 256), (64, 32, 136, 768), (200, 32, 128, 512), (3, 1, 8, 512)])
def test_batched_vs_oracle(ops, bmnk):
    """Strided-batched GEMM: every item against the fp32 oracle (small-row
    kernels with and without K split among the waves, 64x64 tiles and, at 4 x
    1024x1024x256, 128x128 ones)."""
    nb, m, n, k = bmnk
    announce(f"gemm_bf16_batched {nb}x{m}x{n}x{k}")
    g = torch.Generator().manual_seed(nb * 131 + m)
    a = (torch.rand((nb, m, k), generator=g) * 2 - 1).to(torch.bfloat16)
    b = (torch.rand((nb, k, n), generator=g) * 2 - 1).to(torch.bfloat16)
    c = ops.gemm_bf16_batched(a.cuda(), b.cuda())
    torch.cuda.synchronize()
    c = c.cpu()
    for i in range(nb):
        ref = ogemm.gemm_ref(a[i], b[i])
        assert normwise_rel_err(c[i], ref) <= TOL
        assert torch.all((c[i].float() - ref).abs() <= 0.2 + 0.05 * ref.abs())


def _check_elementwise(c, a, b):
    """|C - A.B| within one bf16 rounding (2^-8 relative) plus fp32 sums of K
    terms (K 2^-24 of the sum of magnitudes), against a 64-bit product."""
    a64, b64 = a.double(), b.double()
    ref = a64 @ b64
    bound = ref.abs() * 2.0 ** -8 + (a64.abs() @ b64.abs()) * (a.shape[1] * 2.0 ** -24) + 1e-30
    worst = ((c.double() - ref).abs() / bound).max().item()
    assert worst <= 1.0, f"{worst:.2f} times the bound"


# every kernel of the dispatch: streams of 32 and 64 rows and of 32 and 64
# columns, 64x64, 64x128, 128x128, 128x192 and 256x256 tiles, with K tails on both sides of 32, K
# below one 64-deep block, a single block, and edges off the tiles
RAGGED_K = [(1, 8, 8), (16, 520, 72), (33, 264, 520), (1, 1024, 2056), (50, 5288, 2168), (100, 3200, 1800),
            (129, 200, 24), (300, 1104, 656), (129, 136, 40), (500, 1496, 1048), (1315, 840, 1128),
            (777, 3592, 200), (2000, 2040, 264), (554, 7384, 136), (607, 7040, 104), (3500, 1032, 16),
            (1937, 7024, 104), (4000, 4040, 72), (4096, 4096, 152),
            # 64-column streams: 32 rows (K tails of 8, a last column block 8 wide, a last row of its own), 64
            # rows (from K 3072; wide and tall)
            (65, 4104, 200), (257, 1032, 1032), (130, 2056, 520), (500, 1032, 3080), (1000, 520, 3080),
            (129, 4104, 3072), (3000, 264, 3136),
            # tails that the sizes above leave out: 64x128 (both sides of 32), 128x128, 128x192 and 256x256 tiles,
            # 32-row streams of 32 and 64 columns, 64x64 streams; 64-row streams without one
            (1067, 1136, 1488), (782, 2160, 808), (403, 5136, 168), (1214, 4400, 168), (2330, 4104, 176), (1, 64, 304),
            (92, 4088, 304), (395, 1472, 3896), (436, 856, 384)]


@pytest.mark.parametrize("mnk", RAGGED_K)
def test_any_k_on_every_kernel(ops, mnk):
    """A and B sit inside wider buffers filled with NaN, so anything read past
    K, N or M that reached a sum would show; C's surroundings stay untouched."""
    m, n, k = mnk
    announce(f"gemm_bf16 {m}x{n}x{k} any K")
    lib = import_submodule("_lib")
    a, b = (t.cuda() for t in inputs.gemm_inputs(shapes.GemmShape("t", m, n, k)))
    wide = lambda r, c: torch.full((r + 2, c + 16), float("nan"), dtype=torch.bfloat16, device="cuda")
    aw, bw, cw = wide(m, k), wide(k, n), torch.full((m + 2, n + 16), 7.0, dtype=torch.bfloat16, device="cuda")
    aw[:m, :k], bw[:k, :n] = a, b
    lib.call("mx_gemm_bf16", aw.data_ptr(), bw.data_ptr(), cw.data_ptr(), m, n, k, k + 16, n + 16, n + 16, 0)
    torch.cuda.synchronize()
    _check_elementwise(cw[:m, :n], a, b)
    assert torch.all(cw[m:] == 7.0) and torch.all(cw[:, n:] == 7.0)
    c = ops.gemm_bf16(a, b)
    torch.cuda.synchronize()
    assert torch.equal(c, cw[:m, :n])


# K below 128, where tiles take the whole K to LDS at once, and the 32-row stream: every K chunk count up to
# 32 and beside 64, one and two stages, blocks of eight rows without a row, edges on and off the tiles
SHORT_K = [(1, 8, 8), (64, 64, 64), (65, 72, 120), (152, 392, 40), (7, 3984, 24), (63, 56, 32), (9, 136, 56), (130, 64, 16),
           (816, 1360, 8), (1837, 600, 96), (508, 2720, 40), (797, 2072, 104), (530, 3216, 64), (2268, 1672, 120),
           (3052, 2256, 32), (1215, 3840, 8), (1506, 2752, 48), (4096, 4096, 64), (12, 968, 88), (782, 128, 104),
           (65, 2184, 72), (794, 1016, 104)]


@pytest.mark.parametrize("mnk", SHORT_K)
def test_short_k(ops, mnk):
    test_any_k_on_every_kernel(ops, mnk)


@pytest.mark.parametrize("bmnk", [(1, 1, 8, 8), (3, 9, 64, 40), (7, 65, 72, 120), (57, 2, 392, 48), (24, 3, 912, 72),
                                  (15, 244, 504, 32), (34, 273, 928, 8), (36, 228, 224, 104), (7, 554, 776, 120),
                                  (28, 1, 504, 120), (18, 331, 288, 40)])
def test_batched_short_k(ops, bmnk):
    """Batched items with K below 128: the 64x64, 64x128 and 128x128 tiles."""
    test_batched_larger_items(ops, bmnk)


@pytest.mark.parametrize("mnk", [(40, 600, 328), (300, 1104, 264), (130, 2056, 520), (500, 1032, 3080),
                                 (700, 1400, 520), (2000, 2040, 264), (4000, 4040, 104), (130, 200, 40), (65, 72, 8),
                                 (900, 1360, 24)])
def test_infinity_in_the_last_k_row(ops, mnk):
    """The K tail re-reads the last k-row for the missing ones: an infinity
    there counts once, against zeros it gives NaN only where A holds a zero."""
    m, n, k = mnk
    announce(f"gemm_bf16 {m}x{n}x{k} infinity in the last k-row")
    a, b = (t.cuda() for t in inputs.gemm_inputs(shapes.GemmShape("t", m, n, k)))
    b[-1, 3] = float("inf")
    a[::7, -1] = 0.0
    c = ops.gemm_bf16(a, b)
    torch.cuda.synchronize()
    want = torch.where(a[:, -1] == 0, float("nan"), torch.sign(a[:, -1].float()) * float("inf"))
    assert torch.equal(c[:, 3].float().nan_to_num(nan=123.0), want.nan_to_num(nan=123.0))
    assert torch.isfinite(c[:, :3].float()).all() and torch.isfinite(c[:, 4:].float()).all()


@pytest.mark.parametrize("bmnk", [(5, 40, 1000, 72), (16, 48, 128, 512), (3, 300, 264, 136), (40, 200, 640, 136),
                                  (30, 600, 400, 104), (2, 33, 8, 8), (70, 130, 200, 24),
                                  # chunks of 32 rows: K split among the waves (last chunk 1 and 8 rows, ragged N,
                                  # the most groups and one item more), and one and two chunks of K
                                  (7, 65, 136, 768), (16, 200, 128, 512), (64, 64, 128, 256), (65, 64, 128, 256),
                                  (16, 33, 512, 64), (37, 64, 264, 128), (128, 48, 512, 128), (3, 65, 72, 128),
                                  # ... up to 768 workgroups of 32 x 32 at any M, and one item more
                                  (48, 128, 128, 64), (49, 128, 128, 64), (9, 96, 520, 128), (5, 1000, 72, 128),
                                  # 64x64 to 128x192 tiles from K 128 on, K tails on both sides of 32 and none
                                  (1, 1, 8, 152), (1, 104, 8, 240), (12, 542, 232, 800), (9, 815, 248, 888),
                                  (18, 222, 792, 176), (56, 374, 432, 216), (16, 563, 400, 296),
                                  # small-row tiles of 64 and 128 columns, column tiles or items first in the grid
                                  (64, 2, 496, 64), (137, 1, 232, 192), (119, 1, 616, 320)])
def test_batched_larger_items(ops, bmnk):
    """Batched items with more than 32 rows, or a K that is no whole number of
    64-deep chunks, run the tiled kernels over the batch, or the small-row
    kernels in chunks of 32 rows."""
    nb, m, n, k = bmnk
    announce(f"gemm_bf16_batched {nb}x{m}x{n}x{k}")
    g = torch.Generator().manual_seed(nb + m + n + k)
    a = (torch.rand((nb, m, k), generator=g) * 2 - 1).to(torch.bfloat16).cuda()
    b = (torch.rand((nb, k, n), generator=g) * 2 - 1).to(torch.bfloat16).cuda()
    c = ops.gemm_bf16_batched(a, b)
    torch.cuda.synchronize()
    for i in range(nb):
        _check_elementwise(c[i], a[i], b[i])


@pytest.mark.parametrize("bmnk", [(1, 3, 65535 * 64 + 72, 256), (2, 2, 65535 * 128 + 8, 192)])
def test_batched_many_column_tiles(ops, bmnk):
    """Small-row kernels over more than 65535 column tiles: every column is
    written, those around that tile and at both ends are right."""
    nb, m, n, k = bmnk
    announce(f"gemm_bf16_batched {nb}x{m}x{n}x{k}")
    g = torch.Generator(device="cuda").manual_seed(k)
    a = (torch.rand((nb, m, k), generator=g, device="cuda") * 2 - 1).to(torch.bfloat16)
    b = torch.empty((nb, k, n), dtype=torch.bfloat16, device="cuda").uniform_(-1, 1, generator=g)
    c = torch.full((nb, m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.gemm_bf16_batched(a, b, out=c)
    torch.cuda.synchronize()
    assert not torch.isnan(c).any()
    seam = 65535 * (64 if k % 256 == 0 else 128)
    for lo, hi in ((0, 512), (seam - 512, min(n, seam + 512)), (n - 512, n)):
        for i in range(nb):
            _check_elementwise(c[i, :, lo:hi], a[i], b[i, :, lo:hi])
