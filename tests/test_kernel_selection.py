"""Which kernel the launch rules give the shapes of the GPU tests (host code, no
GPU).  A rule that moves shapes between kernels moves the tests with it; these
fail when a kernel, or its code for a K tail, is left without one."""
from __future__ import annotations

import itertools

import test_gpu_fp8 as fp8
import test_gpu_gemm as gemm
import test_gpu_gqa as gqa
from host_query import query

PATHS = ["None", "Stream32", "Stream32x64", "Stream64", "Stream64x64", "T64", "T64x128", "T128", "T128x192", "T256"]


def cases(test) -> list:
    """The values of a test's only parametrize mark."""
    return next(m.args[1] for m in test.pytestmark if m.name == "parametrize")


def table(rows) -> str:
    return "{" + ", ".join("{" + ", ".join(map(str, r)) + "}" for r in rows) + "}"


def tail(k: int) -> str:
    return "whole" if k % 64 == 0 else "to 32" if k % 64 <= 32 else "past 32"


def test_bf16_gemm(tmp_path):
    """Every kernel with no K tail, one of up to 32 and a longer one, from K 128
    on; below, the whole-K tiles in one and two stages."""
    ragged = gemm.RAGGED_K + gemm.SHORT_K
    whole = [c[0] if isinstance(c[0], tuple) else c
             for t in (gemm.test_parity_vs_oracle, gemm.test_small_grid_paths, gemm.test_direct_load_path,
                       gemm.test_direct_load_128_paths, gemm.test_weight_streaming_small_m,
                       gemm.test_direct_load_256_below_one_tile_per_cu) for c in cases(t)]
    rows = ragged + whole
    got = query(tmp_path, "gemm_bf16.hip", f"""
  static const int c[][3] = {table(rows)};
  for (auto& x : c) printf("%d\\n", (int)mx::gemm::gemm_path(x[0], x[1], x[2], x[2], x[1], 0));""")
    seen, short = set(), set()
    for (m, n, k), p in zip(rows, got):
        if k >= 128:
            seen.add((PATHS[int(p)], tail(k)))
        else:
            short.add((PATHS[int(p)], -(-k // 64)))
    missing = set(itertools.product(PATHS[1:], ("whole", "to 32", "past 32"))) - seen
    assert not missing
    assert not set(itertools.product(("T64", "T64x128", "T128"), (1, 2))) - short


def test_bf16_batched(tmp_path):
    """Tiles with every tail, whole-K tiles in one and two stages, and the
    small-row kernels of every width, K split between waves or not, with one
    row chunk and several."""
    rows = cases(gemm.test_batched_vs_oracle) + cases(gemm.test_batched_larger_items) + cases(gemm.test_batched_short_k)
    got = query(tmp_path, "gemm_bf16.hip", f"""
  using namespace mx::gemm;
  static const int c[][4] = {table(rows)};
  for (auto& x : c) {{
    const int b = x[0], m = x[1], n = x[2], k = x[3];
    if (batched_small(m, k, k, n) || batched_rows(b, m, n, k, k, n))
      printf("%s %d\\n", small_split_k(k) ? "split" : "one", small_width(b, m, n, k));
    else
      printf("%d\\n", (int)gemm_path(m, n, k, k, n, b));
  }}""")
    seen, short, small = set(), set(), set()
    for (b, m, n, k), p in zip(rows, got):
        if p[0] in "os":
            small.add((*p.split(), "rows" if m > 32 else "one chunk"))
        elif k >= 128:
            seen.add((PATHS[int(p)], tail(k)))
        else:
            short.add((PATHS[int(p)], -(-k // 64)))
    assert not set(itertools.product(("T64", "T64x128", "T128", "T128x192"), ("to 32", "past 32"))) - seen
    assert not set(itertools.product(("T64", "T64x128", "T128"), (1, 2))) - short
    want = {("one", "1", "one chunk"), ("one", "2", "one chunk"), ("one", "4", "one chunk"), ("one", "1", "rows"),
            ("split", "1", "one chunk"), ("split", "2", "one chunk"), ("split", "1", "rows"), ("split", "2", "rows")}
    assert not want - small


def test_fp8_gemm(tmp_path):
    """Every kernel; the tiled ones with activation scales four blocks per load and one."""
    names = ["Stream32", "Stream64", "Stream64x64", "T128", "T128x256", "T192x256", "T256"]
    rows = [c for t in (fp8.test_parity_vs_oracle, fp8.test_small_m_path, fp8.test_large_tile_path,
                        fp8.test_wide_tiles_and_streams, fp8.test_scale_alignment) for c in cases(t)]
    got = query(tmp_path, "gemm_fp8_bs.hip", f"""
  static const int c[][3] = {table(rows)};
  for (auto& x : c) printf("%d\\n", (int)mx::gemm8::gemm_path(x[0], x[1], x[2]));""")
    seen = {(names[int(p)], k % 512 == 0) for (m, n, k), p in zip(rows, got)}
    assert {n for n, _ in seen} == set(names)
    assert not set(itertools.product(names[3:], (True, False))) - seen


def test_attention_key_groups(tmp_path):
    """The sizes meant for two and four key groups get them, causal or not."""
    rows = gqa.KEY_GROUPS
    got = query(tmp_path, "gqa_fwd.hip", "  using namespace mx::gqa;\n" + "\n".join(
        f'  printf("%d %d\\n", pick_split<{d}, {d}>({b}, {hq}, {hkv}, {s}, 1).ksp, pick_split<{d}, {d}>({b}, {hq}, {hkv}, {s}, 0).ksp);'
        for b, s, hq, hkv, d in rows))
    groups = {r: tuple(map(int, g.split())) for r, g in zip(rows, got)}
    for r in rows:
        if r in gqa.ONE_GROUP:
            assert 1 in groups[r], r
        else:
            assert min(groups[r]) > 1, r
    for d, most in ((64, {2, 4}), (128, {2})):
        for causal in (0, 1):
            assert {g[causal] for r, g in groups.items() if r[4] == d} - {1} == most


def test_division_of_workgroup_ids(tmp_path):
    """The batched kernels' division by multiplication, exact for every divisor
    and n below 2^31: small divisors, powers of two and their neighbours, primes
    and the largest, at multiples of each and beside them."""
    out = query(tmp_path, "gemm_bf16.hip", r"""
  using namespace mx::gemm;
  const uint32_t top = 0x7fffffffu;
  long long checked = 0;
  auto test = [&](uint32_t d) {
    const Div v = make_div(d);
    auto at = [&](long long n) {
      if (n < 0 || n > top) return true;
      ++checked;
      return quot((uint32_t)n, v) == (uint32_t)n / d;
    };
    bool ok = true;
    for (long long q = 0; q < 40; ++q)
      for (long long m : {q * d, (long long)(top / d - q) * d, (long long)(top / d / (q + 2)) * d})
        ok = ok && at(m - 1) && at(m) && at(m + 1);
    return ok && at(top);
  };
  for (uint32_t d = 1; d <= 70000; ++d)
    if (!test(d)) { printf("wrong for %u\n", d); return 0; }
  for (int b = 0; b < 31; ++b)
    for (int e = -3; e <= 3; ++e) {
      const long long d = (1LL << b) + e;
      if (d >= 1 && d <= top && !test((uint32_t)d)) { printf("wrong for %lld\n", d); return 0; }
    }
  for (uint32_t d : {1000003u, 16777213u, 1073741789u, 2147483629u, 2147483646u, 2147483647u})
    if (!test(d)) { printf("wrong for %u\n", d); return 0; }
  printf("ok %d\n", checked > 10000000);""")
    assert out == ["ok 1"]
