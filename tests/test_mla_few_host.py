"""Row addressing of the MLA decode for up to 16 heads (host code, no GPU)."""
from __future__ import annotations

from host_query import query


def test_row_offsets_of_a_block(tmp_path):
    """Every row of a block, clamped to the sequence's last row, for sequences
    whose length in bytes lies around multiples of 2^32 and blocks all over
    them, the ones 2^32 bytes before the end among them."""
    out = query(tmp_path, "mla_decode_few.hip", r"""
  using namespace mx::mla;
  long long checked = 0;
  const long long wrap = (1LL << 32) / ROW_B;
  for (long long m = 0; m <= 5; ++m)
    for (long long d = -40; d <= 40; ++d) {
      const long long T = m * wrap + d;
      if (T < 1) continue;
      for (long long w = 0; w <= m; ++w)      // blocks w * 2^32 bytes before the end, from 40 tokens early to 40 late
        for (long long e = -40; e <= 40; ++e) {
          const long long tok0 = (T - 1 - w * wrap + e) / BT * BT;
          if (tok0 < 0 || tok0 >= T) continue;
          for (long long r = 0; r < BT; ++r) {
            const long long want = (r < T - 1 - tok0 ? r : T - 1 - tok0) * ROW_B;
            const uint32_t got = min((uint32_t)r * (uint32_t)ROW_B, last_row((int)T, (int)tok0));
            ++checked;
            if (got != want) {
              printf("T %lld block at %lld row %lld: offset %u, not %lld\n", T, tok0, r, got, want);
              return 0;
            }
          }
        }
    }
  printf("ok %d\n", checked > 100000);""")
    assert out == ["ok 1"]
