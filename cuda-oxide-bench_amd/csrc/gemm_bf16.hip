// bf16 GEMM for gfx950:  C[M,N] = A[M,K] · B[K,N], fp32 accumulate, bf16 out.
//
// Semantics follow cutile-matmul-tc-bf16/main.py:59-78 (bf16 x bf16 -> f32
// accumulator -> bf16 store, zero padding at ragged edges) and the bf16 row
// of cutile-matmul-tiled-mixed/main.py:121-130.
//
// The kernels (MI355X-first designs, not translations of the reference's
// cuTile/WMMA kernels) all compute D^T = B^T . A^T, so each lane holds runs
// of four consecutive n of one row of C; workgroup ids are remapped so that
// tiles sharing A rows / B columns run on the same XCD (own L2).  A and B go
// HBM -> LDS by direct loads into rings, and every kernel takes any K (a
// multiple of 8): the K % 64 tail is computed before the K loop, from a ring
// slot that the prologue leaves free.
//
// gemm_bf16_dma16s_kernel: 256x256 tiles, the large products.
// gemm_bf16_dma64_kernel: tiles of 64x64 to 128x192, single and batched;
// gemm_bf16_short_kernel: the smaller ones for K < 128.
// gemm_bf16_stream_kernel: few rows or few tiles; workgroups of 32 or 64
// columns x 32 or 64 rows stream B, their waves splitting K.
// gemm_bf16_smallm_kernel / gemm_bf16_smallm_sk_kernel (batched items of few
// rows): single-wave or K-split 4-wave workgroups over the whole K.
#include <type_traits>

#include "mx_common.h"

namespace mx {
namespace gemm {

constexpr int GROUP_M = 8;

// First row and column of this workgroup's C tile: tiles grouped for L2 reuse
// (GROUP_M tile rows share their columns of B), XCD-aware.
struct Origin {
  int m0, n0;
};
template <int BM, int BN>
__device__ __forceinline__ Origin tile_origin(int M, int N) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int id = xcd_remap(blockIdx.x, tiles_m * tiles_n);
  const int per_group = GROUP_M * tiles_n;
  const int group = id / per_group;
  const int first_m = group * GROUP_M;
  const int gsz = min(tiles_m - first_m, GROUP_M);
  const int tm = first_m + (id % per_group) % gsz;
  const int tn = (id % per_group) / gsz;
  return Origin{tm * BM, tn * BN};
}

// The interface's bound on the leading dimensions of shapes with K % 32 != 0,
// of small grids and of batched items with more than 32 rows: BM rows of A
// and 64 k-rows of B span less than 2^31 bytes.
template <int BM>
inline bool strides_2g(int lda, int ldb) {
  return (long long)lda * 2 * BM < 0x7ffffff0LL && (long long)ldb * 2 * 64 < 0x7ffffff0LL;
}

// A-row chunk swizzle of every kernel here: rows of 128 bytes, whose chunk c
// sits at c ^ swz_a(row).  A 16-lane ds_read_b128 phase reads one chunk of 16
// consecutive rows, which this puts in 16 distinct 16-byte slots of the 256-byte
// bank window.
__device__ __forceinline__ int swz_a(int m) { return (m >> 1) & 7; }

// Below this K a tile takes the whole K to LDS at once (gemm_bf16_short_kernel).
constexpr int kShortK = 128;

// s_waitcnt for "at most min(MAXC, after) chunks of LPC loads in flight".
template <int LPC, int MAXC>
__device__ __forceinline__ void wait_chunks(int after) {
  if constexpr (MAXC > 0) {
    if (after < MAXC) {
      wait_chunks<LPC, MAXC - 1>(after);
      return;
    }
  }
  wait_vmcnt<MAXC * LPC>();
}

// A fragment whose k values lie past K counts as zero on both sides, so
// whatever was loaded in their place (an infinity too) adds nothing.
__device__ __forceinline__ u32x4 keep_if(bool keep, const u32x4& x) { return keep ? x : u32x4{0, 0, 0, 0}; }

// ---------------------------------------------------------------------------
// gemm_bf16_dma64_kernel: tiles of up to 128 x 192 by direct loads, on
// 16x16x32 MFMAs.  Under a sustained full-chip MFMA load the 16x16x32 shape
// delivers about 11% more bf16 throughput than 32x32x16 on MI355X (same
// FLOPs, less operand/accumulator traffic per FLOP, so less power at the same
// clock cap).
//
//  * WM x WN waves, each owning (BM/WM) x (BN/WN) of C as 16x16 fragments.
//  * K advances in 64-deep stages, two k-steps each: a stage holds whole
//    128-byte lines of A, and there is one barrier per two k-steps.
//  * Operand layouts (16x16x32): the "A" operand holds 8 consecutive k of
//    row l%16 at k-group l/16; "B" the same for column l%16; D holds rows
//    4(l/16)..+3 of column l%16.  Issued as D^T = B^T . A^T: B^T fragments
//    come from the K-major B tile by transposing reads (lane (kg, j, a)
//    reads k-row 8kg + 4r + j, columns 4a..+3, r = 0, 1), A^T fragments are
//    one 16-byte read of an A row; each lane's D is four consecutive n of
//    one row of C.
//  * A rows are 128 B: chunk c ^ ((m >> 1) & 7) keeps the 16-lane phases of
//    the A^T reads on distinct bank slots.  B rows of 512 or 256 B start at
//    bank 0: a 32-lane phase of transposing reads covers 8 k-rows (two
//    k-groups x 4) of 32 bytes each, and chunk c ^ 2((k & 3) | ((k >> 3) & 1)
//    << 2) gives the 8 rows distinct 32-byte slots.  The direct loads apply
//    the same XOR on the global side.
//  * Ring of NS stages.  The next half's fragments are read during the
//    current half: B^T ones into the other half of a double buffer at its
//    start, each A^T one in place right after the MFMAs that consumed the
//    previous one's.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int swz_b16(int k) { return 2 * ((k & 3) | (((k >> 3) & 1) << 2)); }
template <int BM_, int BN_, int WM, int WN, int NS_>
struct D64Cfg {
  static constexpr int BM = BM_, BN = BN_, BK = 64, NS = NS_;
  static constexpr int NW = WM * WN, NT = 64 * NW;
  static constexpr int TM = BM / WM, TN = BN / WN;  // wave block
  static constexpr int FM = TM / 16, FN = TN / 16;  // 16x16 fragments
  static constexpr int RA = BK * 2, RB = BN * 2;    // LDS row bytes
  static constexpr int A_B = BM * RA, B_B = BK * RB;
  static constexpr int STAGE = A_B + B_B;
  static constexpr int A_L = A_B / 1024, A_RPL = 1024 / RA;  // direct loads of A per stage, A rows per load
  static constexpr int LPW = STAGE / 1024 / NW;              // 1 KB loads per wave per stage
  static_assert(NS >= 4 && NS * STAGE <= 160 * 1024, "LDS ring");
  static_assert((NS - 1) * LPW < 64, "vmcnt range");
  static_assert(STAGE % (1024 * NW) == 0 && TM % 16 == 0 && TN % 16 == 0, "tile split");
};
// Schedule of one K tile: per row block FN MFMAs, then LDS reads: the 2FN
// B^T reads spread over the first half of the row blocks, each A^T read
// right behind its row block.
template <int FM, int FN, int I = 0>
__device__ __forceinline__ void interleave_rows16() {
  if constexpr (I < FM) {
    constexpr int HB = FM / 2;
    constexpr int nb = I < HB ? (2 * FN * (I + 1)) / HB - (2 * FN * I) / HB : 0;
    __builtin_amdgcn_sched_group_barrier(0x008, FN, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1 + nb, 0);
    interleave_rows16<FM, FN, I + 1>();
  }
}
// B rows of 64 or 192 columns start at two bank phases (k even, odd), 128 B
// apart, so the four rows of each parity take the four 32-byte slots of an
// aligned 128 bytes.
template <int BN>
__device__ __forceinline__ int swz_b16n(int k) {
  static_assert(BN == 64 || BN == 128 || BN == 192 || BN == 256, "row size");
  return BN == 64 || BN == 192 ? 2 * (((k >> 1) & 1) | (((k >> 3) & 1) << 1)) : swz_b16(k);
}

// Steps I .. NS-1 of a period of the K loop: stage I.
template <int NS, int I = 0, typename Step>
__device__ __forceinline__ void step_period(Step& step, int kt) {
  if constexpr (I < NS) {
    step(kt + I, std::integral_constant<int, I>{});
    step_period<NS, I + 1>(step, kt);
  }
}
// The first n (< NS) steps of a period, for the tail of the K loop.
template <int NS, int I = 0, typename Step>
__device__ __forceinline__ void step_tail(Step& step, int kt, int n) {
  if constexpr (I < NS - 1) {
    if (I < n) {
      step(kt + I, std::integral_constant<int, I>{});
      step_tail<NS, I + 1>(step, kt, n);
    }
  }
}

// Store a C tile through LDS: the tile goes there as bf16 rows (padded by 16
// bytes) and is stored as whole rows, each lane 16 contiguous bytes, instead
// of 8-byte pieces that the memory system writes back as partial lines.  The
// lane holds rows am + 16 mf, columns cn + 16 nf .. +3; the LDS is free once
// every wave is past its last fragment reads.
template <int BM, int BN, int NT, int FM, int FN>
__device__ __forceinline__ void store_tile_lds(unsigned char* smem, const f32x4 (&acc)[FM][FN], int am, int cn,
                                               uint16_t* C, int m0, int n0, int M, int N, int ldc) {
  constexpr int CROW = BN * 2 + 16;
  __syncthreads();
#pragma unroll
  for (int mf = 0; mf < FM; ++mf) {
    const int r = am + 16 * mf;
#pragma unroll
    for (int nf = 0; nf < FN; ++nf) {
      const f32x4& a = acc[mf][nf];
      *reinterpret_cast<u32x2*>(smem + r * CROW + 2 * (cn + 16 * nf)) =
          u32x2{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3])};
    }
  }
  __syncthreads();
  constexpr int CPR = BN / 8;  // 16-byte chunks per tile row
  constexpr int CH = BM * CPR;
  static_assert(CH % NT == 0, "whole passes");
  if constexpr (NT % CPR == 0) {
    constexpr int RPI = NT / CPR;  // rows per workgroup-wide store
    const int t = threadIdx.x;
    const int cc = t % CPR, r0 = t / CPR;
    const int gn = n0 + 8 * cc;
#pragma unroll 4
    for (int r = r0; r < BM; r += RPI) {
      const int gm = m0 + r;
      if (gm < M && gn < N)
        st128(C + (size_t)gm * ldc + gn, *reinterpret_cast<const u32x4*>(smem + r * CROW + 16 * cc));
    }
  } else {
#pragma unroll 4
    for (int q = threadIdx.x; q < CH; q += NT) {
      const int r = q / CPR, cc = q % CPR;
      const int gm = m0 + r, gn = n0 + 8 * cc;
      if (gm < M && gn < N)
        st128(C + (size_t)gm * ldc + gn, *reinterpret_cast<const u32x4*>(smem + r * CROW + 16 * cc));
    }
  }
}

template <int BM_, int BN_, int WM_, int WN_, int NS_, bool TAIL>
__global__ __launch_bounds__(64 * WM_ * WN_, 1) void gemm_bf16_dma64_kernel(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, uint16_t* __restrict__ C, int M, int N, int K,
    int lda, int ldb, int ldc, long long sA, long long sB, long long sC) {
  using CF = D64Cfg<BM_, BN_, WM_, WN_, NS_>;
  constexpr int NS = CF::NS, FM = CF::FM, FN = CF::FN, BK = CF::BK;
  extern __shared__ __align__(1024) unsigned char smem[];
  A += (size_t)blockIdx.y * sA;
  B += (size_t)blockIdx.y * sB;
  C += (size_t)blockIdx.y * sC;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN_, wn = wave % WN_;
  const int kg = lane >> 4;  // k-group of the lane's operand and row quad of its result

  const Origin org = tile_origin<CF::BM, CF::BN>(M, N);
  const int m0 = org.m0, n0 = org.n0;
  const int nk = K / BK;

  // ---- direct loads: load ld = wave * LPW + n of a stage fills its bytes
  // 1024 ld .. +1023 (A rows, then B k-rows).  Rows past M / columns past N
  // re-read the last valid ones; their results are never stored. ----
  const uint32_t lds0 = lds_addr(smem);
  uint32_t off[CF::LPW];
#pragma unroll
  for (int n = 0; n < CF::LPW; ++n) {
    const int ld = wave * CF::LPW + n;
    if (ld < CF::A_L) {
      const int row = CF::A_RPL * ld + lane / 8;
      off[n] = (uint32_t)(min(m0 + row, M - 1) - m0) * (uint32_t)lda * 2u + 16u * ((lane % 8) ^ swz_a(row));
    } else {
      const int byte = 1024 * (ld - CF::A_L) + 16 * lane;
      const int row = byte / CF::RB;
      const int col = 8 * (((byte % CF::RB) / 16) ^ swz_b16n<CF::BN>(row));  // elements
      off[n] = (uint32_t)row * (uint32_t)ldb * 2u + 2u * (min(n0 + col, N - 8) - n0);
    }
  }
  auto issue = [&](int kt, int stage) {
    const uint32_t st = lds0 + stage * CF::STAGE;
    const uint16_t* abase = A + (size_t)m0 * lda + (size_t)kt * BK;
    const uint16_t* bbase = B + (size_t)kt * BK * ldb + n0;
#pragma unroll
    for (int n = 0; n < CF::LPW; ++n) {
      const int ld = wave * CF::LPW + n;
      dma16(ld < CF::A_L ? abase : bbase, off[n], st + ld * 1024);
    }
  };

  // ---- fragment lane addresses, one base per ring stage (stages lie past
  // ds_read's 16-bit immediate), fragments at immediates from it ----
  // A^T (B operand): row am + 16 mf, chunk (4 h + kg) ^ swz(am) (swz is the
  // same for every mf).
  const int am = wm * CF::TM + (lane & 15);
  uint32_t a_col[NS][2];
#pragma unroll
  for (int st = 0; st < NS; ++st)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      a_col[st][h] = lds0 + st * CF::STAGE + am * CF::RA + 16 * ((4 * h + kg) ^ swz_a(am));
      asm volatile("" : "+v"(a_col[st][h]));  // keep it a base register
    }
  // B^T (A operand): lane (kg, j, a) reads k-rows 32h + 8kg + 4r + j, columns
  // wn*TN + 16 nf + 4a .. +3 (8 bytes of a 16-byte chunk).
  const int b_j = (lane >> 2) & 3, b_a = lane & 3;
  const int bk = 8 * kg + b_j;  // k-row of the r = 0 read; rows 4 and 32 further share its swizzle
  uint32_t b_col[NS][FN];
#pragma unroll
  for (int st = 0; st < NS; ++st)
#pragma unroll
    for (int nf = 0; nf < FN; ++nf) {
      const int chunk = (wn * CF::TN + 16 * nf + 4 * b_a) >> 3;
      b_col[st][nf] =
          lds0 + st * CF::STAGE + CF::A_B + bk * CF::RB + 16 * (chunk ^ swz_b16n<CF::BN>(bk)) + 8 * (b_a & 1);
      asm volatile("" : "+v"(b_col[st][nf]));
    }

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{};

  u32x4 af[FM];     // A^T fragments of the current half, refilled in place
  u32x4 bf[2][FN];  // B^T fragments of the stage's two halves
  auto read_b = [&](int stg, int h) {
#pragma unroll
    for (int nf = 0; nf < FN; ++nf) {
      const u32x2 lo = lds_read_tr16_at(b_col[stg][nf] + 32 * h * CF::RB);
      const u32x2 hi = lds_read_tr16_at(b_col[stg][nf] + (32 * h + 4) * CF::RB);
      bf[h][nf] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  };
  auto read_a = [&](int stg, int h, int mf) { af[mf] = lds_ld128(a_col[stg][h] + 16 * mf * CF::RA); };
  // the MFMAs of one half, whose fragments are in af and bf[h], while the
  // fragments of half nh of stage nstg are read
  auto half = [&](int h, int nstg, int nh) {
    __builtin_amdgcn_sched_barrier(0);
    read_b(nstg, nh);
#pragma unroll
    for (int mf = 0; mf < FM; ++mf) {
#pragma unroll
      for (int nf = 0; nf < FN; ++nf) acc[mf][nf] = mfma16<BF16>(bf[h][nf], af[mf], acc[mf][nf]);
      read_a(nstg, nh, mf);
    }
    interleave_rows16<FM, FN>();
    __builtin_amdgcn_sched_barrier(0);
  };

  // One K tile: the fragments of its first half are in af and bf[0].
  auto step = [&](int kt, auto stg_tag) {
    constexpr int STG = decltype(stg_tag)::value;
    constexpr int NXT = (STG + 1) % NS;
    half(0, STG, 1);
    // This wave's loads of tile kt+1 have landed (at most the NS-3 tiles
    // issued after it, fewer near the end, are in flight): after the barrier
    // tile kt+1 is readable, and stage (kt-1)%NS, whose last reads every wave
    // waited for before its first half's MFMAs, takes tile kt+NS-1.  After
    // the last tile the reads for a next one get stale fragments nobody uses.
    wait_chunks<CF::LPW, NS - 3>(nk - 2 - kt);
    lds_barrier();
    if (kt + NS - 1 < nk) issue(kt + NS - 1, (STG + NS - 1) % NS);
    half(1, NXT, 0);
  };

  land_args(C);  // C is used only after the K loop
  // The K % 64 tail is computed first, from stage NS-1, which the ring fills
  // only after step 0's barrier: its loads share the prologue's latency
  // instead of adding a round trip at the end.  Chunks and k-rows past K
  // re-read the last valid ones or are left out, and so is the second half of
  // the stage when K ends in the first.
  if constexpr (TAIL) {
    const int kr = K - nk * BK;
    const uint32_t st = lds0 + (NS - 1) * CF::STAGE;
    const uint16_t* abase = A + (size_t)m0 * lda + (size_t)nk * BK;
    const uint16_t* bbase = B + (size_t)nk * BK * ldb + n0;
#pragma unroll
    for (int n = 0; n < CF::LPW; ++n) {
      const int ld = wave * CF::LPW + n;
      if (ld < CF::A_L) {
        const uint32_t swz = 16u * ((lane % 8) ^ swz_a(CF::A_RPL * ld + lane / 8));
        dma16(abase, off[n] - swz + min(swz, (uint32_t)(2 * kr - 16)), st + ld * 1024);
      } else {
        const int row = (1024 * (ld - CF::A_L) + 16 * lane) / CF::RB;
        if (1024 * (ld - CF::A_L) / CF::RB < kr)
          dma16(bbase, off[n] - (uint32_t)(row - min(row, kr - 1)) * (uint32_t)ldb * 2u, st + ld * 1024);
      }
    }
  }
  // Prologue: tiles 0 .. NS-2 in flight (two at least: K >= 128), wait for
  // tile 0, read its fragments.
#pragma unroll
  for (int p = 0; p < NS - 1; ++p)
    if (p < 2 || p < nk) issue(p, p);
  if constexpr (TAIL) {
    wait_chunks<CF::LPW, NS - 1>(nk);
    lds_barrier();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (32 * h >= K - nk * BK) break;
      const bool keep = 32 * h + 8 * kg < K - nk * BK;
      read_b(NS - 1, h);
#pragma unroll
      for (int nf = 0; nf < FN; ++nf) bf[h][nf] = keep_if(keep, bf[h][nf]);
#pragma unroll
      for (int mf = 0; mf < FM; ++mf) {
        read_a(NS - 1, h, mf);
        af[mf] = keep_if(keep, af[mf]);
#pragma unroll
        for (int nf = 0; nf < FN; ++nf) acc[mf][nf] = mfma16<BF16>(bf[h][nf], af[mf], acc[mf][nf]);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the stage's reads are done before the next barrier frees it
  }
  wait_chunks<CF::LPW, NS - 2>(nk - 1);
  lds_barrier();
  read_b(0, 0);
#pragma unroll
  for (int mf = 0; mf < FM; ++mf) read_a(0, 0, mf);
  int kt = 0;
  for (; kt + NS <= nk; kt += NS) step_period<NS>(step, kt);
  step_tail<NS>(step, kt, nk - kt);
  wait_vmcnt<0>();  // no DMA may land in LDS after the workgroup ends

  // ---- epilogue: lane holds m = am + 16 mf, n = wn*TN + 16 nf + 4 kg + {0..3}
  // of the tile ----
  store_tile_lds<CF::BM, CF::BN, CF::NT, FM, FN>(smem, acc, am, wn * CF::TN + 4 * kg, C, m0, n0, M, N, ldc);
}

// ---------------------------------------------------------------------------
// gemm_bf16_short_kernel: the tiles of the kernel above for K < 128, which it
// would spend in its prologue: its ring leaves room for one or two workgroups
// per CU, and its constant waits load the last K tile again into every stage
// that has none of its own.  Here the whole K goes to LDS at once (one wait,
// one barrier, then fragments and MFMAs without another), only what the
// product has of it (no k-rows past K, no rows past M in blocks of eight), in
// one or two stages, so that the workgroups of a CU hide each other's loads
// and stores.  What bounds it is the C tiles' way to memory, or a launch.
// Ring -> this, same tile choice aside: 8192x8192x32 68.6 -> 23.8 us,
// 16121x1672x8 32.1 -> 19, 170 items of 3x992x40 13.7 -> 8.6.  From K = 128 on
// the ring is the faster one (64x64 tiles: by 8% at 128, 16% at 200 to 256).
// ---------------------------------------------------------------------------
template <int BM_, int BN_, int WM_, int WN_>
__global__ __launch_bounds__(64 * WM_ * WN_) void gemm_bf16_short_kernel(
    const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, uint16_t* __restrict__ C, int M, int N, int K,
    int lda, int ldb, int ldc, long long sA, long long sB, long long sC) {
  using CF = D64Cfg<BM_, BN_, WM_, WN_, 4>;
  constexpr int FM = CF::FM, FN = CF::FN, BK = CF::BK;
  extern __shared__ __align__(1024) unsigned char smem[];
  A += (size_t)blockIdx.y * sA;
  B += (size_t)blockIdx.y * sB;
  C += (size_t)blockIdx.y * sC;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN_, wn = wave % WN_;
  const int kg = lane >> 4;
  const Origin org = tile_origin<CF::BM, CF::BN>(M, N);
  const int m0 = org.m0, n0 = org.n0;
  const uint32_t lds0 = lds_addr(smem);

  // ---- direct loads, laid out as in the kernel above.  Loads without a row of
  // the product are left out: what LDS holds there reaches only results that
  // are not stored, and k values that are set to zero. ----
  for (int k0 = 0, st = lds0; k0 < K; k0 += BK, st += CF::STAGE) {
    const int kr = min(K - k0, BK);
    const uint16_t* abase = A + (size_t)m0 * lda + k0;
    const uint16_t* bbase = B + (size_t)k0 * ldb + n0;
#pragma unroll
    for (int n = 0; n < CF::LPW; ++n) {
      const int ld = wave * CF::LPW + n;
      if (ld < CF::A_L) {
        const int row = CF::A_RPL * ld + lane / 8;
        const int chunk = min(8 * ((lane % 8) ^ swz_a(row)), kr - 8);  // elements
        if (CF::A_RPL * ld < M - m0)
          dma16(abase, (uint32_t)(min(m0 + row, M - 1) - m0) * (uint32_t)lda * 2u + 2u * chunk, st + ld * 1024);
      } else {
        const int byte = 1024 * (ld - CF::A_L) + 16 * lane;
        const int row = byte / CF::RB;
        const int col = 8 * (((byte % CF::RB) / 16) ^ swz_b16n<CF::BN>(row));
        if (1024 * (ld - CF::A_L) / CF::RB < kr)
          dma16(bbase, (uint32_t)min(row, kr - 1) * (uint32_t)ldb * 2u + 2u * (min(n0 + col, N - 8) - n0),
                st + ld * 1024);
      }
    }
  }

  // Fragment lane addresses of the first half, as in the kernel above; the
  // second half of a stage is 64 bytes (one bit) across in A and 32 k-rows on
  // in B.
  const int am = wm * CF::TM + (lane & 15);
  uint32_t a_col = lds0 + am * CF::RA + 16 * (kg ^ swz_a(am));
  const int b_j = (lane >> 2) & 3, b_a = lane & 3;
  const int bk = 8 * kg + b_j;
  uint32_t b_col[FN];
#pragma unroll
  for (int nf = 0; nf < FN; ++nf) {
    const int chunk = (wn * CF::TN + 16 * nf + 4 * b_a) >> 3;
    b_col[nf] = lds0 + CF::A_B + bk * CF::RB + 16 * (chunk ^ swz_b16n<CF::BN>(bk)) + 8 * (b_a & 1);
  }

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{};

  land_args(C);
  wait_vmcnt<0>();
  lds_barrier();
  // A loop and not unrolled further: the kernel's code is fetched anew for
  // every short launch.
#pragma unroll 1
  for (int k0 = 0, so = 0; k0 < K; k0 += 32) {
    const bool keep = k0 + 8 * kg < K;
    u32x4 bf[FN], af[FM];
#pragma unroll
    for (int nf = 0; nf < FN; ++nf) {
      const u32x2 lo = lds_read_tr16_at(b_col[nf] + so);
      const u32x2 hi = lds_read_tr16_at(b_col[nf] + so + 4 * CF::RB);
      bf[nf] = keep_if(keep, u32x4{lo[0], lo[1], hi[0], hi[1]});
    }
#pragma unroll
    for (int mf = 0; mf < FM; ++mf) af[mf] = keep_if(keep, lds_ld128(a_col + 16 * mf * CF::RA));
#pragma unroll
    for (int mf = 0; mf < FM; ++mf)
#pragma unroll
      for (int nf = 0; nf < FN; ++nf) acc[mf][nf] = mfma16<BF16>(bf[nf], af[mf], acc[mf][nf]);
    const bool second = k0 & 32;
    a_col = (a_col ^ 64) + (second ? CF::STAGE : 0);
    so += second ? CF::STAGE - 32 * CF::RB : 32 * CF::RB;
  }
  // 64 rows per tile are taken for small grids, where the way of the C tile
  // through LDS is latency (10 items of 62x8x40: 2.85 us, 3.0 through LDS).
  if constexpr (BM_ == 64) {
#pragma unroll
    for (int mf = 0; mf < FM; ++mf) {
      const int gm = m0 + am + 16 * mf;
#pragma unroll
      for (int nf = 0; nf < FN; ++nf) {
        const int gn = n0 + wn * CF::TN + 16 * nf + 4 * kg;
        const f32x4& a = acc[mf][nf];
        if (gm < M && gn < N) st64(C + (size_t)gm * ldc + gn, u32x2{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3])});
      }
    }
  } else {
    store_tile_lds<CF::BM, CF::BN, CF::NT, FM, FN>(smem, acc, am, wn * CF::TN + 4 * kg, C, m0, n0, M, N, ldc);
  }
}

template <int BM, int BN, int WM, int WN>
static int launch_short(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc,
                        hipStream_t stream, int batch, long long sA, long long sB, long long sC) {
  using CF = D64Cfg<BM, BN, WM, WN, 4>;
  const long long tiles = (long long)((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  if (tiles > 0x7fffffffLL || batch > 65535) return MX_ERR_SHAPE;
  constexpr auto kern = gemm_bf16_short_kernel<BM, BN, WM, WN>;
  constexpr int c_tile = BM == 64 ? 0 : BM * (BN * 2 + 16), most = kShortK / CF::BK * CF::STAGE;
  MX_RETURN_IF_HIP(lds_limit_once<kern>(most > c_tile ? most : c_tile));
  const int stages = (K + CF::BK - 1) / CF::BK * CF::STAGE;
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)batch), dim3(CF::NT), stages > c_tile ? stages : c_tile,
                     stream, (const uint16_t*)A, (const uint16_t*)B, (uint16_t*)C, M, N, K, lda, ldb, ldc, sA, sB, sC);
  MX_RETURN_IF_HIP(hipGetLastError());
  return MX_OK;
}

template <int BM, int BN, int WM, int WN, int NS>
static int launch_dma64(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc,
                        hipStream_t stream, int batch = 1, long long sA = 0, long long sB = 0, long long sC = 0) {
  using CF = D64Cfg<BM, BN, WM, WN, NS>;
  const long long tiles = (long long)((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  if (tiles > 0x7fffffffLL || batch > 65535) return MX_ERR_SHAPE;
  auto go = [&](auto tail) {
    constexpr auto kern = gemm_bf16_dma64_kernel<BM, BN, WM, WN, NS, decltype(tail)::value>;
    MX_RETURN_IF_HIP(lds_limit_once<kern>(NS * CF::STAGE));
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)batch), dim3(CF::NT), NS * CF::STAGE, stream,
                       (const uint16_t*)A, (const uint16_t*)B, (uint16_t*)C, M, N, K, lda, ldb, ldc, sA, sB, sC);
    MX_RETURN_IF_HIP(hipGetLastError());
    return MX_OK;
  };
  return K % CF::BK ? go(std::true_type{}) : go(std::false_type{});
}

// ---------------------------------------------------------------------------
// gemm_bf16_dma16s_kernel: 256x256 tiles, eight waves of 128x64 on 16x16x32
// MFMAs, the fragments of the next 32-deep K tile read during the current one's
// MFMAs as in the kernel above.  A single ring of 32-deep stages would hold 64
// bytes of each A row and fetch every 128-byte line of A as two half-line
// requests, which hold up the L1's address unit; 64-deep stages of both would
// leave room for two.  So A goes through its own ring of 64-deep blocks (256
// rows x 128 B, 3 slots) beside a ring of 32-deep B stages (32 k-rows x 512 B,
// 4 slots), 160 KB in all:
//  * step kt computes K tile kt (B stage kt, half kt % 2 of A block kt / 2)
//    and reads tile kt+1's fragments; it issues B stage kt+3 and half kt % 2
//    of A block kt/2 + 2, each into the slot of the stage / block that the
//    barrier just freed, so every step issues the same 4 loads per wave and
//    waits for all but the 4 of the step before.
//  * A rows (128 B) and B rows (512 B) are swizzled by swz_a and swz_b16.
// Shapes: any K of at least 64.  The K % 64 tail is computed before the K loop,
// from A slot 2 and B slots 3 and 2.
// ---------------------------------------------------------------------------
struct S16Cfg {
  static constexpr int BM = 256, BN = 256, BK = 32, BKA = 64;
  static constexpr int WM = 2, WN = 4, NW = WM * WN, NT = 64 * NW;
  static constexpr int TM = BM / WM, TN = BN / WN;   // wave block
  static constexpr int FM = TM / 16, FN = TN / 16;   // 16x16 fragments
  static constexpr int RA = BKA * 2, RB = BN * 2;    // LDS row bytes (A 128, B 512)
  static constexpr int A_B = BM * RA, B_B = BK * RB;  // A block 32 KB, B stage 16 KB
  static constexpr int NSA = 3, NSB = 4;
  static constexpr int B_OFF = NSA * A_B;
  static constexpr int LDS = NSA * A_B + NSB * B_B;
  static constexpr int A_LPW = A_B / 1024 / NW;      // 1 KB loads per wave per A block
  static constexpr int B_LPW = B_B / 1024 / NW;      // ... per B stage
  static constexpr int A_RPL = 1024 / RA;            // A rows per load
  static constexpr int B_CH = RB / 16, B_RPL = 1024 / RB;
  static constexpr int VM = B_LPW + A_LPW / 2;       // loads per step and wave
  static constexpr int P = 12;                        // steps until slots and parity repeat
  static_assert(LDS <= 160 * 1024 && A_LPW % 2 == 0 && A_LPW >= 2 && B_LPW >= 1, "rings");
};

template <bool TAIL>
__global__ __launch_bounds__(S16Cfg::NT, 1) void gemm_bf16_dma16s_kernel(const uint16_t* __restrict__ A,
                                                                        const uint16_t* __restrict__ B,
                                                                        uint16_t* __restrict__ C, int M, int N,
                                                                        int K, int lda, int ldb, int ldc) {
  using CF = S16Cfg;
  constexpr int FM = CF::FM, FN = CF::FN, BK = CF::BK, WN = CF::WN;
  extern __shared__ __align__(1024) unsigned char smem[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int kg = lane >> 4;  // k-group of the lane's operand and row quad of its result

  const Origin org = tile_origin<CF::BM, CF::BN>(M, N);
  const int m0 = org.m0, n0 = org.n0;
  const int nka = K / CF::BKA, nk = 2 * nka;

  // ---- direct-load lane offsets (bytes from the tile's first element).
  // Rows past M / columns past N re-read the last valid ones; their
  // results are never stored. ----
  const uint32_t lds0 = lds_addr(smem);
  const bool full_m = m0 + CF::BM <= M, full_n = n0 + CF::BN <= N;
  uint32_t a_off[CF::A_LPW], b_off[CF::B_LPW];
#pragma unroll
  for (int n = 0; n < CF::A_LPW; ++n) {
    const int row = CF::A_RPL * (wave * CF::A_LPW + n) + lane / 8;
    const int gm = full_m ? m0 + row : min(m0 + row, M - 1);
    a_off[n] = (uint32_t)(gm - m0) * (uint32_t)lda * 2u + 16u * ((lane % 8) ^ swz_a(row));
  }
#pragma unroll
  for (int n = 0; n < CF::B_LPW; ++n) {
    const int row = CF::B_RPL * (wave * CF::B_LPW + n) + lane / CF::B_CH;
    int col = 8 * ((lane % CF::B_CH) ^ swz_b16(row));  // elements
    if (!full_n) col = min(n0 + col, N - 8) - n0;
    b_off[n] = (uint32_t)row * (uint32_t)ldb * 2u + 2u * col;
  }
  // B stage s into B slot s % NSB; half h of A block j into A slot j % NSA.
  // Stages and blocks past the end re-load the last one (into slots no
  // later step reads).
  auto issue_b = [&](int s, int slot) {
    const uint16_t* bbase = B + (size_t)min(s, nk - 1) * BK * ldb + n0;
#pragma unroll
    for (int n = 0; n < CF::B_LPW; ++n)
      dma16(bbase, b_off[n], lds0 + CF::B_OFF + slot * CF::B_B + (wave * CF::B_LPW + n) * 1024);
  };
  auto issue_a = [&](int j, int h, int slot) {
    const uint16_t* abase = A + (size_t)m0 * lda + (size_t)min(j, nka - 1) * CF::BKA;
#pragma unroll
    for (int n = h * CF::A_LPW / 2; n < (h + 1) * CF::A_LPW / 2; ++n)
      dma16(abase, a_off[n], lds0 + slot * CF::A_B + (wave * CF::A_LPW + n) * 1024);
  };

  // ---- fragment lane addresses: one base per A slot and K half, and per
  // B slot and column fragment (slots lie past ds_read's 16-bit immediate) ----
  // A^T (B operand): row am + 16 mf, chunk (4 h + kg) ^ swz(am) (swz is the
  // same for every mf, 16 rows apart).
  const int am = wm * CF::TM + (lane & 15);
  uint32_t a_col[CF::NSA][2];
#pragma unroll
  for (int st = 0; st < CF::NSA; ++st)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      a_col[st][h] = lds0 + st * CF::A_B + am * CF::RA + 16 * ((4 * h + kg) ^ swz_a(am));
      asm volatile("" : "+v"(a_col[st][h]));  // keep it a base register
    }
  // B^T (A operand): lane (kg, j, a) reads k-rows 8kg + 4r + j, columns
  // wn*TN + 16 nf + 4a .. +3 (8 bytes of a 16-byte chunk).
  const int b_j = (lane >> 2) & 3, b_a = lane & 3;
  const int bk = 8 * kg + b_j;
  uint32_t b_col[CF::NSB][FN];
#pragma unroll
  for (int st = 0; st < CF::NSB; ++st)
#pragma unroll
    for (int nf = 0; nf < FN; ++nf) {
      const int chunk = (wn * CF::TN + 16 * nf + 4 * b_a) >> 3;
      b_col[st][nf] = lds0 + CF::B_OFF + st * CF::B_B + bk * CF::RB + 16 * (chunk ^ swz_b16(bk)) + 8 * (b_a & 1);
      asm volatile("" : "+v"(b_col[st][nf]));
    }

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{};

  u32x4 af[FM];     // A^T fragments of the current tile, refilled in place
  u32x4 bf[2][FN];  // B^T fragments, double buffered by tile parity
  auto read_b = [&](int stg, int buf) {
#pragma unroll
    for (int nf = 0; nf < FN; ++nf) {
      const u32x2 lo = lds_read_tr16_at(b_col[stg][nf]);
      const u32x2 hi = lds_read_tr16_at(b_col[stg][nf] + 4 * CF::RB);
      bf[buf][nf] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  };
  auto read_a = [&](int stg, int h, int mf) { af[mf] = lds_ld128(a_col[stg][h] + 16 * mf * CF::RA); };

  // Step kt = 12q + I: tile kt's fragments are in af and bf[I % 2]; B
  // stage kt sits in slot I % 4 and A block kt / 2 in slot (I / 2) % 3.
  auto step = [&](int kt, auto i_tag) {
    constexpr int I = decltype(i_tag)::value;
    constexpr int PAR = I % 2;
    constexpr int NB = (I + 1) % CF::NSB, NA = ((I + 1) / 2) % CF::NSA, NH = (I + 1) % 2;
    // Every wave has read tile kt (during step kt-1) and its own loads up
    // to those of step kt-2 have landed, tile kt+1's among them: after the
    // barrier tile kt+1 is readable, and B stage kt-1 (read during step
    // kt-2) and A block kt/2 - 1 (its last tile read no later) are free.
    wait_vmcnt<CF::VM>();
    lds_barrier();
    issue_b(kt + 3, (I + 3) % CF::NSB);
    issue_a(kt / 2 + 2, I % 2, (I / 2 + 2) % CF::NSA);
    __builtin_amdgcn_sched_barrier(0);
    read_b(NB, PAR ^ 1);
#pragma unroll
    for (int mf = 0; mf < FM; ++mf) {
#pragma unroll
      for (int nf = 0; nf < FN; ++nf) acc[mf][nf] = mfma16<BF16>(bf[PAR][nf], af[mf], acc[mf][nf]);
      read_a(NA, NH, mf);
    }
    interleave_rows16<FM, FN>();
    __builtin_amdgcn_sched_barrier(0);
  };

  land_args(C);  // C is used only after the K loop
  // The K % 64 tail is computed first, from A slot 2 and B slots 3 and 2,
  // which are free until then: its loads share the prologue's latency
  // instead of adding a round trip at the end.  Chunks and k-rows past K
  // re-read the last valid ones.
  const int kr = K - nka * CF::BKA;
  if constexpr (TAIL) {
    const uint16_t* abase = A + (size_t)m0 * lda + (size_t)nka * CF::BKA;
    const uint16_t* bbase = B + (size_t)nka * CF::BKA * ldb + n0;
#pragma unroll
    for (int n = 0; n < CF::A_LPW; ++n) {
      const uint32_t swz = 16u * ((lane % 8) ^ swz_a(CF::A_RPL * (wave * CF::A_LPW + n) + lane / 8));
      dma16(abase, a_off[n] - swz + min(swz, (uint32_t)(2 * kr - 16)), lds0 + 2 * CF::A_B + (wave * CF::A_LPW + n) * 1024);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (32 * h >= kr) break;
#pragma unroll
      for (int n = 0; n < CF::B_LPW; ++n) {
        const int row = CF::B_RPL * (wave * CF::B_LPW + n) + lane / CF::B_CH;
        dma16(bbase + (size_t)32 * h * ldb, b_off[n] - (uint32_t)(row - min(row, kr - 1 - 32 * h)) * (uint32_t)ldb * 2u,
              lds0 + CF::B_OFF + (3 - h) * CF::B_B + (wave * CF::B_LPW + n) * 1024);
      }
    }
  }
  // Prologue, in the order the waits need: A block 0, B stages 0 and 1,
  // A block 1, B stage 2; then tile 0's fragments.
  issue_a(0, 0, 0);
  issue_a(0, 1, 0);
  issue_b(0, 0);
  issue_b(1, 1);
  issue_a(1, 0, 1);
  issue_a(1, 1, 1);
  if constexpr (TAIL) {
    wait_vmcnt<2 * CF::A_LPW + 2 * CF::B_LPW>();  // all but A blocks 0, 1 and B stages 0, 1
    lds_barrier();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (32 * h >= kr) break;
      const bool keep = 32 * h + 8 * kg < kr;
      read_b(3 - h, h);
#pragma unroll
      for (int nf = 0; nf < FN; ++nf) bf[h][nf] = keep_if(keep, bf[h][nf]);
#pragma unroll
      for (int mf = 0; mf < FM; ++mf) {
        read_a(2, h, mf);
        af[mf] = keep_if(keep, af[mf]);
#pragma unroll
        for (int nf = 0; nf < FN; ++nf) acc[mf][nf] = mfma16<BF16>(bf[h][nf], af[mf], acc[mf][nf]);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slots' reads are done before B stage 2 and step 0 refill them
    lds_barrier();
  }
  issue_b(2, 2);
  wait_vmcnt<2 * CF::B_LPW + CF::A_LPW>();  // B stage 1, A block 1 and B stage 2 may be in flight
  lds_barrier();
  read_b(0, 0);
#pragma unroll
  for (int mf = 0; mf < FM; ++mf) read_a(0, 0, mf);
  int kt = 0;
  for (; kt + CF::P <= nk; kt += CF::P) step_period<CF::P>(step, kt);
  step_tail<CF::P>(step, kt, nk - kt);
  wait_vmcnt<0>();  // no DMA may land in LDS after the workgroup ends

  // ---- epilogue: lane holds m = am + 16 mf, n = wn*TN + 16 nf + 4 kg + {0..3} ----
  static_assert(CF::BM * (CF::BN * 2 + 16) <= CF::LDS, "C tile fits the rings");
  store_tile_lds<CF::BM, CF::BN, CF::NT, FM, FN>(smem, acc, am, wn * CF::TN + 4 * kg, C, m0, n0, M, N, ldc);
}

static int launch_dma16s(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc,
                         hipStream_t stream) {
  using CF = S16Cfg;
  const long long tiles = (long long)((M + CF::BM - 1) / CF::BM) * ((N + CF::BN - 1) / CF::BN);
  if (tiles > 0x7fffffffLL) return MX_ERR_SHAPE;
  auto go = [&](auto tail) {
    constexpr auto kern = gemm_bf16_dma16s_kernel<decltype(tail)::value>;
    MX_RETURN_IF_HIP(lds_limit_once<kern>(CF::LDS));
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(CF::NT), CF::LDS, stream, (const uint16_t*)A,
                       (const uint16_t*)B, (uint16_t*)C, M, N, K, lda, ldb, ldc);
    MX_RETURN_IF_HIP(hipGetLastError());
    return MX_OK;
  };
  return K % CF::BKA ? go(std::true_type{}) : go(std::false_type{});
}

// ---------------------------------------------------------------------------
// Small-M batched kernel (e.g. one decode batch against one head's weight; M >
// 32 in chunks of 32 rows): weight-streaming, so it needs enough bytes in flight per CU and
// few rounds of workgroups rather than big tiles.  A workgroup is one wave
// computing a 32 x (32 NF) tile of C over the whole K; 64-deep chunks of A
// [32][64] and B [64][32 NF] go HBM -> LDS by direct loads into an
// NS-stage ring, NS-1 chunks ahead (6 stages for narrow tiles, 4 at NF = 4:
// 48-80 KB of LDS, two workgroups per CU).  A single wave needs no barrier: the ring stage
// it overwrites was consumed by its own MFMAs, which waited for those
// reads.  With three and more chunks of K an item's row chunks and column tiles
// run on one XCD, whose L2 then holds its A and B once (64 items of 32 x 128 x
// 512 6.33 -> 4.31 us, 19 of 3 x 920 x 1024 17.4 -> 9.6); with one or two that
// gains nothing, and the plain order is the faster one (182 items of 2 x 512 x
// 128 7.5 us against 8.8).  A rows (128 B) use the 16-row chunk swizzle of the large kernel;
// B rows (64 NF bytes) put chunk c of k-row k at c ^ (((k & 3) << 2) mod
// (4 NF)) so the 4 consecutive k-rows of a transposing read phase occupy
// distinct 64-byte quarters of the bank sweep (no swizzle needed at NF = 1,
// where those 4 rows are 256 contiguous bytes).
// ---------------------------------------------------------------------------
constexpr int SM_BK = 64;
constexpr int SM_A_B = 32 * SM_BK * 2;  // 4 KB

template <int NF>
__device__ __forceinline__ int sm_swz(int k) {
  return NF == 1 ? 0 : (((k & 3) << 2) & (4 * NF - 1));
}

// Division of n < 2^31 by a number that the host knows: with s = ceil(log2 d) and
// m = ceil(2^(31 + s) / d), n m / 2^(31 + s) exceeds n / d by less than
// n / 2^31 / d.  Four plain divisions took 0.1 to 0.15 us of these 3 us launches.
struct Div {
  uint32_t d, m, shift;
};
inline Div make_div(uint32_t d) {
  uint32_t s = 0;
  while ((1ull << s) < d) ++s;
  return Div{d, (uint32_t)(((1ull << (31 + s)) + d - 1) / d), 31 + s};
}
__host__ __device__ __forceinline__ uint32_t quot(uint32_t n, const Div& v) {
  return (uint32_t)(((uint64_t)n * v.m) >> v.shift);
}

// The tile of a workgroup.  Consecutive ids are the row chunks of a column tile,
// then an item's column tiles; with xcd each XCD takes a contiguous run of them.
struct SmallTile {
  uint32_t item, ct, mc;  // batch item, column tile, row chunk
};
__device__ __forceinline__ SmallTile small_tile(bool xcd, const Div& chunks, const Div& tiles) {
  const uint32_t id = xcd ? (uint32_t)xcd_remap(blockIdx.x, (int)gridDim.x) : blockIdx.x;
  const uint32_t rest = quot(id, chunks), item = quot(rest, tiles);
  return SmallTile{item, rest - item * tiles.d, id - rest * chunks.d};
}

template <int NF>
__global__ __launch_bounds__(64) void gemm_bf16_smallm_kernel(const uint16_t* __restrict__ A,
                                                              const uint16_t* __restrict__ B,
                                                              uint16_t* __restrict__ C, int M, int N, int K,
                                                              int lda, int ldb, int ldc, long long sA, long long sB,
                                                              long long sC, bool xcd, Div chunks, Div tiles) {
  constexpr int TN = 32 * NF;                 // columns per workgroup
  constexpr int RB = TN * 2;                  // B row bytes in LDS
  constexpr int B_B = SM_BK * RB;             // B chunk bytes
  constexpr int STAGE = SM_A_B + B_B;
  constexpr int BL = B_B / 1024;              // B direct loads per chunk
  constexpr int LPC = 4 + BL;                 // direct loads per chunk
  constexpr int BCH = RB / 16;                // 16-byte chunks per B row
  constexpr int BRPL = 1024 / RB;             // B rows per direct load
  constexpr int SM_NS = NF == 4 ? 4 : 6;      // ring stages
  __shared__ __align__(1024) unsigned char smem[SM_NS * STAGE];
  const int lane = threadIdx.x;
  const int g = lane >> 5;
  const SmallTile t = small_tile(xcd, chunks, tiles);
  const size_t item = t.item;
  const int n0 = t.ct * TN, m0 = t.mc * 32;
  A += item * sA + (size_t)m0 * lda;
  B += item * sB;
  C += item * sC + (size_t)m0 * ldc;
  M -= m0;
  const int nk = K / SM_BK;
  const uint32_t lds0 = lds_addr(smem);

  // Direct-load lane offsets.  A load n (0..3): rows 8n + lane/8, chunk
  // (lane%8) ^ swz_a(row); rows past M re-read row M-1.  B load n:
  // k-rows BRPL n + lane/BCH, chunk (lane%BCH) ^ sm_swz(k-row); columns
  // past N re-read the last valid 8.
  uint32_t a_off[4], b_off[BL];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int row = 8 * n + (lane >> 3);
    a_off[n] = (uint32_t)min(row, M - 1) * (uint32_t)lda * 2u + 16u * ((lane & 7) ^ swz_a(row));
  }
#pragma unroll
  for (int n = 0; n < BL; ++n) {
    const int kr = BRPL * n + lane / BCH;
    const int col = min(n0 + 8 * ((lane % BCH) ^ sm_swz<NF>(kr)), N - 8);
    b_off[n] = (uint32_t)kr * (uint32_t)ldb * 2u + 2u * col;
  }
  auto issue = [&](int kt) {
    const uint32_t st = lds0 + (kt % SM_NS) * STAGE;
    const uint16_t* ab = A + (size_t)kt * SM_BK;
    const uint16_t* bb = B + (size_t)kt * SM_BK * ldb;
#pragma unroll
    for (int n = 0; n < 4; ++n) dma16(ab, a_off[n], st + n * 1024);
#pragma unroll
    for (int n = 0; n < BL; ++n) dma16(bb, b_off[n], st + SM_A_B + n * 1024);
  };

  // Fragments (C^T = B^T . A^T): A^T (B operand) row m = lane%32, chunk
  // 2 ks + g; B^T (A operand) of column tile nf by transposing reads, lane
  // (g, sg, 4j+a) at k-row 16 ks + 8 g + 4 r + j, columns 32 nf + 16 sg + 4 a.
  const int am = lane & 31;
  const int b_sg = (lane >> 4) & 1, b_j = (lane >> 2) & 3, b_a = lane & 3;
  const uint32_t a_base = lds0 + am * 128;
  const int ax = swz_a(am);
  uint32_t b_base[NF];
#pragma unroll
  for (int nf = 0; nf < NF; ++nf) {
    const int chunk = (32 * nf + 16 * b_sg + 4 * b_a) >> 3;  // k-row 8g + b_j: swizzle sm_swz(b_j)
    b_base[nf] = lds0 + SM_A_B + (8 * g + b_j) * RB + 16 * (chunk ^ sm_swz<NF>(b_j)) + 8 * (b_a & 1);
  }

  f32x16 acc[NF];
#pragma unroll
  for (int nf = 0; nf < NF; ++nf) acc[nf] = f32x16{};
#pragma unroll
  for (int p = 0; p < SM_NS - 1; ++p)
    if (p < nk) issue(p);
  for (int kt = 0; kt < nk; ++kt) {
    // chunk kt landed once at most min(NS-2, nk-1-kt) later chunks are in flight
    wait_chunks<LPC, SM_NS - 2>(nk - 1 - kt);
    if (kt + SM_NS - 1 < nk) issue(kt + SM_NS - 1);
    const uint32_t so = (kt % SM_NS) * STAGE;
#pragma unroll
    for (int ks = 0; ks < SM_BK / 16; ++ks) {
      const u32x4 af = lds_ld128(a_base + so + 16 * ((2 * ks + g) ^ ax));
#pragma unroll
      for (int nf = 0; nf < NF; ++nf) {
        const uint32_t bp = b_base[nf] + so + 16 * ks * RB;
        const u32x2 lo = lds_read_tr16_at(bp);
        const u32x2 hi = lds_read_tr16_at(bp + 4 * RB);
        acc[nf] = mfma32<BF16>(u32x4{lo[0], lo[1], hi[0], hi[1]}, af, acc[nf]);
      }
    }
  }

  // lane holds m = lane%32, n = n0 + 32 nf + 8 i + 4 g + {0..3}
  if (am < M) {
    uint16_t* crow = C + (size_t)am * ldc;
#pragma unroll
    for (int nf = 0; nf < NF; ++nf)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int gn = n0 + 32 * nf + 8 * i + 4 * g;
        const f32x16& a = acc[nf];
        if (gn < N) st64(crow + gn, u32x2{pack_bf16x2(a[4 * i], a[4 * i + 1]), pack_bf16x2(a[4 * i + 2], a[4 * i + 3])});
      }
  }
}

// Split-K variant for items with a few 64-deep K chunks (4..12, e.g. the
// 32 x 128 x 512 up-projection of the MLA absorbed step): one workgroup of
// KW waves per 32 x (32 NF) tile, wave w taking chunks w*nkw .. w*nkw +
// nkw - 1 and issuing all of them at once into its own LDS region, so a
// tile needs a single round trip to memory and reads A once per column
// tile; the partial sums meet in LDS (waves 1..KW-1 each write theirs into
// their own, consumed region, wave 0 adds and stores).
template <int NF, int KW>
__global__ __launch_bounds__(64 * KW) void gemm_bf16_smallm_sk_kernel(const uint16_t* __restrict__ A,
                                                                     const uint16_t* __restrict__ B,
                                                                     uint16_t* __restrict__ C, int M, int N, int K,
                                                                     int lda, int ldb, int ldc, long long sA,
                                                                     long long sB, long long sC, bool xcd, Div chunks,
                                                                     Div tiles) {
  constexpr int TN = 32 * NF, RB = TN * 2, B_B = SM_BK * RB, STAGE = SM_A_B + B_B;
  constexpr int BL = B_B / 1024, BCH = RB / 16, BRPL = 1024 / RB;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5;
  const SmallTile t = small_tile(xcd, chunks, tiles);
  const size_t item = t.item;
  const int n0 = t.ct * TN, m0 = t.mc * 32;
  A += item * sA + (size_t)m0 * lda;
  B += item * sB;
  C += item * sC + (size_t)m0 * ldc;
  M -= m0;
  const int nkw = K / SM_BK / KW;  // chunks per wave (1..3)
  const int kc0 = wave * nkw;
  const uint32_t lds0 = lds_addr(smem) + wave * nkw * STAGE;

  // Direct-load lane offsets as in the kernel above.
  uint32_t a_off[4], b_off[BL];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int row = 8 * n + (lane >> 3);
    a_off[n] = (uint32_t)min(row, M - 1) * (uint32_t)lda * 2u + 16u * ((lane & 7) ^ swz_a(row));
  }
#pragma unroll
  for (int n = 0; n < BL; ++n) {
    const int kr = BRPL * n + lane / BCH;
    const int col = min(n0 + 8 * ((lane % BCH) ^ sm_swz<NF>(kr)), N - 8);
    b_off[n] = (uint32_t)kr * (uint32_t)ldb * 2u + 2u * col;
  }
  for (int c = 0; c < nkw; ++c) {
    const uint32_t st = lds0 + c * STAGE;
    const uint16_t* ab = A + (size_t)(kc0 + c) * SM_BK;
    const uint16_t* bb = B + (size_t)(kc0 + c) * SM_BK * ldb;
#pragma unroll
    for (int n = 0; n < 4; ++n) dma16(ab, a_off[n], st + n * 1024);
#pragma unroll
    for (int n = 0; n < BL; ++n) dma16(bb, b_off[n], st + SM_A_B + n * 1024);
  }

  const int am = lane & 31;
  const int b_sg = (lane >> 4) & 1, b_j = (lane >> 2) & 3, b_a = lane & 3;
  const uint32_t a_base = lds0 + am * 128;
  const int ax = swz_a(am);
  uint32_t b_base[NF];
#pragma unroll
  for (int nf = 0; nf < NF; ++nf) {
    const int chunk = (32 * nf + 16 * b_sg + 4 * b_a) >> 3;
    b_base[nf] = lds0 + SM_A_B + (8 * g + b_j) * RB + 16 * (chunk ^ sm_swz<NF>(b_j)) + 8 * (b_a & 1);
  }
  f32x16 acc[NF];
#pragma unroll
  for (int nf = 0; nf < NF; ++nf) acc[nf] = f32x16{};
  land_args(C);  // C is used only after the loop
  for (int c = 0; c < nkw; ++c) {
    // chunk c landed once at most nkw-1-c later chunks are in flight
    wait_chunks<4 + BL, 2>(nkw - 1 - c);
    const uint32_t so = c * STAGE;
#pragma unroll
    for (int ks = 0; ks < SM_BK / 16; ++ks) {
      const u32x4 af = lds_ld128(a_base + so + 16 * ((2 * ks + g) ^ ax));
#pragma unroll
      for (int nf = 0; nf < NF; ++nf) {
        const uint32_t bp = b_base[nf] + so + 16 * ks * RB;
        const u32x2 lo = lds_read_tr16_at(bp);
        const u32x2 hi = lds_read_tr16_at(bp + 4 * RB);
        acc[nf] = mfma32<BF16>(u32x4{lo[0], lo[1], hi[0], hi[1]}, af, acc[nf]);
      }
    }
  }

  // Partial sums: waves 1..KW-1 into their own (consumed) LDS region, laid
  // out [nf][e][lane] so consecutive lanes hit consecutive banks.
  float* mine = reinterpret_cast<float*>(smem + wave * nkw * STAGE);
  if (wave > 0) {
#pragma unroll
    for (int nf = 0; nf < NF; ++nf)
#pragma unroll
      for (int e = 0; e < 16; ++e) mine[(nf * 16 + e) * 64 + lane] = acc[nf][e];
  }
  __syncthreads();
  if (wave > 0) return;  // no barrier follows
  for (int w = 1; w < KW; ++w) {
    const float* other = reinterpret_cast<const float*>(smem + w * nkw * STAGE);
#pragma unroll
    for (int nf = 0; nf < NF; ++nf)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[nf][e] += other[(nf * 16 + e) * 64 + lane];
  }

  // lane holds m = lane%32, n = n0 + 32 nf + 8 i + 4 g + {0..3}
  if (am < M) {
    uint16_t* crow = C + (size_t)am * ldc;
#pragma unroll
    for (int nf = 0; nf < NF; ++nf)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int gn = n0 + 32 * nf + 8 * i + 4 * g;
        const f32x16& a = acc[nf];
        if (gn < N) st64(crow + gn, u32x2{pack_bf16x2(a[4 * i], a[4 * i + 1]), pack_bf16x2(a[4 * i + 2], a[4 * i + 3])});
      }
  }
}

// Batched items of few rows: four to twelve 64-deep chunks of K are split among
// four waves, one workgroup per 32 x 64 tile when that still gives >= 256
// workgroups (one per CU), else 32 x 32; other K run one wave per tile, the
// widest that still leaves >= 512 workgroups (two per CU).
static bool small_split_k(int K) { return K / SM_BK % 4 == 0 && K / SM_BK <= 12; }
static int small_width(int batch, int M, int N, int K) {  // 32-column fragments of a tile
  auto groups = [&](int tn) { return (long long)batch * ((M + 31) / 32) * ((N + tn - 1) / tn); };
  if (small_split_k(K)) return groups(64) >= 256 ? 2 : 1;
  return groups(128) >= 512 ? 4 : groups(64) >= 512 ? 2 : 1;
}

static int launch_smallm(const void* A, const void* B, void* C, int batch, int M, int N, int K, int lda, int ldb,
                         int ldc, long long sA, long long sB, long long sC, hipStream_t stream) {
  auto go = [&](auto kern, int threads, int smem, int tn) {
    const int chunks = (M + 31) / 32, tiles = (N + tn - 1) / tn;
    const long long grid = (long long)batch * chunks * tiles;
    if (grid > 0x7fffffffLL) return MX_ERR_SHAPE;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(threads), smem, stream, (const uint16_t*)A, (const uint16_t*)B,
                       (uint16_t*)C, M, N, K, lda, ldb, ldc, sA, sB, sC, K / SM_BK > 2, make_div(chunks),
                       make_div(tiles));
    MX_RETURN_IF_HIP(hipGetLastError());
    return MX_OK;
  };
  const int nkc = K / SM_BK, nf = small_width(batch, M, N, K);
  if (small_split_k(K)) {
    auto split_k = [&](auto nf_tag) {
      constexpr int NF = decltype(nf_tag)::value, STAGE = SM_A_B + SM_BK * 64 * NF;
      constexpr auto kern = gemm_bf16_smallm_sk_kernel<NF, 4>;
      MX_RETURN_IF_HIP(lds_limit_once<kern>(12 * STAGE));
      return go(kern, 256, nkc * STAGE, 32 * NF);
    };
    return nf == 2 ? split_k(std::integral_constant<int, 2>{}) : split_k(std::integral_constant<int, 1>{});
  }
  if (nf == 4) return go(gemm_bf16_smallm_kernel<4>, 64, 0, 128);
  if (nf == 2) return go(gemm_bf16_smallm_kernel<2>, 64, 0, 64);
  return go(gemm_bf16_smallm_kernel<1>, 64, 0, 32);
}


// ---------------------------------------------------------------------------
// gemm_bf16_stream_kernel: products with few tiles (decode batches, small
// M or N with a long K) stream the weights B.  Tiles of 64 or more rows
// would leave most CUs idle.
//  * A workgroup owns 32 NC columns x 32 MF rows of C, NW waves; wave w takes
//    the 64-deep K blocks kb = w, w + NW, ..., so every workgroup streams its
//    columns of B once.  The row chunks of a column block and the
//    neighbouring column blocks run on one XCD, where they share B's
//    128-byte lines in L2; with more rows than columns, the column blocks of a
//    row chunk.
//  * Each wave has a private ring of NSL slots, one K block per slot (A: 32 MF
//    rows x 128 B, chunk c at c ^ ((m >> 1) & 7); B: 64 k-rows x 64 NC B), by
//    direct loads; slots are private, so the block loop has no barrier.
//  * What bounds it is the CU's rate of line requests (about one per 3-4
//    clocks, 64 or 128 bytes alike), so 64 columns where they still fill the
//    CUs; eight waves with rings of two slots keep as many loads in flight as
//    four with four and reach each block sooner, which shows on short K only
//    (against four waves: 27x512x1280 4.14 -> 4.09 us, 16x7168x4096 14.5 either
//    way, 5x712x6272 13.3 -> 13.9).
//  * C^T = B^T . A^T on 32x32x16 MFMAs: B^T fragments by transposing reads
//    from the B rows (swz_sb), A^T fragments by ds_read_b128.
//  * The waves' accumulators meet in LDS at the end; four waves sum and store
//    the result registers holding n = 8i + 4(l/32) + {0..3}, i their number.
// ---------------------------------------------------------------------------
template <int MF, int NC, int NW, int NSL>
struct StreamCfg {
  static constexpr int BN = 32 * NC;          // columns per workgroup
  static constexpr int A_B = 32 * MF * 128;  // 64 k of 32 MF rows
  static constexpr int B_B = 64 * BN * 2;     // 64 k-rows
  static constexpr int SLOT = A_B + B_B;
  static constexpr int A_L = A_B / 1024, B_L = B_B / 1024;
  static constexpr int VM = A_L + B_L;
  static constexpr int LDS = NW * NSL * SLOT;
  static_assert(NW == 4 || NW == 8, "waves");
  static_assert(NC == 1 || NC == 2, "B row swizzle");
  static_assert(LDS <= 160 * 1024, "LDS");
  static_assert((NSL - 1) * VM < 64, "vmcnt range");
  static_assert(NW * MF * NC * 64 * 16 * 4 <= LDS, "reduction area");
};
// B rows of 128 bytes: a transposing read phase (4 consecutive k-rows x 64
// bytes) spans the 256-byte bank window twice, so k-rows 2 and 3 swap their
// halves; rows of 64 bytes fill it once.
template <int NC>
__device__ __forceinline__ int swz_sb(int k) {
  return NC == 1 ? 0 : ((k >> 1) & 1) << 2;
}

template <int MF, int NC, int NW, int NSL, bool TAIL>
__global__ __launch_bounds__(64 * NW, 1) void gemm_bf16_stream_kernel(const uint16_t* __restrict__ A,
                                                                    const uint16_t* __restrict__ B,
                                                                    uint16_t* __restrict__ C, int M, int N, int K,
                                                                    int lda, int ldb, int ldc) {
  using CF = StreamCfg<MF, NC, NW, NSL>;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Workgroup -> (BN-column block, chunk of 32 MF rows), the row chunks of a
  // column block adjacent, so one XCD holds whole column blocks and their
  // neighbours (which share B's lines in L2); with more rows than columns the
  // column blocks of a row chunk, so the XCDs share out A instead.
  const int nmc = (M + 32 * MF - 1) / (32 * MF);
  const int wid = xcd_remap(blockIdx.x, (int)gridDim.x);
  const int ncb = (N + CF::BN - 1) / CF::BN;
  const bool tall = M > N;
  const int n0 = (tall ? wid % ncb : wid / nmc) * CF::BN, m0 = (tall ? wid / ncb : wid % nmc) * 32 * MF;
  A += (size_t)m0 * lda;
  C += (size_t)m0 * ldc;
  M -= m0;  // rows of this chunk (more than 32 MF only past the last row read)
  const int kblocks = K / 64;
  const int cnt = kblocks > wave ? (kblocks - wave + NW - 1) / NW : 0;
  const uint32_t ring = lds_addr(smem) + wave * NSL * CF::SLOT;

  // A load n: rows 8n + l/8, LDS chunk l%8 taking global chunk (l%8) ^
  // swz(row) (rows past M re-read row M-1); B load n: its BR k-rows' chunks in
  // lane order, chunk c of k-row k at c ^ swz_sb(k) (columns past N re-read
  // the last 8 valid ones; never stored).
  uint32_t a_off[CF::A_L];
#pragma unroll
  for (int n = 0; n < CF::A_L; ++n) {
    const int row = 8 * n + (lane >> 3);
    a_off[n] = (uint32_t)min(row, M - 1) * (uint32_t)lda * 2u + 16u * ((lane & 7) ^ swz_a(row));
  }
  constexpr int CH = CF::BN / 8, BR = 64 / CH;  // 16-byte chunks per k-row, k-rows per load
  const int b_row = lane / CH;                   // from k-row BR n; BR n has no part in swz_sb
  const uint32_t b_col_off = 2u * (min(n0 + 8 * ((lane % CH) ^ swz_sb<NC>(b_row)), N - 8) - n0);
  const uint32_t b_off = (uint32_t)b_row * (uint32_t)ldb * 2u + b_col_off;
  auto issue = [&](int i, auto slot_tag) {
    constexpr int I = decltype(slot_tag)::value;
    const int kb = cnt > 0 ? wave + NW * min(i, cnt - 1) : 0;
    const uint32_t st = ring + I * CF::SLOT;
#pragma unroll
    for (int n = 0; n < CF::A_L; ++n) dma16(A + (size_t)kb * 64, a_off[n], st + n * 1024);
    const uint16_t* bb = B + (size_t)kb * 64 * ldb + n0;
#pragma unroll
    for (int n = 0; n < CF::B_L; ++n) dma16(bb + (size_t)BR * ldb * n, b_off, st + CF::A_B + n * 1024);
  };

  // fragment lane addresses within a slot.  A^T (B operand): row am, chunk
  // 2 ks + g.  B^T (A operand): lane 16G + 4j + a reads k-row 8 (G>>1) +
  // 4 r + j (+16 ks), columns 32 c + 16 (G&1) + 4a .. +3.
  const int am = lane & 31, g = lane >> 5;
  uint32_t a_col[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) a_col[ks] = am * 128 + 16 * ((2 * ks + g) ^ swz_a(am));
  const int G = lane >> 4, bj = (lane >> 2) & 3, ba = lane & 3;
  uint32_t b_col[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c)
    b_col[c] = CF::A_B + (8 * (G >> 1) + bj) * (2 * CF::BN) +
               16 * ((4 * c + 2 * (G & 1) + (ba >> 1)) ^ swz_sb<NC>(bj)) + 8 * (ba & 1);

  f32x16 acc[NC][MF];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int f = 0; f < MF; ++f) acc[c][f] = f32x16{};

  // the first kr k values of a slot count (64: all of them)
  auto compute = [&](auto slot_tag, int kr) {
    constexpr int I = decltype(slot_tag)::value;
    const uint32_t st = ring + I * CF::SLOT;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (16 * ks >= kr) break;
      const bool keep = 16 * ks + 8 * g < kr;
      u32x4 bt[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const u32x2 lo = lds_read_tr16_at(st + b_col[c] + 16 * ks * (2 * CF::BN));
        const u32x2 hi = lds_read_tr16_at(st + b_col[c] + (16 * ks + 4) * (2 * CF::BN));
        bt[c] = keep_if(keep, u32x4{lo[0], lo[1], hi[0], hi[1]});
      }
#pragma unroll
      for (int f = 0; f < MF; ++f) {
        const u32x4 at = keep_if(keep, lds_ld128(st + 32 * f * 128 + a_col[ks]));
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c][f] = mfma32<BF16>(bt[c], at, acc[c][f]);
      }
    }
  };

  land_args(C);
  // The K % 64 tail is one more block of the next wave in turn, computed
  // first, from the slot that the prologue leaves free.  Chunks and k-rows
  // past K re-read the last valid ones.
  const int kr = K - kblocks * 64;
  const bool mine = TAIL && wave == kblocks % NW;
  if (mine) {
    const uint32_t st = ring + (NSL - 1) * CF::SLOT;
#pragma unroll
    for (int n = 0; n < CF::A_L; ++n) {
      const uint32_t swz = 16u * ((lane & 7) ^ swz_a(8 * n + (lane >> 3)));
      dma16(A + (size_t)kblocks * 64, a_off[n] - swz + min(swz, (uint32_t)(2 * kr - 16)), st + n * 1024);
    }
#pragma unroll
    for (int n = 0; n < CF::B_L; ++n) {
      if (BR * n >= kr) break;
      dma16(B + ((size_t)kblocks * 64 + BR * n) * ldb + n0,
            (uint32_t)min(b_row, kr - 1 - BR * n) * (uint32_t)ldb * 2u + b_col_off, st + CF::A_B + n * 1024);
    }
  }
  unroll_n<NSL - 1>([&](auto i_tag) { issue(decltype(i_tag)::value, i_tag); });
  if (mine) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"((NSL - 1) * CF::VM) : "memory");
    compute(std::integral_constant<int, NSL - 1>{}, kr);
  }
  // block i: issue block i + NSL - 1 into the slot block i - 1 used (its
  // reads completed), then wait for block i
  auto step = [&](int i, auto slot_tag) {
    constexpr int I = decltype(slot_tag)::value;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    issue(i + NSL - 1, std::integral_constant<int, (I + NSL - 1) % NSL>{});
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"((NSL - 1) * CF::VM) : "memory");
    compute(slot_tag, 64);
  };
  int i = 0;
  for (; i + NSL <= cnt; i += NSL) unroll_n<NSL>([&](auto s_tag) { step(i + decltype(s_tag)::value, s_tag); });
  unroll_n<NSL - 1>([&](auto s_tag) {
    if (i + decltype(s_tag)::value < cnt) step(i + decltype(s_tag)::value, s_tag);
  });
  wait_vmcnt<0>();  // no DMA may land in the ring once it is reused below

  // ---- accumulators meet in LDS: [wave][c][f][e][lane] floats ----
  __syncthreads();
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int f = 0; f < MF; ++f)
#pragma unroll
      for (int e = 0; e < 16; ++e) red[(((wave * NC + c) * MF + f) * 16 + e) * 64 + lane] = acc[c][f][e];
  __syncthreads();
  // result quad 4 i .. 4 i + 3 of column fragment c to wave i (with 8 waves, i or i + 4)
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (wave / 4 != c % (NW / 4)) continue;
    const int gn = n0 + 32 * c + 8 * (wave % 4) + 4 * g;
#pragma unroll
    for (int f = 0; f < MF; ++f) {
      float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += red[(((w * NC + c) * MF + f) * 16 + 4 * (wave % 4) + j) * 64 + lane];
      const int gm = 32 * f + am;
      if (gm < M && gn < N)
        st64(C + (size_t)gm * ldc + gn, u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])});
    }
  }
}

template <int MF, int NC, int NW, int NSL>
static int launch_stream(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb, int ldc,
                         hipStream_t stream) {
  using CF = StreamCfg<MF, NC, NW, NSL>;
  const long long grid = (long long)((N + CF::BN - 1) / CF::BN) * ((M + 32 * MF - 1) / (32 * MF));
  if (grid > 0x7fffffffLL) return MX_ERR_SHAPE;
  auto go = [&](auto tail) {
    constexpr auto kern = gemm_bf16_stream_kernel<MF, NC, NW, NSL, decltype(tail)::value>;
    MX_RETURN_IF_HIP(lds_limit_once<kern>(CF::LDS));
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * NW), CF::LDS, stream, (const uint16_t*)A,
                       (const uint16_t*)B, (uint16_t*)C, M, N, K, lda, ldb, ldc);
    MX_RETURN_IF_HIP(hipGetLastError());
    return MX_OK;
  };
  return K % 64 ? go(std::true_type{}) : go(std::false_type{});
}

// The kernels of mx_gemm_bf16, and what one launch of each takes in
// microseconds: fixed + rounds (round + step K/64) + fill (tiles / slots) K/64
// with rounds = ceil(tiles / slots).  A round of workgroups costs its slowest
// one (round, step), and more workgroups at once share the L2 and the clock
// (fill).  Fitted (relative least squares, no negative term) to 450 random
// shapes, M 1..8192, N and K 512..8192, ragged and whole, each timed on every
// kernel by graph replay; the kernel picked is on average about 1% slower than
// the fastest, there and over 600 more shapes with M and N up to 131072 and K
// from 128 (16x129280x7168 322 us at 5.75 TB/s, 446 with four-wave streams).  3%
// of those are more than 3% slower than the 32-deep ring and register-staged
// tiles, up to 20%, which no kernel here matches: K an odd multiple of 32 below
// 700 (6352x1088x480 13.0 -> 14.7) and 70 to 90 columns under 50000 rows and more
// (109374x72x488 28.7 -> 34.6).  The 64-column streams against the four-wave 32-column ones and
// the tiles alone: 260x3008x6080 30.2 -> 21.8 us, 524x1536x8064 42 -> 27 (64
// rows), 158x1664x6512 25.3 -> 20.4, 142x3032x2408 14.4 -> 12.6 (32 rows); below
// 48 K blocks the 64-row one is 5-10% behind 64x64 tiles (763x1280x1024 8.55
// against 7.91), which its min_k keeps.
enum class Path { None, Stream32, Stream32x64, Stream64, Stream64x64, T64, T64x128, T128, T128x192, T256 };
struct Kernel {
  Path path;
  int bm, bn, slots;  // tile, workgroups resident at once
  float fixed, round, step, fill;
  int min_k;
};
constexpr Kernel kKernels[] = {
    {Path::Stream32, 32, 32, 256, 2.206f, 1.142f, 0.089f, 0.082f, 64},
    {Path::Stream32x64, 32, 64, 256, 2.471f, 1.142f, 0.133f, 0.081f, 64},
    {Path::Stream64, 64, 32, 256, 1.048f, 2.553f, 0.121f, 0.095f, 64},
    {Path::Stream64x64, 64, 64, 256, 1.455f, 2.880f, 0.167f, 0.076f, 48 * 64},
    {Path::T64, 64, 64, 512, 2.301f, 1.117f, 0.184f, 0.298f, 0},
    {Path::T64x128, 64, 128, 256, 2.332f, 1.946f, 0.254f, 0.111f, 0},
    {Path::T128, 128, 128, 256, 1.749f, 2.956f, 0.353f, 0.187f, 0},
    {Path::T128x192, 128, 192, 256, 1.803f, 3.855f, 0.499f, 0.225f, 0},
    {Path::T256, 256, 256, 256, 2.082f, 6.139f, 0.977f, 0.532f, 64},
};

// The tiles over 16 items and more of a batched product: their operands are not
// shared between items, so more of them at once cost more (fill).  Fitted to 670
// random launches, 1 to 256 items of M 1..256, N and K to 2048, contiguous and
// strided by head.  Over 450 others the choice is 1.5% behind the fastest tile on
// average, with the costs of single products 5.4% (92 items of 168x224x384
// 20.9 us with 64x64 tiles, 16.2 with 128x128).  Up to 15 items those are the
// better ones (0.1% against 0.3%; 2 of 404x1048x1392 9.1 us, here 10.8).
constexpr int kManyItems = 16;
constexpr Kernel kBatchedKernels[] = {
    {Path::T64, 64, 64, 512, 1.660f, 1.249f, 0.135f, 0.707f, 0},
    {Path::T64x128, 64, 128, 256, 1.237f, 2.001f, 0.243f, 0.362f, 0},
    {Path::T128, 128, 128, 256, 1.049f, 2.420f, 0.339f, 0.446f, 0},
    {Path::T128x192, 128, 192, 256, 0.620f, 3.439f, 0.460f, 0.477f, 0},
};

// The same below K = 128, where tiles take gemm_bf16_short_kernel: fixed +
// first K/64 + round ceil(x) + (tile + fill K/64) x with x = tiles / 256, since
// a CU holds several workgroups of these.  Fitted to 440 random shapes, single
// and batched, M 1..20000, N 8..16384, K 8..120, operands cached and not; the
// kernel picked is on average 0.4% slower than the fastest of all.  256x256
// tiles are there for B strides whose 64 k-rows pass 4 GiB.
struct ShortKernel {
  Path path;
  int bm, bn;
  float fixed, first, round, tile, fill;
  int min_k;
};
constexpr ShortKernel kShortKernels[] = {
    {Path::T64, 64, 64, 2.316f, 0.502f, 0.070f, 0.531f, 0.184f, 0},
    {Path::T64x128, 64, 128, 2.119f, 0.478f, 0.451f, 0.701f, 0.336f, 0},
    {Path::T128, 128, 128, 2.392f, 0.648f, 0.624f, 0.811f, 0.517f, 0},
    {Path::Stream32, 32, 32, 1.256f, 0.103f, 1.427f, 0.270f, 0.166f, 64},
    {Path::T256, 256, 256, 0.0f, 1.490f, 5.060f, 7.154f, 0.0f, 64},
};

// batch items of a strided-batched product (the tiled kernels only), or 0 for
// a single one.
static Path gemm_path(int M, int N, int K, int lda, int ldb, int batch) {
  Path best = Path::None;
  double least = 0;
  auto consider = [&](const auto& k, auto&& cost) {
    const bool stream = k.path < Path::T64;
    if (K < k.min_k || (batch > 0 && (stream || k.path == Path::T256))) return;
    // The lane offsets of the direct loads are 32-bit: bm rows of A, and the
    // k-rows of B that share a base (8 to 64), span less than 4 GiB.
    const long long brows = stream ? 512 / k.bn : k.path == Path::T256 ? 32 : K < 64 ? K : 64;
    if ((long long)lda * 2 * k.bm > 0xffffffffLL || (long long)ldb * 2 * (brows - 1) + 2 * k.bn > 0xffffffffLL) return;
    const double tiles = (double)((M + k.bm - 1) / k.bm) * ((N + k.bn - 1) / k.bn) * (batch > 0 ? batch : 1);
    const double t = cost(k, tiles);
    if (best == Path::None || t < least) {
      best = k.path;
      least = t;
    }
  };
  const double kb = K / 64.0;
  if (K < kShortK) {
    for (const ShortKernel& k : kShortKernels)
      consider(k, [&](const ShortKernel& c, double tiles) {
        const double x = tiles / 256;
        return c.fixed + c.first * kb + c.round * __builtin_ceil(x) + (c.tile + c.fill * kb) * x;
      });
  } else {
    auto cost = [&](const Kernel& c, double tiles) {
      return c.fixed + __builtin_ceil(tiles / c.slots) * (c.round + c.step * kb) + c.fill * kb * tiles / c.slots;
    };
    if (batch >= kManyItems)
      for (const Kernel& k : kBatchedKernels) consider(k, cost);
    else
      for (const Kernel& k : kKernels) consider(k, cost);
  }
  return best;
}

static int launch_tiled(Path path, const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb,
                        int ldc, hipStream_t s, int batch, long long sA, long long sB, long long sC) {
  if (K < kShortK) {
    switch (path) {
      case Path::T64: return launch_short<64, 64, 2, 2>(A, B, C, M, N, K, lda, ldb, ldc, s, batch, sA, sB, sC);
      case Path::T64x128: return launch_short<64, 128, 2, 4>(A, B, C, M, N, K, lda, ldb, ldc, s, batch, sA, sB, sC);
      case Path::T128: return launch_short<128, 128, 2, 4>(A, B, C, M, N, K, lda, ldb, ldc, s, batch, sA, sB, sC);
      default: return MX_ERR_SHAPE;
    }
  }
  switch (path) {
    case Path::T64: return launch_dma64<64, 64, 2, 2, 4>(A, B, C, M, N, K, lda, ldb, ldc, s, batch, sA, sB, sC);
    case Path::T64x128: return launch_dma64<64, 128, 2, 4, 6>(A, B, C, M, N, K, lda, ldb, ldc, s, batch, sA, sB, sC);
    case Path::T128: return launch_dma64<128, 128, 2, 4, 5>(A, B, C, M, N, K, lda, ldb, ldc, s, batch, sA, sB, sC);
    case Path::T128x192: return launch_dma64<128, 192, 2, 4, 4>(A, B, C, M, N, K, lda, ldb, ldc, s, batch, sA, sB, sC);
    default: return MX_ERR_SHAPE;
  }
}

// The leading dimensions the interface takes, as mx_kernels.h states them: with
// K % 32 != 0 or a small grid, lda * 2 * BM (BM = 256, 128 or 64) and ldb * 2 * 64
// below 2^31; otherwise spans below 4 GiB.  The grid and BM are those of a fixed
// choice of tile by size and not of the kernel that gemm_path picks: a refit of
// its costs must not change which calls are refused.  Every shape taken here has
// a kernel there, whose own bound (4 GiB spans) is the wider one.
static bool strides_ok(int M, int N, int K, int lda, int ldb) {
  const long long la = lda, lb = ldb, four_g = 0xffffffffLL;
  auto tiles = [&](int t) { return (long long)((M + t - 1) / t) * ((N + t - 1) / t); };
  const bool span64 = la * 2 * 64 <= four_g && lb * 2 * 64 <= four_g;
  if (((M <= 64 && N >= 256) || (tiles(64) <= 64 && K >= 512)) && K % 64 == 0 && span64) return true;
  const bool big = tiles(256) >= 256 || 13 * ((tiles(256) + 255) / 256) < 5 * ((tiles(128) + 255) / 256);
  const bool b_fits = lb * 2 * 31 + 512 <= four_g;
  if (big && K % 32 == 0 && la * 2 * 256 <= four_g) return b_fits;
  if (tiles(256) >= 512) return strides_2g<256>(lda, ldb);
  if (tiles(128) >= 256 && K % 32 == 0 && la * 2 * 128 <= four_g) return b_fits;
  if (tiles(128) >= 256) return strides_2g<128>(lda, ldb);
  if (tiles(64) <= 256 && K >= 512 && M % 64 == 0 && N % 64 == 0 && K % 128 == 0 && span64) return true;
  return strides_2g<64>(lda, ldb);
}

}  // namespace gemm
}  // namespace mx

extern "C" int mx_gemm_bf16(const void* A, const void* B, void* C, int M, int N, int K, int lda, int ldb,
                            int ldc, void* stream) {
  if (!A || !B || !C) return MX_ERR_NULL;
  if (M <= 0 || N <= 0 || K <= 0) return MX_ERR_SHAPE;
  if (lda < K || ldb < N || ldc < N) return MX_ERR_SHAPE;
  if ((K % 8) || (N % 8) || (lda % 8) || (ldb % 8) || (ldc % 8)) return MX_ERR_ALIGN;
  if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15) return MX_ERR_ALIGN;
  hipStream_t s = (hipStream_t)stream;
  using namespace mx::gemm;
  if (!strides_ok(M, N, K, lda, ldb)) return MX_ERR_SHAPE;
  const Path path = gemm_path(M, N, K, lda, ldb, 0);
  switch (path) {
    case Path::Stream32: return launch_stream<1, 1, 8, 2>(A, B, C, M, N, K, lda, ldb, ldc, s);
    case Path::Stream32x64: return launch_stream<1, 2, 4, 3>(A, B, C, M, N, K, lda, ldb, ldc, s);
    case Path::Stream64: return launch_stream<2, 1, 4, 3>(A, B, C, M, N, K, lda, ldb, ldc, s);
    case Path::Stream64x64: return launch_stream<2, 2, 4, 2>(A, B, C, M, N, K, lda, ldb, ldc, s);
    case Path::T256: return launch_dma16s(A, B, C, M, N, K, lda, ldb, ldc, s);
    default: return launch_tiled(path, A, B, C, M, N, K, lda, ldb, ldc, s, 1, 0, 0, 0);
  }
}

namespace mx {
namespace gemm {

// Decode-sized items (M <= 32, whole 64-deep K chunks) run the
// weight-streaming small-M kernels.  Their lane offsets are 32-bit.
static bool batched_small(int M, int K, int lda, int ldb) {
  return M <= 32 && K % 64 == 0 && (long long)lda * 2 * 32 <= 0xffffffffLL && (long long)ldb * 2 * 64 <= 0xffffffffLL;
}

// More rows take the same kernels, 32 at a time, where that beats the tiles
// (graph replay; 1200 random items, contiguous and strided by head): K split
// among four waves while a workgroup per CU is enough (N 128, K 512: 16 items of
// 48 rows 4.62 -> 3.49 us, 64 items 5.39 -> 5.22, but 128 items 7.3 -> 9.1), and
// one or two chunks of K, which need a single round trip, while all workgroups
// run at once, three of 32 x 32 to a CU (K 128: 14 items of 46 x 512 3.19 against
// 3.34 us with tiles, 75 of 38 x 512 8.1 against 5.4; K 64: 120 of 36 x 72, 720
// workgroups, 3.00 against 3.30, 133 of 58 x 88, 798, 4.10 against 3.55).
static bool batched_rows(int batch, int M, int N, int K, int lda, int ldb) {
  if (K % 64 || !strides_2g<64>(lda, ldb)) return false;
  const int nkc = K / SM_BK;
  const long long rows = (long long)batch * ((M + 31) / 32);
  if (nkc % 4 == 0 && nkc <= 12) return rows * ((N + 63) / 64) <= 256;
  return nkc <= 2 && small_width(batch, M, N, K) == 1 && rows * ((N + 31) / 32) <= 768;
}

// Every check mx_gemm_bf16_batched makes before it launches, the grid
// limits of the kernel it would pick included, so a caller that chains
// several products can validate them all before enqueuing any.
int batched_check(const void* A, const void* B, void* C, int batch, int M, int N, int K, int lda, int ldb, int ldc,
                  long long strideA, long long strideB, long long strideC) {
  if (!A || !B || !C) return MX_ERR_NULL;
  if (batch <= 0 || M <= 0 || N <= 0 || K <= 0) return MX_ERR_SHAPE;
  if (batch > 65535 || strideA < 0 || strideB < 0 || strideC < 0) return MX_ERR_SHAPE;
  if (lda < K || ldb < N || ldc < N) return MX_ERR_SHAPE;
  if ((K % 8) || (N % 8) || (lda % 8) || (ldb % 8) || (ldc % 8)) return MX_ERR_ALIGN;
  if ((strideA % 8) || (strideB % 8) || (strideC % 8)) return MX_ERR_ALIGN;
  if (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 15) return MX_ERR_ALIGN;
  const auto tiles = [&](int t) { return (long long)((M + t - 1) / t) * ((N + t - 1) / t); };
  const bool small = batched_small(M, K, lda, ldb);
  if (!small && !(M >= 128 && tiles(128) * batch >= 256 ? strides_2g<128>(lda, ldb) : strides_2g<64>(lda, ldb)))
    return MX_ERR_SHAPE;
  const long long grid = small ? (long long)batch * ((N + 31) / 32) : tiles(64);  // widest grid of the kernels
  return grid > 0x7fffffffLL ? MX_ERR_SHAPE : MX_OK;
}

}  // namespace gemm
}  // namespace mx

extern "C" int mx_gemm_bf16_batched(const void* A, const void* B, void* C, int batch, int M, int N, int K, int lda,
                                    int ldb, int ldc, long long strideA, long long strideB, long long strideC,
                                    void* stream) {
  using namespace mx::gemm;
  if (const int e = batched_check(A, B, C, batch, M, N, K, lda, ldb, ldc, strideA, strideB, strideC)) return e;
  hipStream_t s = (hipStream_t)stream;
  if (batched_small(M, K, lda, ldb) || batched_rows(batch, M, N, K, lda, ldb))
    return launch_smallm(A, B, C, batch, M, N, K, lda, ldb, ldc, strideA, strideB, strideC, s);
  return launch_tiled(gemm_path(M, N, K, lda, ldb, batch), A, B, C, M, N, K, lda, ldb, ldc, s, batch, strideA, strideB,
                      strideC);
}
