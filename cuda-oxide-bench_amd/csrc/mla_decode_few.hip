// MLA absorbed decode for up to 16 heads (a tensor-parallel rank's share).
//
// The 128-head kernel of mla_decode.hip spends the matrix and LDS work of 128
// heads whatever H is, and streams the cache at 3 TB/s with 16.  With few heads
// the decode is a stream of the latent cache (1152 B per token), bound by HBM,
// and this kernel is built around the stream:
//
//  * A wave owns all 16 heads and every fourth 16-token block of its
//    workgroup's slice, from scores to values: Q^T (72 VGPRs) and the O^T
//    accumulators (128) stay in its registers.
//  * Each wave has a private ring of two 18 KB slots (16 latent rows of 1 KB,
//    16 rope rows of 128 B) filled by direct loads, so the loop has no
//    barrier: while a block is computed the next one is in flight, four
//    waves' worth (72 KB) per CU.
//  * Scores S^T = K . Q^T on 16x16x32 MFMAs: lane (kg, l) holds head l and
//    tokens 4 kg .. +3 of the block.  That is the B operand of the 16x16x16
//    MFMAs of O^T += V^T . P^T, so the probabilities never leave the
//    registers; V^T fragments are transposing LDS reads of the same rows.
//  * Chunk c of latent row t sits at c ^ 2 (t & 7): a K read's 16-lane group
//    holds all 16 tokens, its chunk's low bit keyed by t's bits 2 and 3, and
//    a V read's half-wave holds 8 consecutive tokens x 32 bytes; both then
//    touch distinct bank slots.  Rope rows: c ^ ((t >> 1) & 7).
//  * The four waves' states meet in LDS by the log-sum-exp rule; a slice
//    writes O (one slice) or its normalised bf16 partial and (m, l).
//
// Measured (decode and merge, rotated caches, against the 128-head kernel with
// its former splits): B48 T6001 114 -> 66 us (5.0 TB/s), B28 T10000 100 -> 68,
// B32 T4096 48 -> 38, B20 T2000 31 -> 19, B1 T32768 26 -> 19, B3 T819 17 -> 14.
// Two head groups per wave (accumulators in AGPRs, 32 heads) measured no
// faster than the 128-head kernel and is not kept.
#include "mla_common.h"

namespace mx {
namespace mla {

namespace {
constexpr int NW = 4;                    // waves per workgroup
constexpr int BT = 16;                   // tokens per block
constexpr int LAT_B = BT * 1024, ROPE_B = BT * 128;
constexpr int SLOT = LAT_B + ROPE_B;     // 18 KB
constexpr int NSLOT = 2;
constexpr int LPB = SLOT / 1024;         // direct loads per block
constexpr int RING = NW * NSLOT * SLOT;  // 144 KB
constexpr int VT = DV / 16;              // 16-column tiles of O^T
constexpr int LA = 6;                    // fragment reads issued ahead of their MFMAs
constexpr int KL = DV / 32, KS = DQK / 32;  // k-steps of the scores: latent, all
static_assert(RING <= 160 * 1024 && NW * VT * 64 * 16 <= RING, "LDS");

__device__ __forceinline__ int swz_l(int t) { return (t & 7) << 1; }
__device__ __forceinline__ int swz_r(int t) { return (t >> 1) & 7; }

// Byte offset, from the first row of the block at token tok0, of the last row
// of it that the sequence has.  Counted in rows first: the rest of a sequence
// of more than 3.7 million tokens is over 2^32 bytes.
__host__ __device__ __forceinline__ uint32_t last_row(int T, int tok0) {
  return (uint32_t)(T - tok0 < BT ? T - tok0 - 1 : BT - 1) * ROW_B;
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f32x4 mfma_k16(const u32x2& a, const u32x2& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0,
                                                   0);
}
}  // namespace

__global__ __launch_bounds__(64 * NW, 1) void mla_decode_few_kernel(const uint16_t* __restrict__ Q,
                                                                const uint16_t* __restrict__ Qr,
                                                                const uint16_t* __restrict__ KV,
                                                                uint16_t* __restrict__ O, uint32_t* __restrict__ ws_o,
                                                                float* __restrict__ ws_ml, int B, int H, int T,
                                                                float sl2, int nsplit, int tps, int q_ld, int qr_ld) {
  extern __shared__ __align__(1024) unsigned char smem[];
  __shared__ float ml[2][NW][16];  // running max, row sum of each wave's heads
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kg = lane >> 4;

  const int id = xcd_remap(blockIdx.x, B * nsplit);
  const int s = id % nsplit, b = id / nsplit;
  const int t0 = s * tps, t1 = min(T, t0 + tps);
  const int nblk = (t1 - t0 + BT - 1) / BT;
  const int cnt = nblk > wave ? (nblk - wave + NW - 1) / NW : 0;  // this wave's blocks: wave, wave + NW, ..

  // ---- direct loads of block i of this wave into ring slot i % 2, in two
  // halves of eight tokens: eight loads of one latent row, one of eight rope
  // rows.  A loop and not unrolled further: the kernel's code is fetched anew
  // for every short launch.  Rows past the sequence re-read its last one, rows
  // past the slice are other slices'; the scores of both are masked. ----
  const unsigned char* kvb = reinterpret_cast<const unsigned char*>(KV + (size_t)b * T * DQK);
  const uint32_t ring = lds_addr(smem) + wave * NSLOT * SLOT;
  auto issue = [&](int i) {
    const int tok0 = t0 + (wave + NW * i) * BT;
    const unsigned char* base = kvb + (size_t)tok0 * ROW_B;
    const uint32_t last = last_row(T, tok0);
    const uint32_t st = ring + (i & 1) * SLOT;
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
      uint32_t l16b = 16u * lane;
      asm volatile("" : "+v"(l16b));  // the per-row XOR stays here instead of in a register per row
#pragma unroll
      for (int r = 0; r < 8; ++r)
        dma16(base + min((8 * h + r) * (uint32_t)ROW_B, last), l16b ^ (16u * swz_l(r)), st + (8 * h + r) * 1024);
      const int r0 = 8 * h + (lane >> 3);
      dma16(base, min(r0 * (uint32_t)ROW_B, last) + 16u * (64 + ((lane & 7) ^ swz_r(r0))), st + LAT_B + h * 1024);
    }
  };
#pragma unroll 1
  for (int i = 0; i < min(cnt, 2); ++i) issue(i);

  // ---- Q^T fragments (B operand): head l16, k 32 ks + 8 kg ..
  // +7.  Heads past H re-read the last one; their results are never stored ----
  u32x4 qf[KS];
  const size_t row = (size_t)b * H + min(l16, H - 1);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    qf[ks] = ks < KL ? ld128(Q + row * q_ld + 32 * ks + 8 * kg) : ld128(Qr + row * qr_ld + 32 * (ks - KL) + 8 * kg);

  // ---- fragment lane offsets in a slot.  K (A operand): token l16, chunk
  // 4 ks + kg at (..) ^ swz: the swizzle flips bits 1..3 of the chunk, so four
  // offsets repeat every 256 bytes.  V^T (A operand) by transposing reads:
  // lane 4j + a of group kg reads token 4 kg + j, columns 16 vt + 4a .. +3. ----
  uint32_t koff[4], kroff[2];
#pragma unroll
  for (int m = 0; m < 4; ++m) koff[m] = l16 * 1024 + 16 * ((4 * m + kg) ^ swz_l(l16));
#pragma unroll
  for (int m = 0; m < 2; ++m) kroff[m] = LAT_B + l16 * 128 + 16 * ((4 * m + kg) ^ swz_r(l16));
  const int vrow = 4 * kg + ((lane >> 2) & 3), va = lane & 3;
  uint32_t voff[8];
#pragma unroll
  for (int m = 0; m < 8; ++m) voff[m] = vrow * 1024 + 16 * ((2 * m + (va >> 1)) ^ swz_l(vrow)) + 8 * (va & 1);

  f32x4 acc[VT];
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) acc[vt] = f32x4{};
  float m_run = -1e30f, l_run = 0.f;
  land_args(O, ws_o, ws_ml);
  // Q and the first two blocks, in flight together, land here: the loop's
  // waits then count the direct loads alone.
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]));

  for (int i = 0; i < cnt; ++i) {
    // block i landed once at most the LPB loads of block i + 1 are in flight
    if (i + 1 < cnt)
      asm volatile("s_waitcnt vmcnt(%0)" ::"i"(LPB) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const uint32_t st = ring + (i & 1) * SLOT;

    // ---- scores, in two chains ----
    f32x4 sc[2] = {f32x4{}, f32x4{}};
    auto kread = [&](int ks) { return lds_ld128(st + (ks < KL ? koff[ks & 3] + 256 * (ks >> 2) : kroff[ks - KL])); };
    u32x4 kf[8];
#pragma unroll
    for (int ks = 0; ks < LA; ++ks) kf[ks] = kread(ks);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + LA < KS) kf[(ks + LA) & 7] = kread(ks + LA);
      sc[ks & 1] = mfma16<BF16>(kf[ks & 7], qf[ks], sc[ks & 1]);
      __builtin_amdgcn_sched_barrier(0);  // keep the read lookahead
    }
    // the first V^T fragments do not depend on the softmax
    auto vread = [&](int vt) { return lds_read_tr16_at(st + voff[vt & 7] + 256 * (vt >> 3)); };
    u32x2 vf[8];
#pragma unroll
    for (int vt = 0; vt < LA; ++vt) vf[vt] = vread(vt);

    // ---- softmax of head l16 over tokens tb + 4 kg + j ----
    const int tb = t0 + (wave + NW * i) * BT;
    f32x4 x = sc[0] + sc[1];
    if (tb + BT > t1) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (tb + 4 * kg + j >= t1) x[j] = -INFINITY;
    }
    const float mx = max_xor32(max_xor16(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])))) * sl2;
    // lazy running max: O and l are rescaled only when a block's max exceeds
    // it by more than 2^kLazy
    if (__any(mx > m_run + kLazy)) {
      const float m_new = fmaxf(m_run, mx);
      const float corr = __builtin_amdgcn_exp2f(m_run - m_new);
      m_run = m_new;
      l_run *= corr;
      if (i > 0) {  // still zero at the first block
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) acc[vt] *= corr;
      }
    }
    float p[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) p[j] = __builtin_amdgcn_exp2f(fmaf(x[j], sl2, -m_run));
    const u32x2 pf{pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3])};
    l_run = dot2_ones<BF16>(pf[1], dot2_ones<BF16>(pf[0], l_run));

    // ---- values ----
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) {
      if (vt + LA < VT) vf[(vt + LA) & 7] = vread(vt + LA);
      acc[vt] = mfma_k16(vf[vt & 7], pf, acc[vt]);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (i + 2 < cnt) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // every read of the slot is done before it is refilled
      issue(i + 2);
    }
  }

  // ---- the waves' states meet: m and l, then the O^T tiles, [wave][vt][lane]
  // x 16 B, wave w summing column tiles 8 w .. 8 w + 7 ----
  const float l_tot = sum_xor32(sum_xor16(l_run));
  if (kg == 0) {
    ml[0][wave][l16] = m_run;
    ml[1][wave][l16] = l_tot;
  }
  constexpr int TPW = VT / NW;
  f32x4* red = reinterpret_cast<f32x4*>(smem);
  __syncthreads();  // the rings are no longer read
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) red[(wave * VT + vt) * 64 + lane] = acc[vt];
  __syncthreads();
  float mx = -1e30f, w[NW], l = 0.f;
#pragma unroll
  for (int v = 0; v < NW; ++v) mx = fmaxf(mx, ml[0][v][l16]);
#pragma unroll
  for (int v = 0; v < NW; ++v) {
    w[v] = __builtin_amdgcn_exp2f(ml[0][v][l16] - mx);
    l += w[v] * ml[1][v][l16];
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const size_t tile = (size_t)b * nsplit + s;
  if (nsplit > 1 && wave == 0 && kg == 0) *reinterpret_cast<float2*>(ws_ml + tile * 32 + 2 * l16) = float2{mx, l};
#pragma unroll
  for (int u = 0; u < TPW; ++u) {
    const int vt = wave * TPW + u;
    f32x4 o{};
#pragma unroll
    for (int v = 0; v < NW; ++v) o += w[v] * red[(v * VT + vt) * 64 + lane];
    const u32x2 y{pack_bf16x2(o[0] * inv, o[1] * inv), pack_bf16x2(o[2] * inv, o[3] * inv)};
    if (nsplit > 1)
      st64(ws_o + ((tile * VT + vt) * 64 + lane) * 2, y);
    else if (l16 < H)
      st64(O + ((size_t)b * H + l16) * DV + 16 * vt + 4 * kg, y);
  }
}

Split few_split(int B, int T) {
  // As many splits as one round of workgroups takes, with two blocks per wave
  // at least (below that the merge costs more than it saves), and 128 at most.
  const int nblk = (T + BT - 1) / BT;
  int ns = 256 / B;
  if (ns > nblk / (2 * NW)) ns = nblk / (2 * NW);
  if (ns > 128) ns = 128;
  if (ns < 1) ns = 1;
  const int per = (nblk + ns - 1) / ns;
  return Split{(nblk + per - 1) / per, per * BT};
}

int launch_few(const void* Q, const void* Qr, int q_ld, int qr_ld, const void* KV, void* O, uint32_t* ws_o,
               float* ws_ml, int B, int H, int T, float sl2, const Split& sp, hipStream_t s) {
  MX_RETURN_IF_HIP(lds_limit_once<mla_decode_few_kernel>(RING));
  hipLaunchKernelGGL(mla_decode_few_kernel, dim3((unsigned)((long long)B * sp.nsplit)), dim3(64 * NW), RING, s,
                     (const uint16_t*)Q, (const uint16_t*)Qr, (const uint16_t*)KV, (uint16_t*)O, ws_o, ws_ml, B, H, T,
                     sl2, sp.nsplit, sp.tps, q_ld, qr_ld);
  MX_RETURN_IF_HIP(hipGetLastError());
  return MX_OK;
}

}  // namespace mla
}  // namespace mx
