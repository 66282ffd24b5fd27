// What the MLA decode kernels share: widths, the split of a sequence's
// tokens and the layout of its partial results.
#pragma once

#include "mx_common.h"

namespace mx {
namespace mla {

constexpr int DQK = 576;                // latent + rope
constexpr int DV = 512;                 // latent
constexpr int ROW_B = DQK * 2;          // 1152 bytes per cache row in HBM
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLazy = 16.0f;          // log2 headroom before a rescale

// The tokens of a sequence go to nsplit slices of tps tokens.
struct Split {
  int nsplit;
  int tps;
};

// Decode with up to 16 heads (mla_decode_few.hip).  Its partial results come
// in tiles of 16 heads (kFewTile), the 128-head kernel's in tiles of 32.
constexpr int kFewHeads = 16;
constexpr int kFewTile = 16;
Split few_split(int B, int T);
int launch_few(const void* Q, const void* Qr, int q_ld, int qr_ld, const void* KV, void* O, uint32_t* ws_o,
               float* ws_ml, int B, int H, int T, float sl2, const Split& sp, hipStream_t s);

}  // namespace mla
}  // namespace mx
