// Prompt-sized forms of the fused element-wise kernels with a LoRA
// up-projection (prompt_ops.hip), chosen by their entry points in
// fused_ops.hip: one adapter bound to every token, 16-bit types.
#pragma once
#include "lora_up.h"

namespace pl {
namespace prompt {

// Where the tokens share their adapter's B rows through MFMA tiles; elsewhere
// the row kernels, which read B once per token.
// SiLU*up: a call of the tiles takes 5.2 us at least, the row kernel 3.8 where
// it fills no CU; the line is where its reads of B pass that.  us, row kernel
// against tiles, rank 16 (8): 100 x 2048 5.2, 5.8 (4.3, 5.7); 24 x 11008 6.2,
// 5.8 (4.9, 5.7); 64 x 12288 10.9, 6.1 (7.5, 6.0); 2112 x 12288 243, 37.5; many
// rows of few columns launch many workgroups: 1000 x 64 7.2, 5.4 (6.2, 5.3).
// Rank 32's two passes over B: 24 x 64 8.0, 5.1.
constexpr int kMinRows = 24, kManyRows = 1000;
constexpr int64_t kMinSiluB = 4 << 20;  // rows x columns x rank
// q/k norm + RoPE + append: a tile's chain of three heads costs 11 us.  Rank 16
// (8): 512 rows x 36 heads 14.3, 14.4 (14.0, 14.4); 600 x 36 16.3, 14.7 (15.5,
// 15.0); 1000 x 6 10.1, 12.4; 2112 x 48 48.1, 23.9.  Rank 32: 1000 x 6 11.6,
// 11.8.
constexpr int kMinQkrRows = 512;
constexpr int64_t kMinQkrHeads = 18000, kMinQkrHeads32 = 6000;  // rows x heads

struct QkrTileArgs {
  const void *qkv, *qn, *kn;
  int64_t ld;
  const int64_t *pos, *pid, *off;
  void *q_out, *kc, *vc;
  int64_t ps, ts, hs, np;
  int page_size, rows, hq, hkv;
  const float* invf;
  float eps;
  LoraUp m[3];
};

// Whether the tile kernels take a call's modules, and SiLU*up's sizes ...
inline bool takes(const LoraUp& m) { return m.adapter >= 0 && (m.rank == 8 || m.rank == 16 || m.rank == 32); }
inline bool takes_silu(int rows, int inter, const LoraUp& m) {
  return takes(m) && rows >= kMinRows &&
         (m.rank == 32 || rows >= kManyRows || (int64_t)rows * inter * m.rank >= kMinSiluB);
}
// ... and the q/k norm + RoPE + append's layout: head_dim 128, 16-byte chunks everywhere.
bool takes_qkr(const QkrTileArgs& a, int head_dim);

void silu_mul(const void* gu, int64_t ldg, void* out, int64_t ldo, int rows, int inter, const LoraUp& lg,
              const LoraUp& lu, bool bf16, hipStream_t s);
void qk_norm_rope_append(const QkrTileArgs& a, bool bf16, hipStream_t s);

}  // namespace prompt
}  // namespace pl
