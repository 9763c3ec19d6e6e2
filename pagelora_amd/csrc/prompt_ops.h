// Prompt-sized forms of the fused element-wise kernels with a LoRA
// up-projection (prompt_ops.hip), chosen by their entry points in
// fused_ops.hip: one adapter bound to every token, 16-bit types.
#pragma once
#include "lora_up.h"

namespace pl {
namespace prompt {

// From these rows on the tokens share their adapter's B rows through MFMA
// tiles; fewer take the row kernels, which read B once per token.
// SiLU*up x 12288, row kernel -> tiles: 24 rows 5.8 -> 5.5 us, 64 8.6 -> 5.6,
// 256 26.5 -> 8.7, 2112 264 -> 40.
constexpr int kMinRows = 24;
// q/k norm + RoPE + append, 48 heads: 2112 rows 45 -> 21 us, 512 rows 16.8 ->
// 13.9, but a tile's chain of three heads costs 11 us where the row kernel
// takes 5.5 (77 rows).
constexpr int kMinQkrRows = 512;

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

// Whether the tile kernels take a call's modules.
inline bool takes(int rows, const LoraUp& m) {
  return rows >= kMinRows && m.adapter >= 0 && (m.rank == 8 || m.rank == 16 || m.rank == 32);
}
// ... and the q/k norm + RoPE + append's layout: head_dim 128, 16-byte chunks everywhere.
bool takes_qkr(const QkrTileArgs& a, int head_dim);

void silu_mul(const void* gu, int64_t ldg, void* out, int64_t ldo, int rows, int inter, const LoraUp& lg,
              const LoraUp& lu, bool bf16, hipStream_t s);
void qk_norm_rope_append(const QkrTileArgs& a, bool bf16, hipStream_t s);

}  // namespace prompt
}  // namespace pl
