// Arguments and the host entry of the GEMM on shuffled weights past decode's
// 16 tokens (wide_gemm.hip).
#pragma once

#include "pl_common.h"

namespace pl {
namespace wgemm {

struct StripArgs {
  const void* x;
  const void* W;
  const void* bias;
  void* out;
  int64_t ldx, ldo;
  int tokens, K, N, m_tiles;
};

struct TileArgs {
  const void* x;
  const void* W;
  const void* bias;
  void* out;
  float* partial;  // splits > 1: planes [splits][tokens][ldp]
  int64_t ldx, ldo, ldp;
  int tokens, K, N, m_tiles, n_tiles, splits, vec_out;
};

// Where split s of `splits` (a power of two) begins, in 64-wide steps of K.
// An even division: with steps >= splits every split has at least one step
// (ceil(steps / splits) steps each would leave the last of 8 splits of 33
// steps empty, and a workgroup loads its first step unasked).
__host__ __device__ inline int split_begin(int steps, int splits, int s) {
  return (int)(((unsigned)steps * (unsigned)s) / (unsigned)splits);
}

// 32-bit byte offsets reach every row of a token tile.
bool wide_supports(int64_t ldx);

// out = x . W^T (+ bias); arguments checked by the caller.  ws (nullable)
// holds a K split's planes where one pays.  kTakeRows16, and nothing done,
// where linear_rows16 is the faster one (up to 64 tokens).
constexpr int kTakeRows16 = -1;
int wide_linear(const void* x, int64_t ldx, int tokens, int K, const void* W, int N, const void* bias, void* out,
                int64_t ldo, void* ws, size_t ws_bytes, int dtype, hipStream_t s);

// The decode GEMM on 16-token tiles (skinny_gemm.hip), each of which streams W.
int linear_rows16(const void* x, int64_t ldx, int tokens, int K, const void* W, int N, const void* bias, void* out,
                  int64_t ldo, int dtype, hipStream_t s);

}  // namespace wgemm
}  // namespace pl
