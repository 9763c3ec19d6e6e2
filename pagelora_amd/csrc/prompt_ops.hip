// Prompt-sized SiLU*up and q/k norm + RoPE + KV append with their LoRA
// up-projections (gfx950): the arithmetic and roundings of the row
// kernels of fused_ops.hip, for rows that all use one adapter.
//
// The row kernels read a module's whole B once per token: 512 bytes of B for
// 48 bytes of SiLU's own traffic.  Here a wave takes 16 tokens x 64 columns
// with one MFMA per 16 columns (the up to 32 ranks are one k-step), B in
// registers over the wave's token tiles, in a column order that leaves each
// lane runs of eight consecutive columns of one token: the rows are read and
// written in 16-byte chunks, 64 bytes of a row per instruction.  2112 rows:
// SiLU*up (12288 columns) 264 -> 40 us, 3.9 TB/s of its own traffic; q/k norm
// + RoPE + append (48 heads) 45 -> 21 us, bound by its angles and latency.
#include <type_traits>

#include "prompt_ops.h"

namespace pl {
namespace prompt {

constexpr int kWave = 64;
constexpr int kThreads = 256;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T> __device__ __forceinline__ f32x4 mfma32(uint4 a, uint4 b, f32x4 c);
template <> __device__ __forceinline__ f32x4 mfma32<bf16_t>(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}
template <> __device__ __forceinline__ f32x4 mfma32<f16_t>(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                0);
}

template <typename T> __device__ __forceinline__ void unpack8(uint4 w, float (&f)[8]) {
  unpack2<T>(w.x, f[0], f[1]);
  unpack2<T>(w.y, f[2], f[3]);
  unpack2<T>(w.z, f[4], f[5]);
  unpack2<T>(w.w, f[6], f[7]);
}
template <typename T> __device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
  return make_uint4(pack2<T>(f[0], f[1]), pack2<T>(f[2], f[3]), pack2<T>(f[4], f[5]), pack2<T>(f[6], f[7]));
}
__device__ __forceinline__ uint4 load16(const void* p) { return *reinterpret_cast<const uint4*>(p); }

// The B operand of 32 columns from c0 (c0 % 32 == 0) as two MFMAs': operand
// row i of MFMA n is column c0 + 8 (i / 4) + 4 n + i % 4, so that a lane's
// results of the two are columns c0 + 8 grp .. +8.  Columns past the module's
// read its last one (their results are not used), ranks past R are zero.
template <typename T, int R>
__device__ __forceinline__ void load_b32(const LoraUp& m, int c0, uint4 (&b)[2]) {
  const int lr = threadIdx.x % 16, grp = threadIdx.x % kWave / 16;
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int c = min(c0 + (lr >> 2) * 8 + n * 4 + (lr & 3), m.out_features - 1);
    b[n] = grp * 8 < R ? *lora_b_piece<T, R>(m, m.adapter, c & ~7, c & 7, grp) : make_uint4(0, 0, 0, 0);
  }
}
// The intermediate of token `row` as the other operand.
template <typename T, int R>
__device__ __forceinline__ uint4 load_y32(const LoraUp& m, int row) {
  const int grp = threadIdx.x % kWave / 16;
  return grp * 8 < R ? load16((const T*)m.y + (int64_t)row * m.ldy + m.y_offset + (int64_t)m.adapter * R + grp * 8)
                     : make_uint4(0, 0, 0, 0);
}
// v (8 columns) + scale * y . B^T, rounded through T.
template <typename T>
__device__ __forceinline__ void add_delta8(float (&v)[8], const uint4 (&b)[2], uint4 y, float scale) {
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
  const f32x4 d0 = mfma32<T>(b[0], y, z), d1 = mfma32<T>(b[1], y, z);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = through<T>(v[i] + d0[i] * scale);
    v[4 + i] = through<T>(v[4 + i] + d1[i] * scale);
  }
}

// ------------------------------------------------------------- SiLU * up ---
constexpr int kSiluTiles = 2;  // token tiles per wave: B's reads stay below a third of the rows' own

template <typename T, int R>
__global__ __launch_bounds__(kThreads) void silu_mul_tile_kernel(const T* __restrict__ gu, int64_t ldg,
                                                                 T* __restrict__ out, int64_t ldo, int rows, int inter,
                                                                 LoraUp lg, LoraUp lu) {
  const int lane = threadIdx.x % kWave, wave = uniform(threadIdx.x / kWave);
  const int lr = lane % 16, grp = lane / 16;
  const int c0 = (blockIdx.x * (kThreads / kWave) + wave) * 64;
  if (c0 >= inter) return;
  const int row0 = blockIdx.y * (16 * kSiluTiles);
  uint4 g[kSiluTiles][2], u[kSiluTiles][2], yg[kSiluTiles], yu[kSiluTiles], bg[2][2], bu[2][2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    load_b32<T, R>(lg, c0 + q * 32, bg[q]);
    load_b32<T, R>(lu, c0 + q * 32, bu[q]);
  }
  int row[kSiluTiles];
#pragma unroll
  for (int t = 0; t < kSiluTiles; ++t) {
    row[t] = row0 + t * 16 + lr;
    const int rc = min(row[t], rows - 1);
    yg[t] = load_y32<T, R>(lg, rc);
    yu[t] = load_y32<T, R>(lu, rc);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const T* p = gu + (int64_t)rc * ldg + min(c0 + q * 32 + grp * 8, inter - 8);
      g[t][q] = load16(p);
      u[t][q] = load16(p + inter);
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load in flight
#pragma unroll
  for (int t = 0; t < kSiluTiles; ++t)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      float gf[8], uf[8], o[8];
      unpack8<T>(g[t][q], gf);
      unpack8<T>(u[t][q], uf);
      add_delta8<T>(gf, bg[q], yg[t], lg.scale);
      add_delta8<T>(uf, bu[q], yu[t], lu.scale);
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = gf[i] / (1.f + expf(-gf[i])) * uf[i];
      const int c = c0 + q * 32 + grp * 8;
      if (row[t] < rows && c < inter) *reinterpret_cast<uint4*>(out + (int64_t)row[t] * ldo + c) = pack8<T>(o);
    }
}

// ------------------------------------------- q/k norm + RoPE + KV append ---
constexpr int kQkrHeads = 3;   // heads per wave: a workgroup's 12 share its tokens' angles
constexpr int kD = 128;
constexpr int kCsPitch = kD + 4;  // floats of a token's (cos, sin) pairs; +4 spreads the rows over the banks

template <typename T, int R>
__global__ __launch_bounds__(kThreads) void qkr_tile_kernel(QkrTileArgs A) {
  __shared__ __align__(16) float s_cs[16 * kCsPitch];
  const int lane = threadIdx.x % kWave, wave = uniform(threadIdx.x / kWave);
  const int lr = lane % 16, grp = lane / 16;
  const int row = blockIdx.y * 16 + lr, rc = min(row, A.rows - 1);
  const int heads = A.hq + 2 * A.hkv;
  for (int i = threadIdx.x; i < 16 * kD / 2; i += kThreads) {
    const int t = i / (kD / 2), pair = i % (kD / 2);
    float sn, cs;
    sincosf((float)A.pos[min((int)blockIdx.y * 16 + t, A.rows - 1)] * A.invf[pair], &sn, &cs);
    s_cs[t * kCsPitch + pair * 2] = cs;
    s_cs[t * kCsPitch + pair * 2 + 1] = sn;
  }
  const int64_t page = A.pid[rc], off = A.off[rc];
  const bool slot_ok = page >= 0 && page < A.np && off >= 0 && off < A.page_size;
  const int64_t slot = page * A.ps + off * A.ts;
  __syncthreads();
#pragma unroll 1
  for (int k = 0; k < kQkrHeads; ++k) {
    const int h = (blockIdx.x * kQkrHeads + k) * (kThreads / kWave) + wave;
    if (h >= heads) return;
    const bool is_q = h < A.hq, is_k = !is_q && h < A.hq + A.hkv;
    const int hm = h - (is_q ? 0 : (is_k ? A.hq : A.hq + A.hkv));  // head within its module
    const LoraUp& m = A.m[is_q ? 0 : (is_k ? 1 : 2)];
    const T* nw = (const T*)(is_q ? A.qn : (is_k ? A.kn : nullptr));
    uint4 in[4], b[4][2], wv[4];
    const uint4 y = load_y32<T, R>(m, rc);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      load_b32<T, R>(m, hm * kD + q * 32, b[q]);
      in[q] = load16((const T*)A.qkv + (int64_t)rc * A.ld + (int64_t)h * kD + q * 32 + grp * 8);
      if (nw != nullptr) wv[q] = load16(nw + q * 32 + grp * 8);
    }
    float v[4][8];
    float ss = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      unpack8<T>(in[q], v[q]);
      add_delta8<T>(v[q], b[q], y, m.scale);
#pragma unroll
      for (int i = 0; i < 8; ++i) ss = fmaf(v[q][i], v[q][i], ss);
    }
    if (is_q || is_k) {
      ss += __shfl_xor(ss, 16);
      ss += __shfl_xor(ss, 32);
      const float rstd = nw != nullptr ? rsqrtf(ss / (float)kD + A.eps) : 1.f;
#pragma unroll
      for (int q = 0; q < 2; ++q) {  // pairs (d, d + 64)
        float wl[8], wh[8];
        if (nw != nullptr) {
          unpack8<T>(wv[q], wl);
          unpack8<T>(wv[q + 2], wh);
        }
        const float* cs = &s_cs[lr * kCsPitch + (q * 32 + grp * 8) * 2];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float2 a = *reinterpret_cast<const float2*>(cs + i * 2);
          const float lo = v[q][i] * (nw != nullptr ? rstd * wl[i] : rstd);
          const float hi = v[q + 2][i] * (nw != nullptr ? rstd * wh[i] : rstd);
          v[q][i] = lo * a.x - hi * a.y;
          v[q + 2][i] = hi * a.x + lo * a.y;
        }
      }
    }
    T* dst = is_q ? (T*)A.q_out + ((int64_t)rc * A.hq + h) * kD
                  : (T*)(is_k ? A.kc : A.vc) + slot + (int64_t)hm * A.hs;
    if (row < A.rows && (is_q || slot_ok)) {  // a slot outside the pool is skipped, never written
#pragma unroll
      for (int q = 0; q < 4; ++q) *reinterpret_cast<uint4*>(dst + q * 32 + grp * 8) = pack8<T>(v[q]);
    }
  }
}

// ------------------------------------------------------------- host side ---
template <typename F>
static void by_rank(int rank, F f) {
  if (rank == 8) f(std::integral_constant<int, 8>{});
  else if (rank == 16) f(std::integral_constant<int, 16>{});
  else f(std::integral_constant<int, 32>{});
}

void silu_mul(const void* gu, int64_t ldg, void* out, int64_t ldo, int rows, int inter, const LoraUp& lg,
              const LoraUp& lu, bool bf16, hipStream_t s) {
  const dim3 grid((inter + 255) / 256, (rows + 16 * kSiluTiles - 1) / (16 * kSiluTiles));
  by_rank(lg.rank, [&](auto rank) {
    constexpr int R = decltype(rank)::value;
    if (bf16)
      hipLaunchKernelGGL((silu_mul_tile_kernel<bf16_t, R>), grid, dim3(kThreads), 0, s, (const bf16_t*)gu, ldg,
                         (bf16_t*)out, ldo, rows, inter, lg, lu);
    else
      hipLaunchKernelGGL((silu_mul_tile_kernel<f16_t, R>), grid, dim3(kThreads), 0, s, (const f16_t*)gu, ldg,
                         (f16_t*)out, ldo, rows, inter, lg, lu);
  });
}

bool takes_qkr(const QkrTileArgs& a, int head_dim) {
  const void* ptrs[] = {a.qkv, a.qn, a.kn, a.q_out, a.kc, a.vc};
  for (const void* p : ptrs)
    if ((uintptr_t)p % 16) return false;
  return head_dim == kD && a.ld % 8 == 0 && a.ps % 8 == 0 && a.ts % 8 == 0 && a.hs % 8 == 0 &&
         a.rows >= kMinQkrRows && takes(a.m[0]) &&
         (int64_t)a.rows * (a.hq + 2 * a.hkv) >= (a.m[0].rank == 32 ? kMinQkrHeads32 : kMinQkrHeads);
}

void qk_norm_rope_append(const QkrTileArgs& a, bool bf16, hipStream_t s) {
  const int heads = a.hq + 2 * a.hkv, per = kQkrHeads * (kThreads / kWave);
  const dim3 grid((heads + per - 1) / per, (a.rows + 15) / 16);
  by_rank(a.m[0].rank, [&](auto rank) {
    constexpr int R = decltype(rank)::value;
    if (bf16)
      hipLaunchKernelGGL((qkr_tile_kernel<bf16_t, R>), grid, dim3(kThreads), 0, s, a);
    else
      hipLaunchKernelGGL((qkr_tile_kernel<f16_t, R>), grid, dim3(kThreads), 0, s, a);
  });
}

}  // namespace prompt
}  // namespace pl
