// GEMM on pre-shuffled weights (gfx950) past decode's 16 tokens:
// out = x . W^T (+ bias) with W in pl_weight_shuffle's 1 KiB blocks (16 rows
// x 32 k in MFMA lane order), so prefill and large decode batches read the
// one stored copy of the weight instead of a row-major one.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "wide_gemm.h"

namespace pl {
namespace wgemm {

constexpr int kWave = 64;
constexpr int kBlockBytes = 1024;  // 16 rows x 32 k

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

template <typename T> __device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c);
template <> __device__ __forceinline__ f32x4 mfma32<bf16_t>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}
template <> __device__ __forceinline__ f32x4 mfma32<f16_t>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                0);
}

// ------------------------------------------------------------ strip kernel ---
// One workgroup of 16 waves per NF*16 output columns x MF*16 tokens; the
// waves split K (wave w: 32-wide steps w*per .. of ceil(steps / 16)), so
// every weight byte is read once per token tile straight into MFMA
// registers, and the 16 partial tiles are summed in wave order through LDS:
// the order of shuffled_gemm_kernel's sums, whose results it reproduces.
constexpr int kStripWaves = 16;
constexpr int kStripThreads = kStripWaves * kWave;

template <typename T, int MF, int NF, int U>
__global__ __launch_bounds__(kStripThreads) void strip_gemm_kernel(StripArgs g) {
  // a round of the cross-wave sum covers 4 16x16 tiles: one cell per thread
  constexpr int kRound = 4;
  constexpr int kTiles = MF * NF;
  __shared__ __align__(16) float s_red[kStripWaves][kRound * 256];
  const int lane = threadIdx.x % kWave, wave = uniform(threadIdx.x / kWave);
  const int lr = lane % 16, grp = lane / 16;
  const int ct = blockIdx.x / g.m_tiles, mt = blockIdx.x % g.m_tiles;  // column tile, token tile
  const int t0 = mt * (MF * 16);
  const int ksteps = g.K / 32;
  const int per = (ksteps + kStripWaves - 1) / kStripWaves;
  const int sb = min(ksteps, wave * per), se = min(ksteps, sb + per);
  const int n_blocks = (g.N + 15) / 16;
  // rows and blocks past the end read the last one: their results are not stored
  const char* wb[NF];
#pragma unroll
  for (int n = 0; n < NF; ++n)
    wb[n] = (const char*)g.W + (int64_t)min(ct * NF + n, n_blocks - 1) * ksteps * kBlockBytes;
  const char* xb = (const char*)g.x + (int64_t)t0 * g.ldx * 2;
  uint32_t xoff[MF];
#pragma unroll
  for (int m = 0; m < MF; ++m)
    xoff[m] = (uint32_t)(min(m * 16 + lr, g.tokens - 1 - t0) * (int)g.ldx * 2 + grp * 16);
  const uint32_t woff = lane * 16;

  f32x4 acc[MF][NF];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int n = 0; n < NF; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  int s = sb;
  for (; s + U <= se; s += U) {
    u32x4 w[U][NF], a[U][MF];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int n = 0; n < NF; ++n)
        w[u][n] = *reinterpret_cast<const u32x4*>(wb[n] + (int64_t)(s + u) * kBlockBytes + woff);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < MF; ++m)
        a[u][m] = *reinterpret_cast<const u32x4*>(xb + (s + u) * 64 + xoff[m]);
    __builtin_amdgcn_sched_barrier(0);  // a batch's loads before its first MFMA
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int n = 0; n < NF; ++n) acc[m][n] = mfma32<T>(w[u][n], a[u][m], acc[m][n]);
  }
  for (; s < se; ++s) {
    u32x4 w[NF], a[MF];
#pragma unroll
    for (int n = 0; n < NF; ++n) w[n] = *reinterpret_cast<const u32x4*>(wb[n] + (int64_t)s * kBlockBytes + woff);
#pragma unroll
    for (int m = 0; m < MF; ++m) a[m] = *reinterpret_cast<const u32x4*>(xb + s * 64 + xoff[m]);
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
      for (int n = 0; n < NF; ++n) acc[m][n] = mfma32<T>(w[n], a[m], acc[m][n]);
  }

  // tile j = m * NF + n; lane: token lr of m, columns 4*grp .. +4 of n
  constexpr int kRounds = (kTiles + kRound - 1) / kRound;
#pragma unroll
  for (int r = 0; r < kRounds; ++r) {
    if (r > 0) __syncthreads();
#pragma unroll
    for (int j = 0; j < kRound; ++j) {
      const int tile = r * kRound + j;
      if (tile < kTiles)
        *reinterpret_cast<f32x4*>(&s_red[wave][j * 256 + lr * 16 + grp * 4]) = acc[tile / NF][tile % NF];
    }
    __syncthreads();
    // thread -> cell: 16 columns of a token, the NF tiles of a token side by side
    const int cell = threadIdx.x % 16;
    const int q = threadIdx.x / 16;  // 0..63: (tile of the round, token) pairs
    int j, tok;
    if constexpr (NF == 1) {
      j = q / 16;
      tok = q % 16;
    } else if constexpr (NF == 2) {
      j = (q / 32) * 2 + q % 2;
      tok = (q / 2) % 16;
    } else {
      j = q % 4;
      tok = q / 4;
    }
    const int tile = r * kRound + j;
    const int t = t0 + (tile / NF) * 16 + tok;
    const int c = (ct * NF + tile % NF) * 16 + cell;
    if (tile < kTiles && t < g.tokens && c < g.N) {
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < kStripWaves; ++w) sum += s_red[w][j * 256 + tok * 16 + cell];
      if (g.bias != nullptr) sum += to_float<T>(((const T*)g.bias)[c]);
      ((T*)g.out)[(int64_t)t * g.ldo + c] = from_float<T>(sum);
    }
  }
}

// ------------------------------------------------------------- tile kernel ---
// 8 waves side by side over the columns, each NF 16-column blocks x the
// workgroup's MF*16 tokens; K in steps of 64, S steps in flight.  x goes
// through LDS by asynchronous global->LDS loads (S buffers), W straight from
// its shuffled blocks into registers (no other wave needs them), both issued
// S - 1 steps ahead of their use and spread over the step's MFMAs.
// Bound by the MFMAs where tiles are many (24608 x 4096, 2112 tokens, 192 x
// 384 tiles: 327 us, 1.30 PFLOP/s; MFMAs and LDS reads alone take 1.06 us of a
// 256 x 256 tile's step) and by the weight stream where tokens are few (64
// tokens: 41 us, 4.9 TB/s).  What got it there, 256 x 256 tiles at 2112
// tokens: waves 2 x 4 with one step in flight 550 us, two steps in flight and
// whole 128-byte lines of x per load 428 us, waves 1 x 8 (each weight block
// loaded by one wave, not two) 369 us.  The library GEMM it replaces took 437
// us, and 33 us to write the row-major weight it reads.
// A last half step (K an odd multiple of 32) goes round LDS: 4112 x 2080, 2112
// tokens, 42 us, where the strip kernel, which streams the weights once per 64
// tokens, took 222.
constexpr int kTileThreads = 512;

// s_waitcnt vmcnt(N) as the compiler's own instruction (exp and lgkm counts
// open), so that it knows which asynchronous LDS loads are done.
template <int N> __device__ __forceinline__ void wait_vm() {
  static_assert(N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0xF70);
}

// A buffer of `bytes` from p on; loads past it read 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (uint32_t)min(bytes, (int64_t)0xffffffff),
                                           0x00027000);
}

template <typename T, int MF, int NF, int S>
__device__ __forceinline__ void tile_gemm(const TileArgs& g) {
  constexpr int BM = 16 * MF;
  constexpr int XB = BM / 8;            // 1 KiB x blocks per 64-wide step: 8 rows x 64 k
  constexpr int XPW = (XB + 7) / 8;     // per wave (a wave past the end repeats the last block)
  constexpr int kBuf = XB * kBlockBytes;
  constexpr int kLoads = XPW + 2 * NF;  // per wave and step
  // one object per buffer: loads into one never alias reads of another
  __shared__ __align__(16) char s_x0[kBuf];
  __shared__ __align__(16) char s_x1[kBuf];
  __shared__ __align__(16) char s_x2[kBuf];
  __shared__ __align__(16) char s_x3[S > 3 ? kBuf : 16];
  __shared__ __align__(16) char s_x4[S > 4 ? kBuf : 16];
  __shared__ __align__(16) char s_x5[S > 5 ? kBuf : 16];
  auto buf = [&](int i) -> char* {
    return i == 0 ? s_x0 : i == 1 ? s_x1 : i == 2 ? s_x2 : i == 3 ? s_x3 : i == 4 ? s_x4 : s_x5;
  };
  const int lane = threadIdx.x % kWave, wave = uniform(threadIdx.x / kWave);
  const int lr = lane % 16, grp = lane / 16;
  // workgroup -> tile: consecutive workgroups land on different XCDs; each
  // XCD gets a contiguous run of tiles (token tiles fastest), which share
  // their weight blocks in its L2
  int id = blockIdx.x;
  {
    const int n = gridDim.x, per = n / 8, rem = n % 8;
    const int xcd = id % 8, idx = id / 8;
    id = xcd * per + min(xcd, rem) + idx;
  }
  const int mt = id % g.m_tiles, nt = (id / g.m_tiles) % g.n_tiles, split = id / (g.m_tiles * g.n_tiles);
  const int t0 = mt * BM;
  const int all_steps = g.K / 64;
  const int step0 = split_begin(all_steps, g.splits, split);
  const int steps = split_begin(all_steps, g.splits, split + 1) - step0;  // >= 1
  const int ksteps = g.K / 32;
  const int n_blocks = (g.N + 15) / 16;
  const int nb0 = nt * (8 * NF) + wave * NF;

  // buffer descriptors: the wave's weight blocks and the tile's x rows, each
  // to its tensor's end (blocks, rows and steps past the last are clamped to
  // it), offsets in scalar registers
  const int nbc = min(nb0, n_blocks - 1);
  const int64_t w_at = ((int64_t)nbc * ksteps + 2 * step0) * kBlockBytes, x_at = (int64_t)t0 * g.ldx * 2 + step0 * 128;
  const auto wr = make_rsrc((const char*)g.W + w_at, (int64_t)n_blocks * ksteps * kBlockBytes - w_at);
  const auto xr = make_rsrc((const char*)g.x + x_at, ((int64_t)(g.tokens - 1) * g.ldx + g.K) * 2 - x_at);
  int wso[NF];
#pragma unroll
  for (int n = 0; n < NF; ++n) wso[n] = uniform((min(nb0 + n, n_blocks - 1) - nbc) * ksteps * kBlockBytes);
  const int woff = lane * 16;
  // Lane l of an x block fetches row l/8, 16-byte chunk (l%8)^(l/8) of the
  // row's 128-byte line, so that the fragment reads (16 rows, one chunk) hit
  // every bank once.
  int xoff[XPW], xblk[XPW];
#pragma unroll
  for (int j = 0; j < XPW; ++j) {
    xblk[j] = min(wave * XPW + j, XB - 1);
    xoff[j] = min(xblk[j] * 8 + lane / 8, g.tokens - 1 - t0) * (int)g.ldx * 2 + ((lane % 8) ^ (lane / 8)) * 16;
  }
  auto load_x = [&](int step, char* dst) {
#pragma unroll
    for (int j = 0; j < XPW; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          xr, (__attribute__((address_space(3))) void*)(dst + xblk[j] * kBlockBytes), 16, xoff[j], step * 128, 0, 0);
  };
  auto load_w = [&](int step, u32x4 (&d)[2][NF]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int n = 0; n < NF; ++n)
        d[h][n] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, woff, wso[n] + (2 * step + h) * kBlockBytes, 0));
  };
  int aoff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) aoff[h] = lr * 128 + ((h * 4 + grp) ^ (lr % 8)) * 16;
  f32x4 acc[MF][NF];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int n = 0; n < NF; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 w[S][2][NF];
  const int last = steps - 1;
#pragma unroll
  for (int p = 0; p < S - 1; ++p) {
    load_x(min(p, last), buf(p));
    load_w(min(p, last), w[p]);
    __builtin_amdgcn_sched_barrier(0);
  }
  wait_vm<(S - 2) * kLoads>();
  __builtin_amdgcn_s_barrier();
  auto body = [&](int step, char* cur, char* nxt, u32x4 (&wc)[2][NF], u32x4 (&wn)[2][NF]) {
    const int nx = min(step + S - 1, last);
    __builtin_amdgcn_sched_barrier(0);
    load_x(nx, nxt);
    load_w(nx, wn);
    u32x4 a[2][MF];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int m = 0; m < MF; ++m) a[h][m] = *reinterpret_cast<const u32x4*>(cur + aoff[h] + m * 2 * kBlockBytes);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int n = 0; n < NF; ++n) acc[m][n] = mfma32<T>(wc[h][n], a[h][m], acc[m][n]);
    // LDS reads kAhead fragments ahead of their MFMAs, the loads spread over them
    constexpr int kAhead = MF < 3 ? MF : 3;
    constexpr int kPer = (kLoads + 2 * MF - 1) / (2 * MF);
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);
#pragma unroll
    for (int i = 0; i < 2 * MF; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, NF, 0);
      if (i + kAhead < 2 * MF) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (i * kPer < kLoads) __builtin_amdgcn_sched_group_barrier(0x020, kPer, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    wait_vm<(S - 2) * kLoads>();  // the next step's operands are in place
    __builtin_amdgcn_s_barrier();
  };
  int step = 0;
  for (; step + S <= steps; step += S) {
#pragma unroll
    for (int i = 0; i < S; ++i) body(step + i, buf(i), buf((i + S - 1) % S), w[i], w[(i + S - 1) % S]);
  }
#pragma unroll
  for (int i = 0; i < S - 1; ++i)
    if (step + i < steps) body(step + i, buf(i), buf((i + S - 1) % S), w[i], w[(i + S - 1) % S]);
  wait_vm<0>();  // no load into LDS outlives the workgroup
  // an odd multiple of 32: the last split takes the last 32 k, as the strip
  // kernel does, straight into registers
  if (g.K % 64 != 0 && split == g.splits - 1) {
    u32x4 wt[NF];
#pragma unroll
    for (int n = 0; n < NF; ++n)
      wt[n] = *reinterpret_cast<const u32x4*>(
          (const char*)g.W + ((int64_t)min(nb0 + n, n_blocks - 1) * ksteps + ksteps - 1) * kBlockBytes + woff);
    const char* xt = (const char*)g.x + (int64_t)t0 * g.ldx * 2 + (g.K - 32) * 2 + grp * 16;
#pragma unroll
    for (int m = 0; m < MF; ++m) {
      const u32x4 a = *reinterpret_cast<const u32x4*>(xt + (int64_t)min(m * 16 + lr, g.tokens - 1 - t0) * g.ldx * 2);
#pragma unroll
      for (int n = 0; n < NF; ++n) acc[m][n] = mfma32<T>(wt[n], a, acc[m][n]);
    }
  }

  // lane: token lr of m tile, columns 4*grp .. +4 of n tile
#pragma unroll
  for (int m = 0; m < MF; ++m) {
    const int t = t0 + m * 16 + lr;
    if (t >= g.tokens) continue;
    if (g.splits > 1) {
      float* prow = g.partial + ((int64_t)split * g.tokens + t) * g.ldp;
#pragma unroll
      for (int n = 0; n < NF; ++n) {
        const int c = (nb0 + n) * 16 + grp * 4;
        if (c < g.ldp) *reinterpret_cast<f32x4*>(prow + c) = acc[m][n];
      }
      continue;
    }
    T* orow = (T*)g.out + (int64_t)t * g.ldo;
#pragma unroll
    for (int n = 0; n < NF; ++n) {
      const int c = (nb0 + n) * 16 + grp * 4;
      f32x4 v = acc[m][n];
      if (g.bias != nullptr) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += c + i < g.N ? to_float<T>(((const T*)g.bias)[c + i]) : 0.f;
      }
      if (c + 4 <= g.N && g.vec_out) {
        *reinterpret_cast<u32x2*>(orow + c) = u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (c + i < g.N) orow[c + i] = from_float<T>(v[i]);
      }
    }
  }
}

template <typename T, int MF, int NF, int S>
__global__ __launch_bounds__(kTileThreads) void tile_gemm_kernel(TileArgs g) {
  tile_gemm<T, MF, NF, S>(g);
}

// out[t][c] = the splits' partial sums in order (+ bias), one rounding.
template <typename T>
__global__ void split_sum_kernel(const float* __restrict__ partial, int splits, int64_t ldp, int tokens, int N,
                                 const T* __restrict__ bias, T* __restrict__ out, int64_t ldo, int vec_out) {
  const int c4 = (N + 3) / 4;
  const int64_t total = (int64_t)tokens * c4;
  const int64_t plane = (int64_t)tokens * ldp;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int t = (int)(i / c4), c = (int)(i % c4) * 4;
    const float* p = partial + (int64_t)t * ldp + c;
    f32x4 v = *reinterpret_cast<const f32x4*>(p);
    for (int s = 1; s < splits; ++s) {
      const f32x4 q = *reinterpret_cast<const f32x4*>(p + s * plane);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += q[e];
    }
    T* o = out + (int64_t)t * ldo + c;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (bias != nullptr && c + e < N) v[e] += to_float<T>(bias[c + e]);
    if (c + 4 <= N && vec_out) {
      *reinterpret_cast<u32x2*>(o) = u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < N) o[e] = from_float<T>(v[e]);
    }
  }
}

// ------------------------------------------------------------ host side ---
// Tile shapes (token fragments, column fragments per wave, steps in flight).
struct TileShape {
  int mf, nf, stages, per_cu;  // per_cu: workgroups a CU holds (registers, LDS)
};
constexpr TileShape kShapes[] = {{2, 1, 4, 4},  {3, 1, 4, 3},  {4, 1, 4, 3},  {5, 1, 4, 3},  {6, 1, 4, 3}, {8, 1, 4, 2},
                                 {12, 1, 4, 1}, {8, 2, 4, 1}, {12, 2, 3, 1}, {16, 2, 3, 1}, {10, 3, 3, 1}, {12, 3, 3, 1}};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);
constexpr int kCUs = 256;
constexpr int kStripMaxTokens = 32;
constexpr int kMaxSplitCells = 1 << 25;  // fp32 cells of a split's planes (128 MB)

struct Choice {
  int shape, splits;
  double us;
};

// The estimated time of every tile shape and K split, fitted to timings on
// MI355X (ten weights of 1000 .. 24608 outputs over K = 1024 .. 12288, 33 ..
// 2112 tokens; the shape taken is within 1.0 % of the fastest one in the
// geometric mean): a workgroup alone on its CU takes 0.34 + 0.024 u us per
// 64-wide step of u = mf * nf fragments per wave, plus four steps to fill and
// drain its pipeline; with every CU busy a step costs its MFMAs, 0.0485 u
// where u >= 24 and 0.067 u below, or its operands at the 52 KB/us that a CU
// gets out of the L2 (16 nf KB of weights, which every further token tile
// streams again, and 2 mf KB of x), whichever is more; the weights stream from
// memory at 5.3 TB/s; a split adds a launch and its planes' traffic.  Without
// the L2 term few tokens took tiles of 32 (77 x 24608 x 4096: 74 us, now 44).
static Choice choose(int tokens, int N, int K, bool allow_split) {
  Choice best{0, 1, 1e30};
  const int steps = K / 64;
  for (int i = 0; i < kNumShapes; ++i) {
    const TileShape& s = kShapes[i];
    const int u = s.mf * s.nf;
    const double alone = 0.34 + 0.024 * u;
    const double busy = std::max((u >= 24 ? 0.0485 : 0.067) * u, (16 * s.nf + 2 * s.mf) / 52.0);
    const int64_t tiles = (int64_t)((tokens + 16 * s.mf - 1) / (16 * s.mf)) * ((N + 128 * s.nf - 1) / (128 * s.nf));
    for (int sp = 1; sp <= (allow_split ? 8 : 1); sp *= 2) {
      if (sp > 1 && (steps < 4 * sp || (int64_t)tokens * N * sp > (int64_t)kMaxSplitCells)) break;
      const double r = (double)tiles * sp / kCUs;  // workgroups per CU
      double step_us;
      if (s.per_cu == 1) {
        const double whole = std::floor(r), part = r - whole;
        step_us = whole * std::max(alone, busy) + (part > 0 ? alone + std::max(0.0, busy - alone) * part : 0.0);
      } else {
        step_us = std::max(alone * std::ceil(r / s.per_cu), r > 1 ? std::ceil(r) * busy : 0.0);
      }
      const double mem = ((double)N * K * 2 + (double)tokens * K * 2) / 5.3e6;
      double us = 4.0 + std::max(step_us * ((steps + sp - 1) / sp + 4), mem);
      if (sp > 1) us += 4.5 + (double)tokens * N * 8 * sp / 8e6;
      if (us < best.us) best = Choice{i, sp, us};
    }
  }
  return best;
}

// linear_rows16's time back to back in a graph, fitted (sd 9 %) to 864 products
// of 33 .. 64 tokens, 1000 .. 8192 outputs, K = 1024 .. 12288: a workgroup's own
// chain, or the rounds of 256 workgroups, of which a further token tile costs
// less where it runs on the XCD that holds the same columns' weights
// (consecutive workgroups go round the eight XCDs).
static double rows16_us(int tokens, int N, int K) {
  const int nb = (N + 15) / 16, mt = (tokens + 15) / 16;
  const double more = mt - 1.5 + (tokens - 16 * (mt - 1)) / 32.0;  // token tiles past the first, the last by its fill
  return 2.0 + K * 1e-3 * std::max(1.05, 0.32 + 1.95 * nb * (1 + (nb % 8 ? 0.8 : 0.55) * more) / 256);
}

// Up to 64 tokens the 16-token kernel is still the faster one for few columns:
// its workgroups are 16 columns x 16 tokens, so all of them run at once where
// these kernels leave CUs idle.
struct Route {
  bool rows16;
  Choice c;  // tile kernel (K >= 64, more than kStripMaxTokens)
};
static Route route(int tokens, int N, int K, bool allow_split) {
  const int nb = (N + 15) / 16, mt = (tokens + 15) / 16;
  if (tokens <= 16) return {true, {}};
  // Against the strip kernel of two token tiles per workgroup, wherever the
  // 16-token kernel is one round: 32 tokens x 1000 x 8192 12.7 us against 17.9,
  // 1902 x 4096 8.0 against 10.2; 2854 x 4096 (358 workgroups) 13.0 against
  // 10.3; a second tile of one token costs it a whole one (17 x 1902 x 12288
  // 19.5 against 18.6).
  if (tokens <= kStripMaxTokens) return {tokens >= 18 && nb * mt <= kCUs, {}};
  if (K < 64) return {tokens <= PL_LINEAR_MAX_TOKENS, {}};  // no whole step for the tile kernel
  Choice c = choose(tokens, N, K, allow_split);
  if (tokens > PL_LINEAR_MAX_TOKENS) return {false, c};
  // Against the tile kernel, by their estimates back to back (choose's are of
  // calls alone) and by what a call takes the host, 9 us, 9.5 with a query for
  // the workspace and 13.7 with the allocation and a split's second launch:
  // 37 x 1902 x 2112 7.5 us against 8.6, enqueued alone 8.7 against 13.9; 37 x
  // 1902 x 6144 17.0 against 10.2.  A split that the host would bound gives way
  // to an unsplit call.
  auto cost = [](double us, double host) { return std::max(us, host) + 0.01 * us; };
  const double rows16 = cost(rows16_us(tokens, N, K), 9.0);
  if (c.splits == 1) return {rows16 <= cost(1.46 + 0.51 * (c.us - 4), 9.5), c};
  const double split = 0.73 + 0.82 * (c.us - 4);
  if (rows16 <= cost(split, 13.7)) return {true, c};
  if (split < 13.7) {
    const Choice one = choose(tokens, N, K, false);
    const double us = 1.46 + 0.51 * (one.us - 4);
    if (us < 13.0 && cost(us, 9.5) <= cost(split, 13.7)) c = one;
  }
  return {c.splits == 1 && rows16 <= cost(1.46 + 0.51 * (c.us - 4), 9.5), c};
}

static int64_t split_ld(int N) { return (int64_t)(N + 15) / 16 * 16; }

template <typename T, int I>
static void launch_tile(int shape, const TileArgs& g, dim3 grid, hipStream_t s) {
  if constexpr (I < kNumShapes) {
    if (shape == I)
      hipLaunchKernelGGL((tile_gemm_kernel<T, kShapes[I].mf, kShapes[I].nf, kShapes[I].stages>), grid,
                         dim3(kTileThreads), 0, s, g);
    else
      launch_tile<T, I + 1>(shape, g, grid, s);
  }
}

template <typename T>
static int wide(const void* x, int64_t ldx, int tokens, int K, const void* W, int N, const void* bias, void* out,
                int64_t ldo, void* ws, size_t ws_bytes, hipStream_t s) {
  const bool vec = ldo % 4 == 0 && (uintptr_t)out % 8 == 0;
  Route r = route(tokens, N, K, true);
  const int64_t ldp = split_ld(N);
  if (!r.rows16 && r.c.splits > 1 && (ws == nullptr || ws_bytes < (size_t)r.c.splits * tokens * ldp * sizeof(float)))
    r = route(tokens, N, K, false);
  if (r.rows16) return kTakeRows16;
  if (tokens <= kStripMaxTokens || K < 64) {
    StripArgs g{x, W, bias, out, ldx, ldo, tokens, K, N, (tokens + 31) / 32};
    const bool narrow = N < 32 * 128;
    // two column blocks per workgroup halve the x traffic; one where that
    // would leave half the CUs idle (1000 x 2048, 17 tokens: 5.2 vs 6.0 us;
    // 24576 x 4096: 48.3 vs 46.4)
    const int nf = narrow ? 1 : 2;
    const dim3 grid(g.m_tiles * (((N + 15) / 16 + nf - 1) / nf)), block(kStripThreads);
    if (narrow)
      hipLaunchKernelGGL((strip_gemm_kernel<T, 2, 1, 2>), grid, block, 0, s, g);
    else
      hipLaunchKernelGGL((strip_gemm_kernel<T, 2, 2, 2>), grid, block, 0, s, g);
    PL_LAUNCH_CHECK("strip_gemm_kernel");
    return PL_OK;
  }
  const Choice& c = r.c;
  const TileShape& sh = kShapes[c.shape];
  TileArgs g{};
  g.x = x;
  g.W = W;
  g.bias = c.splits > 1 ? nullptr : bias;
  g.out = out;
  g.partial = (float*)ws;
  g.ldx = ldx;
  g.ldo = ldo;
  g.ldp = ldp;
  g.tokens = tokens;
  g.K = K;
  g.N = N;
  g.m_tiles = (tokens + 16 * sh.mf - 1) / (16 * sh.mf);
  g.n_tiles = (N + 128 * sh.nf - 1) / (128 * sh.nf);
  g.splits = c.splits;
  g.vec_out = vec;
  launch_tile<T, 0>(c.shape, g, dim3((unsigned)(g.m_tiles * g.n_tiles * c.splits)), s);
  PL_LAUNCH_CHECK("tile_gemm_kernel");
  if (c.splits > 1) {
    const int64_t cells = (int64_t)tokens * ((N + 3) / 4);
    hipLaunchKernelGGL((split_sum_kernel<T>), dim3((unsigned)std::min<int64_t>((cells + 255) / 256, 2048)), dim3(256),
                       0, s, (const float*)ws, c.splits, ldp, tokens, N, (const T*)bias, (T*)out, ldo, (int)vec);
    PL_LAUNCH_CHECK("split_sum_kernel");
  }
  return PL_OK;
}

bool wide_supports(int64_t ldx) { return ldx < (int64_t)1 << 22; }

int wide_linear(const void* x, int64_t ldx, int tokens, int K, const void* W, int N, const void* bias, void* out,
                int64_t ldo, void* ws, size_t ws_bytes, int dtype, hipStream_t s) {
  return dtype == PL_DTYPE_BF16 ? wide<bf16_t>(x, ldx, tokens, K, W, N, bias, out, ldo, ws, ws_bytes, s)
                                : wide<f16_t>(x, ldx, tokens, K, W, N, bias, out, ldo, ws, ws_bytes, s);
}

}  // namespace wgemm
}  // namespace pl

using namespace pl;
using namespace pl::wgemm;

extern "C" size_t pl_linear_shuffled_wide_workspace_size(int num_tokens, int in_features, int out_features) {
  if (num_tokens <= kStripMaxTokens || in_features < 64 || out_features <= 0) return 0;
  const Route r = route(num_tokens, out_features, in_features, true);
  const Choice& c = r.c;
  return !r.rows16 && c.splits > 1 ? (size_t)c.splits * num_tokens * split_ld(out_features) * sizeof(float) : 0;
}

extern "C" int pl_linear_shuffled_wide_splits(int num_tokens, int in_features, int out_features,
                                              int32_t* step_begin_h) {
  if (num_tokens <= kStripMaxTokens || in_features < 64 || out_features <= 0) return 1;
  const Route r = route(num_tokens, out_features, in_features, true);
  const int splits = r.rows16 ? 1 : r.c.splits;
  for (int s = 0; s <= splits && step_begin_h != nullptr; ++s)
    step_begin_h[s] = split_begin(in_features / 64, splits, s);
  return splits;
}

extern "C" int pl_linear_shuffled_wide(const void* x, int64_t ldx, int num_tokens, int in_features,
                                       const void* shuffled, int out_features, const void* bias, void* out,
                                       int64_t ldo, void* workspace, size_t workspace_bytes, int dtype, void* stream) {
  if (num_tokens < 0) return fail(PL_ERR_INVALID, "num_tokens must be >= 0 (got %d)", num_tokens);
  if (num_tokens == 0) return ok();
  if (in_features <= 0 || in_features % 32 || out_features <= 0)
    return fail(PL_ERR_INVALID, "in_features must be a positive multiple of 32 and out_features > 0");
  if (!x || !shuffled || !out) return fail(PL_ERR_INVALID, "null pointer argument");
  if (ldx < in_features || ldx % 8 || (uintptr_t)x % 16 || (uintptr_t)shuffled % 16)
    return fail(PL_ERR_INVALID, "x rows and the shuffled weight must be 16-byte aligned");
  if (ldo < out_features) return fail(PL_ERR_INVALID, "ldo < out_features");
  if ((uintptr_t)workspace % 16) return fail(PL_ERR_INVALID, "workspace must be 16-byte aligned");
  if (dtype != PL_DTYPE_BF16 && dtype != PL_DTYPE_F16)
    return fail(PL_ERR_UNSUPPORTED, "pl_linear_shuffled_wide dtype must be F16 or BF16 (got %d)", dtype);
  // (rows too far apart for these kernels' offsets: the 16-token kernel)
  int st = kTakeRows16;
  if (wide_supports(ldx))
    st = wide_linear(x, ldx, num_tokens, in_features, shuffled, out_features, bias, out, ldo, workspace,
                     workspace_bytes, dtype, (hipStream_t)stream);
  if (st == kTakeRows16)
    st = linear_rows16(x, ldx, num_tokens, in_features, shuffled, out_features, bias, out, ldo, dtype,
                       (hipStream_t)stream);
  return st ? st : ok();
}
