// Paged prefill attention for head_dim 128 over page sizes of a multiple of 4
// (gfx950): the softmax of paged_prefill.hip with the kv range of an item
// split where the rows alone would leave the chip idle.
//
// A work item is 128 rows (query position, head of the GQA group) of one
// request over a range of 64-token kv tiles; the host plan cuts the ranges
// and lists the items longest first.  Grid = items x kv heads, heads fastest: workgroups go
// round the XCDs, so an XCD's L2 serves few heads, and the row items of one kv
// range run side by side.  Four waves of 32 rows each.
//
// K and V tiles go from the pages straight into LDS (asynchronous 16-byte
// loads, two buffers: the next tile's loads fly during a tile's work and cost
// no registers); rows are 256 bytes without padding, their 16-byte chunks
// permuted by the row so that the operand reads are free of bank conflicts.
// S^T = K Q^T keeps one query per lane as in paged_prefill.hip, two 16-query
// columns per wave sharing each K operand; V^T comes out of LDS transposed
// (ds_read_b64_tr_b16) and serves both columns.  An item of a split range
// leaves its unnormalized output and softmax state in the workspace, and
// merge_kernel combines a row's parts in order.
//
// Bound by the matrix and vector units' shared issue: 8192 tokens of 32768
// (GQA 4, bf16) 7770 us with 64-row items and 16 rows per wave -> 4600 us (4410
// a launch in a kernel trace), the MFMAs busy 58 % of the cycles (bf16's P is
// two planes, a third of them).  One wave's softmax beside its own
// neighbouring half tiles' MFMAs (software pipelining) was slower (5190 us):
// two waves per SIMD overlap already, and its registers spill.
#include <algorithm>
#include <type_traits>
#include <vector>

#include "pl_common.h"

namespace pl {
namespace prefill_split {

constexpr int kWave = 64;
constexpr int kWaves = 4;
constexpr int kThreads = kWave * kWaves;
constexpr int kCols = 2;                     // 16-query columns per wave
constexpr int kWaveRows = 16 * kCols;
constexpr int kRows = kWaveRows * kWaves;    // rows per item
constexpr int kTile = 64;                    // kv tokens per tile
constexpr int D = 128;
constexpr int kRowBytes = D * 2;
constexpr int kBufBytes = kTile * kRowBytes;
constexpr int kPartFloats = kRows * (D + 2);  // a part: outputs [row][dim], then (max, sum) per row

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// One work item, or (in the merge list) one row item split into parts.
struct Item {
  int32_t request, row0;
  int32_t tile_begin, tile_end;  // kv tiles
  int32_t slot;                  // first partial slot of the row item; -1: writes the output itself
  int32_t part, parts;
  int32_t pad;
};
static_assert(sizeof(Item) == 32, "the plan's record");

template <typename T> __device__ __forceinline__ f32x4 mfma32(u32x4 a, u32x4 b, f32x4 c);
template <> __device__ __forceinline__ f32x4 mfma32<bf16_t>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}
template <> __device__ __forceinline__ f32x4 mfma32<f16_t>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                0);
}

// Two probabilities (finite) packed with the hardware conversion.
template <typename T> __device__ __forceinline__ uint32_t pack_p(float a, float b);
template <> __device__ __forceinline__ uint32_t pack_p<bf16_t>(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2_t));
}
template <> __device__ __forceinline__ uint32_t pack_p<f16_t>(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, half2_t));
}

// The largest of the four lanes l, l ^ 16, l ^ 32, l ^ 48.
__device__ __forceinline__ float column_max(float v) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ void load_lds16(const char* g, char* l) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                   (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

__device__ __forceinline__ u32x2 read_tr(const char* p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)p));
}

struct Args {
  const char *q, *k, *v;
  char* o;
  float* part;
  const int32_t *qo_indptr, *kv_indptr, *kv_indices, *kv_last;
  const Item* items;
  int64_t q_st, q_sh, o_st, o_sh, page_stride, token_stride, head_stride, num_pages;  // elements
  int batch, hq, hkv, page_size, causal;
  float scale_log2;  // > 0; a negative scale negates q instead
  uint32_t q_flip;
};

template <typename T, bool PAGE16>
__global__ __launch_bounds__(kThreads, 2) void prefill_split_kernel(Args A) {
  constexpr int NPP = std::is_same<T, bf16_t>::value ? 2 : 1;  // P planes: hi (+ lo)
  // A column's running maximum follows only scores more than this above it,
  // which takes the rescale (64 multiplies and the lanes' exchange) out of
  // the steady state.  P's two planes hold probabilities up to 2^8 as well as
  // those up to 1; the one fp16 plane is exact for the largest only where
  // that is 1 (2.6e-4 against 2.5e-4 with a lag, from 64 bits).
  constexpr float kLag = NPP == 2 ? 8.f : 0.f;
  // one object per buffer: loads into one never alias reads of another
  __shared__ __align__(16) char s_k0[kBufBytes];
  __shared__ __align__(16) char s_v0[kBufBytes];
  __shared__ __align__(16) char s_k1[kBufBytes];
  __shared__ __align__(16) char s_v1[kBufBytes];
  const int h = blockIdx.x % A.hkv;
  const Item it = A.items[blockIdx.x / A.hkv];
  const int r = uniform(it.request), row0 = uniform(it.row0);
  if (r < 0 || r >= A.batch) return;
  const int g = A.hq / A.hkv;
  const int qo_begin = uniform(A.qo_indptr[r]);
  const int qo_len = uniform(A.qo_indptr[r + 1]) - qo_begin;
  const int pb = uniform(A.kv_indptr[r]), n_pages = uniform(A.kv_indptr[r + 1]) - pb;
  if (n_pages <= 0) return;
  const int last = min(max(uniform(A.kv_last[r]), 1), A.page_size);
  const int kv_len = (n_pages - 1) * A.page_size + last;
  const int n_rows = qo_len * g;
  const int32_t* ind = A.kv_indices + pb;

  const int lane = threadIdx.x % kWave, wave = uniform(threadIdx.x / kWave);
  const int lr = lane % 16, grp = lane / 16;

  // the wave's rows: their last visible kv positions lie in lim_lo .. lim_hi
  const int wrow = row0 + wave * kWaveRows;
  const int base = A.causal ? kv_len - qo_len : kv_len - 1;
  auto limit = [&](int row) { return min(A.causal ? base + row / g : base, kv_len - 1); };
  const bool wave_on = wrow < n_rows;
  const int lim_lo = wave_on ? limit(wrow) : -1;
  const int lim_hi = wave_on ? limit(min(wrow + kWaveRows, n_rows) - 1) : -1;
  int lim[kCols];
  u32x4 qb[kCols][4];
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    const int row = wrow + c * 16 + lr;
    const int rc = min(row, n_rows - 1);  // rows past the end repeat the last one; their results are not stored
    const int pos = rc / g;
    lim[c] = limit(rc);
    const char* qp = A.q + ((int64_t)(qo_begin + pos) * A.q_st + (int64_t)(h * g + rc - pos * g) * A.q_sh) * 2 + grp * 16;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      u32x4 v = *reinterpret_cast<const u32x4*>(qp + ks * 64);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] ^= A.q_flip;
      qb[c][ks] = v;
    }
  }

  // loads: wave w fetches tokens 16 w .. +16 of a tile, four per instruction;
  // lane l fetches token l / 16 of the four, chunk (l % 16) permuted by the row
  int64_t koff[4], voff[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int row = j * 4 + grp;
    const int64_t tok = (PAGE16 ? (int64_t)row : (int64_t)grp) * A.token_stride * 2 + (int64_t)h * A.head_stride * 2;
    koff[j] = tok + (lr ^ row) * 16;
    voff[j] = tok + (lr ^ (2 * (row % 8))) * 16;
  }
  auto clamp_page = [&](int page) -> int64_t {
    return page < 0 ? 0 : ((int64_t)page >= A.num_pages ? A.num_pages - 1 : (int64_t)page);
  };
  // PAGE16: page ids of 16 tiles (64 pages), one per lane
  int ids = 0, ids_next = 0;
  auto load_ids = [&](int tile) { return ind[min(tile / 16 * 64 + lane, n_pages - 1)]; };
  auto load_tile = [&](int tile, char* kd, char* vd) {
    kd += wave * 16 * kRowBytes;
    vd += wave * 16 * kRowBytes;
    if constexpr (PAGE16) {
      const int64_t off = clamp_page(__builtin_amdgcn_readlane(ids, (tile % 16) * 4 + wave)) * A.page_stride * 2;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        load_lds16(A.k + off + koff[j], kd + j * 4 * kRowBytes);
        load_lds16(A.v + off + voff[j], vd + j * 4 * kRowBytes);
      }
    } else {
      // page_size % 4 == 0: the four tokens of a load share a page
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = min(tile * kTile + wave * 16 + j * 4, (kv_len - 1) & ~3);
        const int64_t off = (clamp_page(uniform(ind[t / A.page_size])) * A.page_stride +
                             (int64_t)(t % A.page_size) * A.token_stride) * 2;
        load_lds16(A.k + off + koff[j], kd + j * 4 * kRowBytes);
        load_lds16(A.v + off + voff[j], vd + j * 4 * kRowBytes);
      }
    }
  };

  // operand reads: K row blk*16 + lr, chunk 4 ks + grp; V tokens 4 grp + lr/4
  // (+16 per half, +32 per kc), dims 16 a + 4 (lr % 4)
  int kaddr[4], vaddr[8];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) kaddr[ks] = lr * kRowBytes + ((ks * 4 + grp) ^ lr) * 16;
#pragma unroll
  for (int a = 0; a < 8; ++a) {
    const int row = grp * 4 + lr / 4;
    vaddr[a] = row * kRowBytes + (((2 * a + (lr % 4) / 2) ^ (2 * (row % 8))) * 16) + (lr % 2) * 8;
  }

  f32x4 acc[kCols][8];
  float m[kCols], l[kCols];
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    m[c] = -INFINITY;
    l[c] = 0.f;
#pragma unroll
    for (int a = 0; a < 8; ++a) acc[c][a] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float sc = A.scale_log2;

  auto body = [&](int tile, int end, const char* kb, char* vb, char* kn, char* vn) {
    // this wave's loads of the tile are done, and past the barrier everyone's
    // are, and every wave is done with the other buffers
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xF70);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (tile + 1 < end) {
      const bool turn = PAGE16 && (tile + 1) % 16 == 0;
      if (turn) ids = ids_next;
      load_tile(tile + 1, kn, vn);
      if (turn) ids_next = load_ids(tile + 17);
    }
    if ((tile + 1) * kTile > kv_len) {
      // past the last token the pages hold anything: zero V there (0 * NaN)
      for (int c = threadIdx.x; c < kTile * 16; c += kThreads)
        if (tile * kTile + c / 16 >= kv_len) *reinterpret_cast<u32x4*>(vb + c * 16) = u32x4{0u, 0u, 0u, 0u};
      __syncthreads();
    }
    if (tile * kTile > lim_hi) return;  // (uniform) no row of the wave sees the tile

    f32x4 s[kCols][4];
    // four independent accumulations in turn, here and below: an MFMA waits
    // for the one before it on the same accumulator
#pragma unroll
    for (int b0 = 0; b0 < 4; b0 += 2) {
#pragma unroll
      for (int c = 0; c < kCols; ++c)
#pragma unroll
        for (int b = 0; b < 2; ++b) s[c][b0 + b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        u32x4 ka[2];
#pragma unroll
        for (int b = 0; b < 2; ++b)
          ka[b] = *reinterpret_cast<const u32x4*>(kb + kaddr[ks] + (b0 + b) * 16 * kRowBytes);
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int c = 0; c < kCols; ++c) s[c][b0 + b] = mfma32<T>(ka[b], qb[c][ks], s[c][b0 + b]);
      }
    }
    if (tile * kTile + kTile - 1 > lim_lo) {
      const int t0 = tile * kTile + 4 * grp;
#pragma unroll
      for (int c = 0; c < kCols; ++c)
#pragma unroll
        for (int blk = 0; blk < 4; ++blk)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[c][blk][i] = t0 + blk * 16 + i <= lim[c] ? s[c][blk][i] : -INFINITY;
    }
    float mx[kCols];
    bool rose = false;
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      float v = -INFINITY;
#pragma unroll
      for (int blk = 0; blk < 4; ++blk)
#pragma unroll
        for (int i = 0; i < 4; ++i) v = fmaxf(v, s[c][blk][i]);
      mx[c] = v * sc;
      rose |= mx[c] > m[c] + kLag;
    }
    // the columns' maxima are reduced over their lanes, and the sums and
    // accumulators rescaled, only where some lane saw a score kLag past its
    // maximum
    if (__builtin_amdgcn_ballot_w64(rose) != 0) {
#pragma unroll
      for (int c = 0; c < kCols; ++c) {
        const float mn = fmaxf(m[c], column_max(mx[c]));
        const float alpha = fast_exp2(m[c] - (mn == -INFINITY ? 0.f : mn));
        m[c] = mn;
        l[c] *= alpha;
#pragma unroll
        for (int a = 0; a < 8; ++a)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[c][a][i] *= alpha;
      }
    }
    u32x4 pb[kCols][2][NPP];
#pragma unroll
    for (int c = 0; c < kCols; ++c) {
      const float mu = m[c] == -INFINITY ? 0.f : m[c];
      float ps = 0.f;
#pragma unroll
      for (int blk = 0; blk < 4; ++blk)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = fast_exp2(__builtin_fmaf(s[c][blk][i], sc, -mu));
          s[c][blk][i] = e;
          ps += e;
        }
      l[c] += ps;  // per lane; the column's lanes meet after the last tile
      // P^T as the B operand: k = 8*grp + e <-> tokens of blocks 2kc (e < 4) and 2kc+1 (e >= 4)
#pragma unroll
      for (int kc = 0; kc < 2; ++kc)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4 src = s[c][2 * kc + e / 2];
          const float p0 = src[(e % 2) * 2], p1 = src[(e % 2) * 2 + 1];
          const uint32_t hw = pack_p<T>(p0, p1);
          pb[c][kc][0][e] = hw;
          if constexpr (NPP == 2) {
            float h0, h1;
            unpack2<T>(hw, h0, h1);
            pb[c][kc][NPP - 1][e] = pack_p<T>(p0 - h0, p1 - h1);
          }
        }
    }
#pragma unroll
    for (int kc = 0; kc < 2; ++kc)
#pragma unroll
      for (int a0 = 0; a0 < 8; a0 += 2) {
        u32x4 va[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          const u32x2 v0 = read_tr(vb + vaddr[a0 + a] + kc * 32 * kRowBytes);
          const u32x2 v1 = read_tr(vb + vaddr[a0 + a] + (kc * 32 + 16) * kRowBytes);
          va[a] = u32x4{v0[0], v0[1], v1[0], v1[1]};
        }
#pragma unroll
        for (int pl = 0; pl < NPP; ++pl)
#pragma unroll
          for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int c = 0; c < kCols; ++c) acc[c][a0 + a] = mfma32<T>(va[a], pb[c][kc][pl], acc[c][a0 + a]);
      }
  };

  const int t_begin = uniform(it.tile_begin), t_end = uniform(it.tile_end);
  if (t_begin < t_end) {
    if (PAGE16) {
      ids = load_ids(t_begin);
      ids_next = load_ids(t_begin + 16);
    }
    load_tile(t_begin, s_k0, s_v0);
  }
  int tile = t_begin;
  for (; tile + 2 <= t_end; tile += 2) {
    body(tile, t_end, s_k0, s_v0, s_k1, s_v1);
    body(tile + 1, t_end, s_k1, s_v1, s_k0, s_v0);
  }
  if (tile < t_end) body(tile, t_end, s_k0, s_v0, s_k1, s_v1);

  const int slot = uniform(it.slot);
#pragma unroll
  for (int c = 0; c < kCols; ++c) {
    float sum = l[c];
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    const int row = wrow + c * 16 + lr;
    if (row >= n_rows) continue;
    if (slot >= 0) {
      float* p = A.part + ((int64_t)(slot + it.part) * A.hkv + h) * kPartFloats;
      const int pr = wave * kWaveRows + c * 16 + lr;
#pragma unroll
      for (int a = 0; a < 8; ++a) *reinterpret_cast<f32x4*>(p + pr * D + a * 16 + grp * 4) = acc[c][a];
      if (grp == 0) *reinterpret_cast<f32x2*>(p + kRows * D + pr * 2) = f32x2{m[c], sum};
      continue;
    }
    const float inv = sum > 0.f ? 1.f / sum : (sum == 0.f ? 0.f : sum);
    const int pos = row / g;
    T* op = (T*)A.o + (int64_t)(qo_begin + pos) * A.o_st + (int64_t)(h * g + row - pos * g) * A.o_sh + grp * 4;
#pragma unroll
    for (int a = 0; a < 8; ++a)
      *reinterpret_cast<u32x2*>(op + a * 16) = u32x2{pack2<T>(acc[c][a][0] * inv, acc[c][a][1] * inv),
                                                     pack2<T>(acc[c][a][2] * inv, acc[c][a][3] * inv)};
  }
}

// One wave per row of a split row item, two dims per lane: parts in order.
template <typename T>
__global__ __launch_bounds__(kThreads) void merge_kernel(Args A, const Item* merges) {
  const int h = blockIdx.x % A.hkv;
  const Item it = merges[blockIdx.x / A.hkv];
  const int r = uniform(it.request);
  if (r < 0 || r >= A.batch) return;
  const int g = A.hq / A.hkv;
  const int qo_begin = uniform(A.qo_indptr[r]);
  const int n_rows = (uniform(A.qo_indptr[r + 1]) - qo_begin) * g;
  const int pr = blockIdx.y * kWaves + uniform(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int row = uniform(it.row0) + pr;
  if (row >= n_rows) return;
  const int parts = uniform(it.parts);
  const float* p = A.part + ((int64_t)uniform(it.slot) * A.hkv + h) * kPartFloats;
  const int64_t step = (int64_t)A.hkv * kPartFloats;
  // the parts' states one per lane, their outputs eight loads at a time
  const float* ml = p + kRows * D + pr * 2;
  float top = -INFINITY;
  for (int b = lane; b < parts; b += kWave) top = fmaxf(top, ml[b * step]);
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) top = fmaxf(top, __shfl_xor(top, d));
  if (top == -INFINITY) top = 0.f;
  float sum = 0.f, o0 = 0.f, o1 = 0.f;
  for (int b0 = 0; b0 < parts; b0 += kWave) {
    const int n = min(parts - b0, kWave);
    const f32x2 own = lane < n ? *reinterpret_cast<const f32x2*>(ml + (b0 + lane) * step) : f32x2{-INFINITY, 0.f};
    const float w = fast_exp2(own[0] - top);
    const float lw = own[1] * w;
    const float* q = p + b0 * step + pr * D + lane * 2;
    for (int i0 = 0; i0 < n; i0 += 8) {
      f32x2 v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const f32x2*>(q + min(i0 + i, n - 1) * step);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (i0 + i >= n) break;
        const float wi = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), i0 + i));
        sum += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(lw), i0 + i));
        o0 = fmaf(v[i][0], wi, o0);
        o1 = fmaf(v[i][1], wi, o1);
      }
    }
  }
  const float inv = sum > 0.f ? 1.f / sum : (sum == 0.f ? 0.f : sum);
  const int pos = row / g;
  T* op = (T*)A.o + (int64_t)(qo_begin + pos) * A.o_st + (int64_t)(h * g + row - pos * g) * A.o_sh + lane * 2;
  *reinterpret_cast<uint32_t*>(op) = pack2<T>(o0 * inv, o1 * inv);
}

// ------------------------------------------------------------ host plan ---
constexpr int kSlots = 512;     // workgroups the chip holds: two per CU
constexpr int kMinTiles = 4;    // fewest tiles of a part

template <typename T>
int launch(const Args& a, int num_items, int num_merges, hipStream_t s) {
  const dim3 grid((unsigned)a.hkv * num_items);
  if (a.page_size == 16)
    hipLaunchKernelGGL((prefill_split_kernel<T, true>), grid, dim3(kThreads), 0, s, a);
  else
    hipLaunchKernelGGL((prefill_split_kernel<T, false>), grid, dim3(kThreads), 0, s, a);
  PL_LAUNCH_CHECK("prefill_split_kernel");
  if (num_merges > 0) {
    hipLaunchKernelGGL(merge_kernel<T>, dim3((unsigned)a.hkv * num_merges, kRows / kWaves), dim3(kThreads), 0, s, a,
                       a.items + num_items);
    PL_LAUNCH_CHECK("prefill merge_kernel");
  }
  return ok();
}

}  // namespace prefill_split
}  // namespace pl

using namespace pl;
using namespace pl::prefill_split;

extern "C" int pl_prefill_split_plan(const int32_t* qo_indptr_h, const int32_t* kv_indptr_h,
                                     const int32_t* kv_last_page_len_h, int batch, int num_qo_heads, int num_kv_heads,
                                     int page_size, int causal, int32_t* items_h, int max_records, int* num_items_h,
                                     int* num_merges_h, size_t* workspace_bytes_h) {
  if (!num_items_h || !num_merges_h || !workspace_bytes_h)
    return fail(PL_ERR_INVALID, "num_items_h, num_merges_h and workspace_bytes_h must not be null");
  *num_items_h = *num_merges_h = 0;
  *workspace_bytes_h = 0;
  if (batch < 0) return fail(PL_ERR_INVALID, "batch must be >= 0");
  if (batch > 0 && (!qo_indptr_h || !kv_indptr_h || !kv_last_page_len_h))
    return fail(PL_ERR_INVALID, "null table pointer");
  if (num_kv_heads <= 0 || num_qo_heads <= 0 || num_qo_heads % num_kv_heads)
    return fail(PL_ERR_INVALID, "num_qo_heads (%d) must be a multiple of num_kv_heads (%d)", num_qo_heads,
                num_kv_heads);
  if (page_size <= 0 || page_size % 4)
    return fail(PL_ERR_INVALID, "page_size must be a positive multiple of 4 (got %d)", page_size);
  const int g = num_qo_heads / num_kv_heads;
  if (batch > 0 && (qo_indptr_h[0] != 0 || kv_indptr_h[0] != 0))
    return fail(PL_ERR_INVALID, "qo_indptr_h[0] and kv_indptr_h[0] must be 0");
  struct Rows {
    int32_t r, row0, tiles;
  };
  std::vector<Rows> list;
  int64_t work = 0;
  int longest = 0;
  for (int r = 0; r < batch; ++r) {
    const int qo_len = qo_indptr_h[r + 1] - qo_indptr_h[r];
    const int pages = kv_indptr_h[r + 1] - kv_indptr_h[r];
    if (qo_len < 0) return fail(PL_ERR_INVALID, "qo_indptr_h must be non-decreasing (row %d)", r);
    if (pages < 0) return fail(PL_ERR_INVALID, "kv_indptr_h must be non-decreasing (row %d)", r);
    const int last = kv_last_page_len_h[r];
    if (pages > 0 && (last < 1 || last > page_size))
      return fail(PL_ERR_INVALID, "last_page_len[%d] = %d outside [1, %d]", r, last, page_size);
    const int64_t kv_len = pages > 0 ? (int64_t)(pages - 1) * page_size + last : 0;
    if (kv_len > INT32_MAX / 2) return fail(PL_ERR_INVALID, "row %d: kv_len %lld too large", r, (long long)kv_len);
    if (causal && qo_len > kv_len)
      return fail(PL_ERR_INVALID, "row %d: qo_len %d exceeds kv_len %lld under the causal mask", r, qo_len,
                  (long long)kv_len);
    if (qo_len > 0 && kv_len == 0) return fail(PL_ERR_INVALID, "row %d has queries but no kv", r);
    const int64_t rows = (int64_t)qo_len * g;
    if (rows > INT32_MAX / 2) return fail(PL_ERR_INVALID, "row %d: %lld query rows too many", r, (long long)rows);
    for (int64_t r0 = 0; r0 < rows; r0 += kRows) {
      const int64_t last_row = std::min<int64_t>(r0 + kRows, rows) - 1;
      const int64_t max_pos = causal ? kv_len - qo_len + last_row / g : kv_len - 1;
      const int tiles = (int)(max_pos / kTile) + 1;
      list.push_back(Rows{r, (int32_t)r0, tiles});
      work += tiles;
      longest = std::max(longest, tiles);
    }
  }
  if (list.size() > (size_t)INT32_MAX / 64) return fail(PL_ERR_INVALID, "too many prefill work items");
  // A part's length: an even share of the work per slot.  Ranges are cut where
  // the longest row item is more than twice that, and by four tiles more, which
  // the partial results and the merge cost: 2119 tokens MHA (34 tiles, share
  // 20) 56.5 us whole, 68 cut; 3 x 300 behind 300 GQA 4 (10, 4) 23.2 whole, 42.6
  // cut; 3 x 300 behind 1500 (29, 13) 51.3 whole, 71.0 cut; 500 behind 800 (21,
  // 5) 39.5 whole, 33.6 cut; 77 behind 32000 (501, 16) 700 whole, 77 cut.  Over
  // 624 calls of 1 to 3 requests of 2 to 2200 tokens behind 0 to 30000 the
  // choice is 5 % from the better of the two in the mean, without the four
  // tiles 6.3 %, with eight 6.9.
  const int64_t share = std::max<int64_t>(kMinTiles, (work * num_kv_heads + kSlots - 1) / kSlots);
  const int64_t chunk = longest > 2 * share + 4 ? share : INT32_MAX;
  std::vector<Item> items, merges;
  int slots = 0;
  for (const Rows& e : list) {
    const int parts = (int)((e.tiles + chunk - 1) / chunk);
    for (int p = 0; p < parts; ++p)
      items.push_back(Item{e.r, e.row0, (int32_t)((int64_t)e.tiles * p / parts),
                           (int32_t)((int64_t)e.tiles * (p + 1) / parts), parts > 1 ? slots : -1, p, parts, 0});
    if (parts > 1) {
      merges.push_back(Item{e.r, e.row0, 0, 0, slots, 0, parts, 0});
      slots += parts;
    }
  }
  // longest first; items of one length by request and kv range, so that the
  // row items sharing a range run side by side
  std::stable_sort(items.begin(), items.end(), [](const Item& a, const Item& b) {
    const int la = a.tile_end - a.tile_begin, lb = b.tile_end - b.tile_begin;
    if (la != lb) return la > lb;
    if (a.request != b.request) return a.request < b.request;
    return a.tile_begin < b.tile_begin;
  });
  *num_items_h = (int)items.size();
  *num_merges_h = (int)merges.size();
  *workspace_bytes_h = (size_t)slots * num_kv_heads * kPartFloats * sizeof(float);
  if (items_h == nullptr) return ok();
  if (items.size() + merges.size() > (size_t)max_records)
    return fail(PL_ERR_WORKSPACE, "%zu prefill plan records exceed the %d provided", items.size() + merges.size(),
                max_records);
  std::copy(items.begin(), items.end(), reinterpret_cast<Item*>(items_h));
  std::copy(merges.begin(), merges.end(), reinterpret_cast<Item*>(items_h) + items.size());
  return ok();
}

extern "C" int pl_prefill_split_run(const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k_cache,
                                    const void* v_cache, int64_t page_stride, int64_t token_stride,
                                    int64_t head_stride, int64_t num_pages, const int32_t* qo_indptr,
                                    const int32_t* kv_indptr, const int32_t* kv_indices,
                                    const int32_t* kv_last_page_len, const int32_t* items, int num_items,
                                    int num_merges, void* o, int64_t o_stride_t, int64_t o_stride_h, int batch,
                                    int num_qo_heads, int num_kv_heads, int page_size, int causal, float sm_scale,
                                    void* workspace, size_t workspace_bytes, size_t plan_workspace_bytes, int dtype,
                                    void* stream) {
  if (num_items < 0 || num_merges < 0 || batch < 0)
    return fail(PL_ERR_INVALID, "num_items, num_merges and batch must be >= 0");
  if (num_items == 0 || batch == 0) return ok();
  if (num_kv_heads <= 0 || num_qo_heads <= 0 || num_qo_heads % num_kv_heads)
    return fail(PL_ERR_INVALID, "num_qo_heads (%d) must be a multiple of num_kv_heads (%d)", num_qo_heads,
                num_kv_heads);
  if (page_size <= 0 || page_size % 4 || num_pages <= 0)
    return fail(PL_ERR_INVALID, "page_size must be a positive multiple of 4 and num_pages > 0");
  if (!q || !k_cache || !v_cache || !qo_indptr || !kv_indptr || !kv_indices || !kv_last_page_len || !items || !o)
    return fail(PL_ERR_INVALID, "null pointer argument");
  const int64_t strides[] = {q_stride_t, q_stride_h, o_stride_t, o_stride_h, page_stride, token_stride, head_stride};
  for (int64_t st : strides)
    if (st % 8) return fail(PL_ERR_INVALID, "strides must be multiples of 8 elements");
  const void* ptrs[] = {q, k_cache, v_cache, o, items, workspace};
  for (const void* p : ptrs)
    if ((uintptr_t)p % 16) return fail(PL_ERR_INVALID, "q, o, the caches, items and workspace must be 16-byte aligned");
  if ((int64_t)num_items * num_kv_heads > INT32_MAX)
    return fail(PL_ERR_INVALID, "grid of %d items x %d heads too large", num_items, num_kv_heads);
  if (num_merges > 0 && (!workspace || workspace_bytes < plan_workspace_bytes))
    return fail(PL_ERR_WORKSPACE, "prefill workspace of %zu bytes < %zu needed", workspace_bytes,
                plan_workspace_bytes);
  if (dtype != PL_DTYPE_BF16 && dtype != PL_DTYPE_F16)
    return fail(PL_ERR_UNSUPPORTED, "prefill dtype must be F16 or BF16 (got %d)", dtype);
  Args a{};
  a.q = (const char*)q;
  a.k = (const char*)k_cache;
  a.v = (const char*)v_cache;
  a.o = (char*)o;
  a.part = (float*)workspace;
  a.qo_indptr = qo_indptr;
  a.kv_indptr = kv_indptr;
  a.kv_indices = kv_indices;
  a.kv_last = kv_last_page_len;
  a.items = reinterpret_cast<const Item*>(items);
  a.q_st = q_stride_t;
  a.q_sh = q_stride_h;
  a.o_st = o_stride_t;
  a.o_sh = o_stride_h;
  a.page_stride = page_stride;
  a.token_stride = token_stride;
  a.head_stride = head_stride;
  a.num_pages = num_pages;
  a.batch = batch;
  a.hq = num_qo_heads;
  a.hkv = num_kv_heads;
  a.page_size = page_size;
  a.causal = causal;
  // the kernel takes maxima before scaling: a positive scale (a zero one as
  // one far below any score's rounding), the sign moved into q
  const float s2 = sm_scale * 1.44269504088896340736f;
  a.scale_log2 = std::max(s2 < 0 ? -s2 : s2, 1e-30f);
  a.q_flip = s2 < 0 ? 0x80008000u : 0u;
  return dtype == PL_DTYPE_BF16 ? launch<bf16_t>(a, num_items, num_merges, (hipStream_t)stream)
                                : launch<f16_t>(a, num_items, num_merges, (hipStream_t)stream);
}
