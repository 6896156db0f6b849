// MoE-layer LATENT expert FFN over the row layout in fp32 on matrix cores.
//
// For 32 to 512 routed pairs: the pairs are grouped into units of at most four
// pairs of one expert, and four launches follow,
//   A   x . A_g | A_u            items (unit, factor, range of d)
//   BC  g . B_g, u . B_u -> h = SiLU(g) u (LDS); h . A_d
//                                items (unit, 256 columns of ff)
//   D   d_lat . B_d -> y rows    items (unit, 512 columns of d)
//   combine                      weighted slot sum, or per-slot copy
// Every sum is fp32 and runs in a fixed order (K ranges of a wave, waves of a
// workgroup, workgroups), so calls are bit-reproducible.  Replaces, like
// moe.hip, the per-(token, slot) chain of
// kernels/latent_fused_expert_ffn.cu:27-108.
//
// The factors go from HBM to the matrix cores in rowblock.hpp's blocks.  Each
// value meets the activations of its row in v_mfma_f32_4x4x1_16b_f32: sixteen
// 4 x 4 products a step, every lane's own value against four pairs, 8 cycles
// for 64 values.  The four lanes of such a product share their 32-column
// group, so the group's scale multiplies the activation (one product a row,
// exact for 16-bit x) and a value is a level from a byte table in LDS, never
// scaled.  The waves of a workgroup share K, not columns, where N is a rank.
//
// Units of four: a 16-pair unit on v_mfma_f32_16x16x4_f32 pays 32 cycles for
// 64 values however few its pairs (a decode batch has one to four), and no
// fewer cycles a pair when full.  An expert's further units find its factors
// in L2.
//
// What bounds it: the MFMA issue (512 cycles a block of 32 x 128 values, of
// which the decode's VALU covers 450), and below some 200 pairs the latency
// of the five launches (about 5 us each).
#include "chain32.hpp"
#include "rowblock.hpp"

#include <algorithm>
#include <cmath>

namespace latent {
namespace chain32 {
namespace {

using namespace rowblock;

enum { F_GATE_A = 0, F_GATE_B, F_UP_A, F_UP_B, F_DOWN_A, F_DOWN_B };

constexpr int kT = 512;       // threads per workgroup
constexpr int kW = kT / kWave;
constexpr int kM = kUnitPairs;
constexpr int kCB = 256;      // BC: ff columns per item
constexpr int kCD = 512;      // D: d columns per item
constexpr int kHStr = kCB + 4;
constexpr int kCopies = 16;   // of the level table, by lane
constexpr int kLutBytes = 256 * kCopies * 8;
constexpr int kTileStr = 128 + 4;  // floats per row of a wave's products in LDS
constexpr int kRedBytes = kW * kM * kTileStr * 4;  // products of every wave

struct Params {
  Factor fac[6];
  const void* x;
  const int32_t* ids;
  const void* weights;
  const int32_t* ranks;
  Grouping g;
  float* part_a;  // [n_a][2][P][R]
  float* part_c;  // [n_c][P][R]
  float* y;       // [P][d]
  float* out;
  int x_dtype, w_dtype, T, d, ff, E, K, R, P, wbd, out_mode;
  int a_rows, n_a, n_c, n_d;
};

__device__ __forceinline__ int rank_of(const Params& p, int e, int kind) {
  if (!p.ranks) return p.R;
  const int r = p.ranks[e * 3 + kind];
  return r < 0 ? 0 : (r > p.R ? p.R : r);
}

// Level table: entry b = (level(b & 15), level(b >> 4)), kCopies copies of
// each entry side by side so that a wave's random lookups spread over the banks.
__device__ __forceinline__ void lut_fill(uint32_t lut, int tid) {
  const int b = tid >> 1;
  const float lo = nf4_level(b & 15), hi = nf4_level(b >> 4);
  const u32x4 two = {__float_as_uint(lo), __float_as_uint(hi), __float_as_uint(lo), __float_as_uint(hi)};
#pragma unroll
  for (int i = 0; i < kCopies / 4; ++i)
    lds_st<u32x4>(lut + b * (kCopies * 8) + ((tid & 1) * (kCopies / 4) + i) * 16, two);
}

// Products of a unit's four pairs with 16 CPL columns.  While summing, a lane
// holds all four pairs of its columns over its own rows (kq apart); finish()
// adds the four row sets, pair kq to the lanes of kq.
template <int CPL>
struct Acc {
  float4v a[CPL];
  float r[CPL];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int c = 0; c < CPL; ++c) a[c] = float4v{0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ void finish() {
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const float4v v = a[c];
      const auto lo = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[0]), __float_as_uint(v[2]), false, false);
      const auto hi = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[1]), __float_as_uint(v[3]), false, false);
      const float s0 = __uint_as_float(lo[0]) + __uint_as_float(lo[1]);
      const float s1 = __uint_as_float(hi[0]) + __uint_as_float(hi[1]);
      const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(s0), __float_as_uint(s1), false, false);
      r[c] = __uint_as_float(q[0]) + __uint_as_float(q[1]);
    }
  }
};

// acc += act . block.  act[i]: the activation of row 8 kq + i and the lane's
// pair; refill(h) reloads rows 2 h, 2 h + 1 once they are used.  A block's
// products are summed apart before they join acc: a chain of n terms rounds as
// sqrt(n), and one chain over a wave's rows more than doubled the result's error.
template <int CPL, bool kInt8, typename Refill>
__device__ __forceinline__ void block_mfma(const Block<CPL>& b, const float (&act)[8], uint32_t lut, const Factor& f,
                                           int e, int row, int col, Acc<CPL>& acc, Refill&& refill) {
  Acc<CPL> part;
  part.clear();
#pragma unroll
  for (int h = 0; h < 4; ++h) {
#pragma unroll
    for (int i = 2 * h; i < 2 * h + 2; ++i) {
      const float a = act[i] * half_bits_to_float(b.s[i >> 1][i & 1]);
      float v[CPL];
#pragma unroll
      for (int j = 0; j < CPL / 2; ++j) {
        const uint32_t byte = (b.c[i] >> (8 * j)) & 0xFFu;
        const float2v lv = lds_ld<float2v>(lut + byte * (kCopies * 8));
        v[2 * j] = lv[0];
        v[2 * j + 1] = lv[1];
      }
      if (kInt8 && f.ext.bitmap) {
        uint32_t q[(CPL + 3) / 4];
        if (int8_row<CPL>(f, e, row + i, col, q)) {
#pragma unroll
          for (int c = 0; c < CPL; ++c)
            v[c] = static_cast<float>(static_cast<int8_t>((q[c >> 2] >> (8 * (c & 3))) & 0xFFu));
        }
      }
#pragma unroll
      for (int c = 0; c < CPL; ++c) part.a[c] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, v[c], part.a[c], 0, 0, 0);
    }
    refill(h);
  }
#pragma unroll
  for (int c = 0; c < CPL; ++c) acc.a[c] += part.a[c];
}

// A wave's walk over blocks [b0, b1) of 32 rows from `row0` of the factor: one
// block of codes in registers, its rows reloaded from the next block as they
// are used (with four waves per SIMD a block's time covers the loads; a
// second block in registers spilled).  start() issues the first loads (as
// early as the caller can), run() does the rest.  act.load(b, raw) and
// act.get(b, raw, a) give the lane's activations of block b.
template <int CPL, bool kInt8, class Act>
struct Walk {
  const Factor& f;
  int e, row0, b0, b1, col, kq8;
  Src<CPL> src;
  Act act;
  Block<CPL> k;
  typename Act::Raw r;
  __device__ __forceinline__ Walk(const Factor& f_, int e_, int col0, int row0_, int b0_, int b1_, int lane,
                                  const Act& act_)
      : f(f_), e(e_), row0(row0_), b0(b0_), b1(b1_),
        col(min(col0 + CPL * (lane & 15), static_cast<int>(f_.cols) - CPL)), kq8(8 * (lane >> 4)),
        src(make_src<CPL>(f_, e_, col0, lane)), act(act_) {}
  __device__ __forceinline__ int clamped(int b) const { return max(0, min(b, b1 - 1)); }  // the same loads on every path
  __device__ __forceinline__ void start() {
    const int b = clamped(b0);
    act.load(b, r);
#pragma unroll
    for (int h = 0; h < 4; ++h) load_rows<CPL>(src, row0 + 32 * b, h, k);
  }
  __device__ __forceinline__ void run(uint32_t lut, Acc<CPL>& acc) {
    acc.clear();
    for (int b = b0; b < b1; ++b) {
      const int next = clamped(b + 1);
      float a[8];
      act.get(b, r, a);
      act.load(next, r);
      block_mfma<CPL, kInt8>(k, a, lut, f, e, row0 + 32 * b + kq8, col, acc,
                                [&](int h) __attribute__((always_inline)) { load_rows<CPL>(src, row0 + 32 * next, h, k); });
    }
    acc.finish();
  }
};

// Activations from x rows in HBM (any dtype), row `row0` of the factor at
// column row0 of x.  Lane n feeds pair n & 3.
template <bool kF32>
struct ActX {
  struct Raw {
    u32x4 v[kF32 ? 2 : 1];
  };
  const char* src;  // the lane's x row at column row0 + 8 kq
  bool bf16;
  __device__ __forceinline__ void load(int b, Raw& r) const {
#pragma unroll
    for (int q = 0; q < (kF32 ? 2 : 1); ++q)
      r.v[q] = *reinterpret_cast<const u32x4*>(src + static_cast<int64_t>(b) * 32 * (kF32 ? 4 : 2) + 16 * q);
  }
  __device__ __forceinline__ void get(int, const Raw& r, float (&a)[8]) const {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (kF32) {
        a[i] = __uint_as_float(r.v[(i >> 2) & (kF32 ? 1 : 0)][i & 3]);
      } else {
        const uint32_t h = (r.v[0][i >> 1] >> (16 * (i & 1))) & 0xFFFFu;
        a[i] = bf16 ? __uint_as_float(h << 16) : half_bits_to_float(static_cast<uint16_t>(h));
      }
    }
  }
};
// Activations from fp32 rows in LDS: at = the lane's row, column 8 kq.
struct ActLds {
  struct Raw {};
  uint32_t at;
  __device__ __forceinline__ void load(int, Raw&) const {}
  __device__ __forceinline__ void get(int b, const Raw&, float (&a)[8]) const {
    const float4v lo = lds_ld<float4v>(at + b * 128), hi = lds_ld<float4v>(at + b * 128 + 16);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a[i] = lo[i];
      a[4 + i] = hi[i];
    }
  }
};

// f(columns per lane, column tiles) for N columns: a tile of 64 columns that
// all waves share by K, or tiles of 128 columns (the waves of a tile share its K).
template <typename F>
__device__ __forceinline__ void with_columns(int n, F&& f) {
  using std::integral_constant;
  if (n <= 64)
    f(integral_constant<int, 4>{}, integral_constant<int, 1>{});
  else if (n <= 128)
    f(integral_constant<int, 8>{}, integral_constant<int, 1>{});
  else if (n <= 256)
    f(integral_constant<int, 8>{}, integral_constant<int, 2>{});
  else
    f(integral_constant<int, 8>{}, integral_constant<int, 4>{});
}

// A lane's results (pair kq) in LDS at `at`, CPL floats.
template <int CPL>
__device__ __forceinline__ void store_tile(uint32_t at, const Acc<CPL>& acc) {
#pragma unroll
  for (int c = 0; c < CPL; c += 4)
    lds_st<float4v>(at + 4u * c, float4v{acc.r[c], acc.r[c + 1], acc.r[c + 2], acc.r[c + 3]});
}
template <int CPL>
__device__ __forceinline__ void add_tile(uint32_t at, Acc<CPL>& acc) {
#pragma unroll
  for (int c = 0; c < CPL; c += 4) {
    const float4v t = lds_ld<float4v>(at + 4u * c);
#pragma unroll
    for (int q = 0; q < 4; ++q) acc.r[c + q] += t[q];
  }
}

// Products of 32 nblk rows (from row0 of the factor) with `cols` columns of
// one unit, summed over the waves in a fixed order: dst[row][0 .. cols) for the
// unit's m pairs, rows `stride` floats apart.  ready(): the level table and
// the activations are in LDS (the first factor loads are issued before it).
// red: LDS byte address of kRedBytes the table and the activations may overlap.
template <bool kInt8, class Act, typename Ready>
__device__ __forceinline__ void rank_gemm(const Factor& f, int e, int row0, int nblk, int cols, int m, uint32_t lut,
                                          uint32_t red, const Act& act, Ready&& ready, float* dst, int stride) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid >> 6);
  const int n = lane & 15, kq = lane >> 4;
  with_columns(cols, [&](auto cpl, auto nt) __attribute__((always_inline)) {
    constexpr int CPL = decltype(cpl)::value, NT = decltype(nt)::value, KP = kW / NT;
    const int tile = wave % NT, kp = wave / NT;
    Walk<CPL, kInt8, Act> walk(f, e, tile * 16 * CPL, row0, kp * nblk / KP, (kp + 1) * nblk / KP, lane, act);
    walk.start();
    ready();
    Acc<CPL> acc;
    walk.run(lut, acc);
    lds_barrier();  // every wave is done with the table and the activations
    store_tile(red + static_cast<uint32_t>((wave * kM + kq) * kTileStr + n * CPL) * 4u, acc);
    lds_barrier();
    const int c4 = cols / 4;
    for (int i = tid; i < m * c4; i += kT) {
      const int r = i / c4, c = (i - r * c4) * 4;
      const int t = c / (16 * CPL);  // wave t + NT k holds the columns' k-th share of K
      const uint32_t at = red + static_cast<uint32_t>((t * kM + r) * kTileStr + c - t * 16 * CPL) * 4u;
      float4v s[KP];
#pragma unroll
      for (int k = 0; k < KP; ++k) s[k] = lds_ld<float4v>(at + static_cast<uint32_t>(k * NT * kM * kTileStr) * 4u);
#pragma unroll
      for (int w = KP / 2; w > 0; w /= 2)
#pragma unroll
        for (int k = 0; k < w; ++k) s[k] += s[k + w];
      *reinterpret_cast<float4v*>(dst + static_cast<int64_t>(r) * stride + c) = s[0];
    }
  });
}

// Sum of n partial rows [.][P][R] at `src` (`step` floats apart), in order.
__device__ __forceinline__ float4v sum_parts(const float* src, int n, int64_t step) {
  float4v s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int i = 0; i < n; ++i) s += *reinterpret_cast<const float4v*>(src + i * step);
  return s;
}

template <bool kInt8, bool kXF32>
__global__ void __launch_bounds__(kT, kInt8 ? 2 : 4) a_kernel(Params p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int per = 2 * p.n_a, u = blockIdx.x / per, item = blockIdx.x - u * per;
  const int4 unit = p.g.unit_info[u];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int tok = p.g.unit_tok[u * kM + (lane & 3)];
  if (u >= p.g.meta[4]) return;
  const int kind = item & 1, split = item >> 1;
  const int cols = min(p.R, (rank_of(p, unit.x, kind) + 31) & ~31);
  if (cols == 0) return;
  const uint32_t lut0 = lds_addr(smem), lut = lut0 + (lane & (kCopies - 1)) * 8;
  const int row0 = split * p.a_rows, rows = min(p.a_rows, p.d - row0);
  ActX<kXF32> act;
  act.src = static_cast<const char*>(p.x) +
            (static_cast<int64_t>(tok) * p.d + row0 + 8 * (lane >> 4)) * (kXF32 ? 4 : 2);
  act.bf16 = p.x_dtype == LATENT_BF16;
  auto ready = [&]() __attribute__((always_inline)) {
    lut_fill(lut0, tid);
    lds_barrier();
  };
  rank_gemm<kInt8>(p.fac[kind ? F_UP_A : F_GATE_A], unit.x, row0, rows / 32, cols, unit.z, lut, lut0, act, ready,
                   p.part_a + (static_cast<int64_t>(split * 2 + kind) * p.P + unit.y) * p.R, p.R);
}

template <bool kInt8>
__global__ void __launch_bounds__(kT, kInt8 ? 2 : 4) bc_kernel(Params p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int u = blockIdx.x / p.n_c, item = blockIdx.x - u * p.n_c;
  const int4 unit = p.g.unit_info[u];
  if (u >= p.g.meta[4]) return;
  const int e = unit.x, m = unit.z;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid >> 6);
  const int n = lane & 15, kq = lane >> 4;
  // LDS: h rows, level table, then the latents (gate and up halves of a row),
  // whose place the waves' products take.
  const int lstr = 2 * p.R + 4;
  const uint32_t L_h = lds_addr(smem), lut0 = L_h + kM * kHStr * 4, L_lat = lut0 + kLutBytes;
  const uint32_t lut = lut0 + (lane & (kCopies - 1)) * 8;
  const int rk[2] = {rank_of(p, e, 0), rank_of(p, e, 1)}, rd = rank_of(p, e, 2);
  // Waves: (gate, up) x (columns 0-127, 128-255) x halves of the rank.
  const int c0 = item * kCB, ncol = min(kCB, p.ff - c0);
  const int kind = wave & 1, tile = (wave >> 1) & 1, kp = wave >> 2;
  const int nb = ((kind ? rk[1] : rk[0]) + 31) / 32, live = tile * 128 < ncol ? nb : 0;
  Walk<8, kInt8, ActLds> walk(p.fac[kind ? F_UP_B : F_GATE_B], e, c0 + tile * 128, 0, kp * live / 2,
                              (kp + 1) * live / 2, lane,
                              ActLds{L_lat + static_cast<uint32_t>((n & 3) * lstr + kind * p.R + 8 * kq) * 4u});
  walk.start();
  lut_fill(lut0, tid);
  const int r4 = p.R / 4;
  for (int i = tid; i < kM * 2 * r4; i += kT) {  // latents: A's partials in range order, zero past the rank
    const int r = i / (2 * r4), k = (i / r4) & 1, c = (i % r4) * 4;
    float4v s = {0.f, 0.f, 0.f, 0.f};
    if (r < m && c < rk[k])
      s = sum_parts(p.part_a + (static_cast<int64_t>(k) * p.P + unit.y + r) * p.R + c, p.n_a,
                    2 * static_cast<int64_t>(p.P) * p.R);
#pragma unroll
    for (int q = 0; q < 4; ++q) s[q] = c + q < rk[k] ? s[q] : 0.f;
    lds_st<float4v>(L_lat + static_cast<uint32_t>(r * lstr + k * p.R + c) * 4u, s);
  }
  lds_barrier();
  Acc<8> acc;
  walk.run(lut, acc);
  lds_barrier();  // the latents are read
  const uint32_t slot = L_lat + static_cast<uint32_t>(((kind * 2 + tile) * kM + kq) * kTileStr + n * 8) * 4u;
  const uint32_t hat = L_h + static_cast<uint32_t>(kq * kHStr + tile * 128 + n * 8) * 4u;
  if (kp == 1) store_tile(slot, acc);
  lds_barrier();
  if (kp == 0) {
    add_tile(slot, acc);
    if (kind == 0) store_tile(hat, acc);
  }
  lds_barrier();
  if (kp == 0 && kind == 1) {
    const float w = p.wbd && kq < m ? p.g.pair_w[unit.y + kq] : 1.f;
#pragma unroll
    for (int c = 0; c < 8; c += 4) {
      const float4v g = lds_ld<float4v>(hat + 4u * c);
      float4v h;
#pragma unroll
      for (int q = 0; q < 4; ++q) h[q] = g[q] / (1.0f + expf(-g[q])) * acc.r[c + q] * w;
      lds_st<float4v>(hat + 4u * c, h);
    }
  }
  const int cols = min(p.R, (rd + 31) & ~31);
  if (cols == 0) return;
  rank_gemm<kInt8>(p.fac[F_DOWN_A], e, c0, ncol / 32, cols, m, lut, L_lat,
                   ActLds{L_h + static_cast<uint32_t>((n & 3) * kHStr + 8 * kq) * 4u}, [] { lds_barrier(); },
                   p.part_c + (static_cast<int64_t>(item) * p.P + unit.y) * p.R, p.R);
}

template <bool kInt8>
__global__ void __launch_bounds__(kT, kInt8 ? 2 : 4) d_kernel(Params p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int u = blockIdx.x / p.n_d, item = blockIdx.x - u * p.n_d;
  const int4 unit = p.g.unit_info[u];
  if (u >= p.g.meta[4]) return;
  const int e = unit.x, m = unit.z;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid >> 6);
  const int n = lane & 15, kq = lane >> 4;
  const uint32_t lut0 = lds_addr(smem), L_lat = lut0 + kLutBytes;
  const uint32_t lut = lut0 + (lane & (kCopies - 1)) * 8;
  const int rd = rank_of(p, e, 2), lstr = p.R + 4, r4 = p.R / 4;
  // Waves: four tiles of 128 columns x halves of the rank.
  const int tile = wave & 3, kp = wave >> 2, c0 = item * kCD + tile * 128;
  const int live = c0 < p.d ? (rd + 31) / 32 : 0;
  Walk<8, kInt8, ActLds> walk(p.fac[F_DOWN_B], e, c0, 0, kp * live / 2, (kp + 1) * live / 2, lane,
                              ActLds{L_lat + static_cast<uint32_t>((n & 3) * lstr + 8 * kq) * 4u});
  walk.start();
  lut_fill(lut0, tid);
  for (int i = tid; i < kM * r4; i += kT) {
    const int r = i / r4, c = (i - r * r4) * 4;
    float4v s = {0.f, 0.f, 0.f, 0.f};
    if (r < m && c < rd)
      s = sum_parts(p.part_c + (static_cast<int64_t>(unit.y) + r) * p.R + c, p.n_c, static_cast<int64_t>(p.P) * p.R);
#pragma unroll
    for (int q = 0; q < 4; ++q) s[q] = c + q < rd ? s[q] : 0.f;
    lds_st<float4v>(L_lat + static_cast<uint32_t>(r * lstr + c) * 4u, s);
  }
  lds_barrier();
  Acc<8> acc;
  walk.run(lut, acc);
  lds_barrier();  // the latents are read
  const uint32_t slot = L_lat + static_cast<uint32_t>((tile * kM + kq) * kTileStr + n * 8) * 4u;
  if (kp == 1) store_tile(slot, acc);
  lds_barrier();
  const int col = c0 + n * 8;
  if (kp == 1 || col >= p.d || kq >= m) return;
  add_tile(slot, acc);
  float* dst = p.y + static_cast<int64_t>(unit.y + kq) * p.d + col;
#pragma unroll
  for (int c = 0; c < 8; c += 4)
    *reinterpret_cast<float4v*>(dst + c) = float4v{acc.r[c], acc.r[c + 1], acc.r[c + 2], acc.r[c + 3]};
}

// Output rows from the y rows: the weighted sum over a token's slots in slot
// order, or each slot's row (zero where dropped).  One float4 per thread.
constexpr int kCombineT = 256;
__global__ void __launch_bounds__(kCombineT) combine_kernel(Params p) {
  const int d4 = p.d / 4;
  const int row = blockIdx.y, c = blockIdx.x * kCombineT + threadIdx.x;
  if (c >= d4) return;
  const float4v* y = reinterpret_cast<const float4v*>(p.y) + c;
  float4v s = {0.f, 0.f, 0.f, 0.f};
  if (p.out_mode == LATENT_OUT_REDUCED) {
#pragma unroll 8
    for (int k = 0; k < p.K; ++k) {
      const int slot = row * p.K + k, e = p.ids[slot];
      if (e < 0 || e >= p.E) continue;
      const float w = p.wbd ? 1.f : load_act(p.weights, p.w_dtype, slot);
      s += w * y[static_cast<int64_t>(p.g.pos_of[slot]) * d4];
    }
  } else {
    const int e = p.ids[row];
    if (e >= 0 && e < p.E) s = y[static_cast<int64_t>(p.g.pos_of[row]) * d4];
  }
  reinterpret_cast<float4v*>(p.out)[static_cast<int64_t>(row) * d4 + c] = s;
}

inline size_t align256(size_t v) { return (v + 255) / 256 * 256; }

template <bool kInt8>
int launch(const Params& p, unsigned units, hipStream_t s) {
  const size_t lds_a = std::max(kRedBytes, kLutBytes);  // the products go over the table
  const size_t lds_bc = kM * kHStr * 4 + kLutBytes + std::max<size_t>(kM * (2 * p.R + 4) * 4, kRedBytes);
  const size_t lds_d = kLutBytes + std::max<size_t>(kM * (p.R + 4) * 4, kRedBytes);
  const bool xf32 = p.x_dtype == LATENT_F32;
  auto a_k = xf32 ? a_kernel<kInt8, true> : a_kernel<kInt8, false>;
  hipLaunchKernelGGL(a_k, dim3(units * 2 * p.n_a), dim3(kT), lds_a, s, p);
  hipLaunchKernelGGL(bc_kernel<kInt8>, dim3(units * p.n_c), dim3(kT), lds_bc, s, p);
  hipLaunchKernelGGL(d_kernel<kInt8>, dim3(units * p.n_d), dim3(kT), lds_d, s, p);
  const unsigned rows = static_cast<unsigned>(p.out_mode == LATENT_OUT_REDUCED ? p.T : p.P);
  hipLaunchKernelGGL(combine_kernel, dim3((p.d / 4 + kCombineT - 1) / kCombineT, rows), dim3(kCombineT), 0, s, p);
  return hipGetLastError() == hipSuccess ? LATENT_OK : LATENT_E_HIP;
}

}  // namespace

bool supported(const latent_moe_args& a) {
  const int64_t P = a.n_tokens * a.n_expert_used;
  if (a.layout != LATENT_LAYOUT_ROWS || P < kMinPairs || P > kMaxPairs || a.n_expert > kMaxExpert) return false;
  if (a.max_rank > 512 || (reinterpret_cast<uintptr_t>(a.x) & 15u) != 0) return false;  // 16-byte loads of x
  // A factor's INT8 side buffer stays below 2^31 bytes even if every group is
  // INT8 (the same bound as the row-layout fp16 phases').
  const latent_factor* fs[6] = {&a.gate_a, &a.gate_b, &a.up_a, &a.up_b, &a.down_a, &a.down_b};
  for (const latent_factor* f : fs)
    if (f->int8_bitmap && a.n_expert * f->rows * f->cols >= (int64_t{1} << 31)) return false;
  return true;
}

int64_t max_units(const latent_moe_args& a) {
  const int64_t P = a.n_tokens * a.n_expert_used;
  return std::min(P, std::min(P, a.n_expert) + P / kUnitPairs);
}

Layout layout_for(const latent_moe_args& a) {
  const int64_t T = a.n_tokens, K = a.n_expert_used, E = a.n_expert, R = a.max_rank, P = T * K;
  // Phase A items at the units a uniform routing gives: the range of d (whole
  // blocks of 32 rows for each of eight waves) whose rounds of 512 workgroups
  // (two per CU) take the fewest rows, a round costing some 128 rows besides.
  const double active = static_cast<double>(E) * (1.0 - std::pow(1.0 - static_cast<double>(K) / E, static_cast<double>(T)));
  const double units = std::max(active, static_cast<double>(P) / kUnitPairs);
  int64_t best = 0, best_rows = 256;
  for (int64_t n = 1; n <= 16; ++n) {
    const int64_t rows = ((a.n_embd + n - 1) / n + 255) / 256 * 256;
    const int64_t rounds = static_cast<int64_t>(std::ceil(2.0 * units * ((a.n_embd + rows - 1) / rows) / 512.0));
    const int64_t cost = rounds * (rows + 128);
    if (best == 0 || cost < best) {
      best = cost;
      best_rows = rows;
    }
  }
  Layout L{};
  L.a_rows = static_cast<int>(best_rows);
  L.n_a = static_cast<int>((a.n_embd + L.a_rows - 1) / L.a_rows);
  L.n_c = static_cast<int>((a.n_ff + kCB - 1) / kCB);
  L.n_d = static_cast<int>((a.n_embd + kCD - 1) / kCD);
  size_t off = 0;
  L.units = off;  off = align256(off + max_units(a) * (sizeof(int4) + kUnitPairs * sizeof(int)));
  L.pos_of = off; off = align256(off + P * sizeof(int));
  L.part_a = off; off = align256(off + static_cast<size_t>(L.n_a) * 2 * P * R * 4);
  L.part_c = off; off = align256(off + static_cast<size_t>(L.n_c) * P * R * 4);
  L.y = off;      off = align256(off + static_cast<size_t>(P) * a.n_embd * 4);
  L.total = off;
  return L;
}

int forward(const latent_moe_args& a, const Factor* fac, const Grouping& g, char* scratch, hipStream_t s) {
  const Layout L = layout_for(a);
  Params p{};
  bool int8 = false;
  for (int i = 0; i < 6; ++i) {
    p.fac[i] = fac[i];
    int8 = int8 || fac[i].ext.bitmap != nullptr;
  }
  p.x = a.x;
  p.ids = a.ids;
  p.weights = a.weights;
  p.ranks = a.ranks;
  p.g = g;
  p.part_a = reinterpret_cast<float*>(scratch + L.part_a);
  p.part_c = reinterpret_cast<float*>(scratch + L.part_c);
  p.y = reinterpret_cast<float*>(scratch + L.y);
  p.out = static_cast<float*>(a.out);
  p.x_dtype = a.x_dtype;
  p.w_dtype = a.weights_dtype;
  p.T = static_cast<int>(a.n_tokens);
  p.d = static_cast<int>(a.n_embd);
  p.ff = static_cast<int>(a.n_ff);
  p.E = static_cast<int>(a.n_expert);
  p.K = static_cast<int>(a.n_expert_used);
  p.R = static_cast<int>(a.max_rank);
  p.P = p.T * p.K;
  p.wbd = a.weight_before_down ? 1 : 0;
  p.out_mode = a.out_mode;
  p.a_rows = L.a_rows;
  p.n_a = L.n_a;
  p.n_c = L.n_c;
  p.n_d = L.n_d;
  const unsigned units = static_cast<unsigned>(max_units(a));
  return int8 ? launch<true>(p, units, s) : launch<false>(p, units, s);
}

}  // namespace chain32
}  // namespace latent
