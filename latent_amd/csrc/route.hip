// Router front end of a LATENT MoE layer on gfx950: logits, softmax, top-k,
// renormalisation and the optional drop rules, producing the (ids, weights)
// operands of latent_moe_ffn_forward on the device.
//
// The reference leaves routing to the graph builder (build_moe_ffn_latent,
// README.md:111-113, patch 004 empty) and restates the adaptive drop on the
// host (loader/adaptive_topk.py:29-90).  Here it is two kernels, so a whole
// decode layer (route + expert FFN) is stream-ordered device work that a HIP
// graph can hold:
//
//   logits_kernel  partial logits of x . W_r over one 64-row slice of d for a
//                  64-expert x 32-token tile; slices go to their own slot of the
//                  workspace (no atomics, fixed summation order).
//   split_logits_kernel  the same for longer batches: 128-token x 128-expert
//                  tiles over a few long slices of d, on bf16 matrix cores
//                  with every fp32 operand split into three bf16 parts.
//   topk_kernel    one workgroup per token: sum the slices in slice order (or
//                  read caller logits), top-k by repeated wave arg-max (ties ->
//                  the lower expert id), weights exp(l - max) renormalised over
//                  the kept k, then the drop rule.
//
// Work per call: the router matrix is read once per token block (d*E*4 B in
// fp32 = 7.3 MB at d=7168, E=256); short batches are bound by that read,
// top-k by latency.
#include "common.hpp"

#include <algorithm>
#include <type_traits>

namespace latent {
namespace route {
namespace {

constexpr int kThreads = 256;
constexpr int kRows = 64;      // rows of d per logits workgroup
constexpr int kCols = 64;      // experts per logits workgroup
constexpr int kTok = 32;       // tokens per logits workgroup
constexpr int kMaxE = 1024;    // experts: 16 per lane in topk_kernel
constexpr int kPerLane = kMaxE / kWave;
constexpr int kMaxK = kWave;  // slot s lives in lane s
constexpr int kSliceBatch = 128;  // logit slices a topk thread loads at once
constexpr int kFewSlices = 32;    // most slices of the split kernel

struct Params {
  const void* x;
  int x_dtype;
  const void* router;
  int router_dtype;
  const float* logits_in;
  float* logits_out;
  int32_t* ids;
  float* weights;
  float* partial;  // [nslice][T][E]
  int T, d, E, K, nslice, drop_rule;
  int slice_rows;  // rows of d per slice (split_logits_kernel)
  float drop_param;
  bool vec_router, vec_x;  // 4-element vector loads allowed (alignment, row length)
};

// Four consecutive elements [i, i+4) of a row of `n` elements (f32 / f16 /
// bf16), zero beyond n.  `vec`: the row start and i are 4-element aligned and
// the base is 16-byte (f32) or 8-byte (16-bit types) aligned.
__device__ __forceinline__ float4 load4(const void* base, int dtype, int64_t row_off, int i, int n, bool vec) {
  float v[4];
  if (vec && i + 4 <= n) {
    if (dtype == LATENT_F32) return *reinterpret_cast<const float4*>(static_cast<const float*>(base) + row_off + i);
    const uint2 u = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(base) + row_off + i);
    const uint32_t h[4] = {u.x & 0xFFFFu, u.x >> 16, u.y & 0xFFFFu, u.y >> 16};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = dtype == LATENT_BF16 ? __uint_as_float(h[q] << 16) : half_bits_to_float(static_cast<uint16_t>(h[q]));
    return make_float4(v[0], v[1], v[2], v[3]);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = i + q < n ? load_act(base, dtype, row_off + i + q) : 0.f;
  return make_float4(v[0], v[1], v[2], v[3]);
}

// grid (ceil(E/64), nslice, ceil(T/32)); 256 threads.  Every thread issues its
// 4 router chunks and 2 activation chunks (4 elements each) before the first
// LDS store, so a workgroup costs about one memory round trip.  The 32 x 64
// tile is then computed on fp32 matrix cores (v_mfma_f32_16x16x4_f32: fp32
// products and accumulation): wave w owns experts 16w..16w+15 and both
// 16-token halves, 16 steps of 4 rows (64-row slices: the dependent MFMA
// chains of 128-row slices took 9.7 us against 7.2 at d = 7168, batch 32).
typedef float float4v __attribute__((ext_vector_type(4)));
constexpr int kWPitch = kCols + 4;  // router tile row pitch (floats): fewer bank conflicts
__global__ void __launch_bounds__(kThreads) logits_kernel(Params p) {
  __shared__ float xs[kTok][kRows + 4];
  __shared__ float ws[kRows][kWPitch];
  const int tid = threadIdx.x;
  const int e0 = blockIdx.x * kCols, r0 = blockIdx.y * kRows, t0 = blockIdx.z * kTok;
  const int nr = min(kRows, p.d - r0), nt = min(kTok, p.T - t0), ne = min(kCols, p.E - e0);
  constexpr int kWChunks = kRows * kCols / 4 / kThreads;  // 8
  constexpr int kXChunks = kTok * kRows / 4 / kThreads;   // 4
  float4 wv[kWChunks], xv[kXChunks];
#pragma unroll
  for (int u = 0; u < kWChunks; ++u) {
    const int i = tid + u * kThreads, r = i / (kCols / 4), c = (i % (kCols / 4)) * 4;
    wv[u] = r < nr ? load4(p.router, p.router_dtype, static_cast<int64_t>(r0 + r) * p.E + e0, c, ne, p.vec_router)
                   : make_float4(0.f, 0.f, 0.f, 0.f);
  }
#pragma unroll
  for (int u = 0; u < kXChunks; ++u) {
    const int i = tid + u * kThreads, t = i / (kRows / 4), r = (i % (kRows / 4)) * 4;
    xv[u] = t < nt ? load4(p.x, p.x_dtype, static_cast<int64_t>(t0 + t) * p.d + r0, r, nr, p.vec_x)
                   : make_float4(0.f, 0.f, 0.f, 0.f);
  }
#pragma unroll
  for (int u = 0; u < kWChunks; ++u) {
    const int i = tid + u * kThreads, r = i / (kCols / 4), c = (i % (kCols / 4)) * 4;
    *reinterpret_cast<float4*>(&ws[r][c]) = wv[u];
  }
#pragma unroll
  for (int u = 0; u < kXChunks; ++u) {
    const int i = tid + u * kThreads, t = i / (kRows / 4), r = (i % (kRows / 4)) * 4;
    *reinterpret_cast<float4*>(&xs[t][r]) = xv[u];
  }
  __syncthreads();
  // Lane l: A = x[16h + l % 16][k + l / 16], B = W[k + l / 16][16w + l % 16];
  // C lane l holds rows 4 (l / 16) .. + 3 of column l % 16.
  const int lane = tid & (kWave - 1), w = tid >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  float4v acc[2] = {float4v{0.f, 0.f, 0.f, 0.f}, float4v{0.f, 0.f, 0.f, 0.f}};
#pragma unroll 8
  for (int k = 0; k < kRows; k += 4) {  // rows beyond nr hold zeros
    const float b = ws[k + lk][w * 16 + lr];
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[lr][k + lk], b, acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[16 + lr][k + lk], b, acc[1], 0, 0, 0);
  }
  const int c = w * 16 + lr;
  if (c < ne) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = h * 16 + lk * 4 + i;
        if (t < nt) p.partial[(static_cast<int64_t>(blockIdx.y) * p.T + t0 + t) * p.E + e0 + c] = acc[h][i];
      }
  }
}

// ---- split_logits_kernel -------------------------------------------------------
// Logits of longer batches.  A product of fp32 values is the sum of products of
// their bf16 parts: v = v1 + v2 + v3 exactly, each part what the earlier ones
// left rounded to the nearest bf16 (bf16 x is one part, f16 x two), and bf16
// products are exact in fp32.  Three bf16 MFMAs (bf16 x, fp32 router) replace
// the eight v_mfma_f32_16x16x4_f32 of the same 16x16x32 block at a sixteenth of
// their cycles each.  x2 w3, x3 w2 and x3 w3 are left out: |v2| <= 2^-8 |v| and
// |v3| <= 2^-16 |v|, so each is at most 2^-24 of the product, the rounding of one
// fp32 product, and of either sign (parts cut off instead of rounded leave terms
// up to 2^-22, all of the product's sign: on positive data a bias).
//
// Workgroup: 128 tokens (two workgroups per CU) or 256 (one) x 128 experts,
// waves of 64 x 64, one slice of d in steps of 32 rows, the next two steps'
// x and router rows in flight in registers (barriers wait for LDS only).  With
// 256 tokens each router value is split half as often per token and, one
// workgroup filling the CU, the LDS tile is double-buffered: a step's MFMAs
// run beside the splitting of the next.  Slices of equal index land on one XCD (workgroups go to the 8 XCDs
// round robin), whose L2 then holds that slice of the router for all token
// tiles.  The terms below x1 w1 are summed in accumulators of their own: added
// to the leading sums they would round at those sums' magnitude.
//
// A non-finite operand, or one that rounds to infinity, has no such parts (inf -
// inf): its logits come out NaN, and topk_kernel computes every NaN logit again
// in fp32.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
constexpr int kSTok = 128, kSExp = 128, kSStep = 32;  // kSTok: the smaller token tile
constexpr int kSPitch = kSStep + 8;  // bf16 per LDS row: 16-byte reads of 16 rows on distinct banks

// The parts of 8 consecutive values as bf16x8 words.
template <int N>
__device__ __forceinline__ void split8(const float (&v)[8], u32x4 (&part)[N]) {
  float r[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) r[j] = v[j];
#pragma unroll
  for (int n = 0; n < N; ++n) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      part[n][j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(float2v{r[2 * j], r[2 * j + 1]}, bf16x2));
      if (n + 1 < N) {
        r[2 * j] -= __uint_as_float(part[n][j] << 16);
        r[2 * j + 1] -= __uint_as_float(part[n][j] & 0xFFFF0000u);
      }
    }
  }
}

// Workgroup barrier over LDS only (__syncthreads() would also wait for the
// loads issued ahead).
__device__ __forceinline__ void lds_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt left at their maxima
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// kXType: LATENT_* of x; kWF32: fp32 router (else bf16); kVecX: x rows are
// 16-byte aligned; kTok: tokens per workgroup.  d is a multiple of kSStep.
template <int kXType, bool kWF32, bool kVecX, int kTok>
__global__ void __launch_bounds__(2 * kTok, 2) split_logits_kernel(Params p) {
  constexpr int NX = kXType == LATENT_F32 ? 3 : kXType == LATENT_F16 ? 2 : 1;
  constexpr int NW = kWF32 ? 3 : 1;
  constexpr int kWRows = kSStep * kSExp / (2 * kTok);  // router rows a thread loads per step
  constexpr int kBufs = kTok > kSTok ? 2 : 1;
  __shared__ __attribute__((aligned(16))) uint16_t xs[kBufs][NX][kTok][kSPitch];
  __shared__ __attribute__((aligned(16))) uint16_t ws[kBufs][NW][kSExp][kSPitch];
  const int tid = threadIdx.x;
  const int slice = blockIdx.x % p.nslice, tile = blockIdx.x / p.nslice;
  const int neb = (p.E + kSExp - 1) / kSExp;
  const int e0 = (tile % neb) * kSExp, t0 = (tile / neb) * kTok;
  const int k_begin = slice * p.slice_rows, k_end = min(p.d, k_begin + p.slice_rows);
  const int nt = min(kTok, p.T - t0), ne = min(kSExp, p.E - e0);
  // x pieces of 8 values: thread -> rows tid / 4 and tid / 4 + kTok / 2, piece
  // tid % 4.  Router: column tid % 128, kWRows rows from kWRows (tid / 128).
  const int xr = tid >> 2, xk = (tid & 3) * 8;
  const int we = tid & (kSExp - 1), wk = (tid >> 7) * kWRows;
  struct Ahead {
    u32x4 x[2][kXType == LATENT_F32 ? 2 : 1];
    uint32_t w[kWRows];
  };
  const char* xrow[2];  // rows and columns beyond nt, ne: their results are not stored
#pragma unroll
  for (int h = 0; h < 2; ++h)
    xrow[h] = static_cast<const char*>(p.x) + (static_cast<int64_t>(t0 + min(xr + kTok / 2 * h, nt - 1)) * p.d + xk) *
                                                  (kXType == LATENT_F32 ? 4 : 2);
  const char* wcol = static_cast<const char*>(p.router) +
                     (static_cast<int64_t>(wk) * p.E + e0 + min(we, ne - 1)) * (kWF32 ? 4 : 2);
  const int64_t wrow = static_cast<int64_t>(p.E) * (kWF32 ? 4 : 2);
  auto load = [&](int k0, Ahead& r) __attribute__((always_inline)) {
    k0 = min(k0, k_end - kSStep);  // the same loads on every path
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < (kXType == LATENT_F32 ? 2 : 1); ++q) {
        const char* src = xrow[h] + static_cast<int64_t>(k0) * (kXType == LATENT_F32 ? 4 : 2) + 16 * q;
        if (kVecX) {
          r.x[h][q] = *reinterpret_cast<const u32x4*>(src);
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            r.x[h][q][j] = kXType == LATENT_F32 ? reinterpret_cast<const uint32_t*>(src)[j]
                                                : reinterpret_cast<const uint16_t*>(src)[2 * j] |
                                                      static_cast<uint32_t>(reinterpret_cast<const uint16_t*>(src)[2 * j + 1]) << 16;
        }
      }
    const char* src = wcol + k0 * wrow;
#pragma unroll
    for (int j = 0; j < kWRows; ++j, src += wrow)
      r.w[j] = kWF32 ? *reinterpret_cast<const uint32_t*>(src)
                     : static_cast<uint32_t>(*reinterpret_cast<const uint16_t*>(src)) << 16;
  };
  auto stage = [&](int buf, const Ahead& r) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4 part[NX];
      if (kXType == LATENT_BF16) {
        part[0] = r.x[h][0];
      } else {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          v[j] = kXType == LATENT_F32 ? __uint_as_float(r.x[h][(j >> 2) & (kXType == LATENT_F32 ? 1 : 0)][j & 3])
                                      : half_bits_to_float(static_cast<uint16_t>(r.x[h][0][j >> 1] >> (16 * (j & 1))));
        split8<NX>(v, part);
      }
#pragma unroll
      for (int n = 0; n < NX; ++n) *reinterpret_cast<u32x4*>(&xs[buf][n][xr + kTok / 2 * h][xk]) = part[n];
    }
#pragma unroll
    for (int g = 0; g < kWRows / 8; ++g) {
      u32x4 part[NW];
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = __uint_as_float(r.w[8 * g + j]);
      split8<NW>(v, part);
#pragma unroll
      for (int n = 0; n < NW; ++n) *reinterpret_cast<u32x4*>(&ws[buf][n][we][wk + 8 * g]) = part[n];
    }
  };
  const int lane = tid & (kWave - 1), w = tid >> 6;
  const int lr = lane & 15, lk = (lane >> 4) * 8;
  const int tw = (w >> 1) * 64, ew = (w & 1) * 64;
  constexpr bool kLow = NX * NW > 1;
  float4v acc[4][4] = {}, low[kLow ? 4 : 1][kLow ? 4 : 1] = {};
  // Two buffers: buffer buf holds step k0, r the registers of the step after
  // it.  One buffer: r holds step k0.
  auto step = [&](int buf, int k0, Ahead& r) __attribute__((always_inline)) {
    lds_barrier();  // two: buffer buf is complete and 1 - buf read; one: the buffer is read
    if (kBufs == 1) {
      stage(0, r);
      lds_barrier();
      load(k0 + 2 * kSStep, r);
    }
    bf16x8 a[NX][4];
#pragma unroll
    for (int n = 0; n < NX; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) a[n][i] = *reinterpret_cast<const bf16x8*>(&xs[buf][n][tw + 16 * i + lr][lk]);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int m = 0; m < NW; ++m) {
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(&ws[buf][m][ew + 16 * j + lr][lk]);
#pragma unroll
        for (int n = 0; n < NX; ++n) {
          if (n + m > 2) continue;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float4v& d = kLow && n + m > 0 ? low[kLow ? i : 0][kLow ? j : 0] : acc[i][j];
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[n][i], b, d, 0, 0, 0);
          }
        }
      }
    if (kBufs == 2) {
      stage(1 - buf, r);  // past the slice's end: never read
      load(k0 + 3 * kSStep, r);
    }
  };
  Ahead r0, r1;
  load(k_begin, r0);
  load(k_begin + kSStep, r1);
  if (kBufs == 2) {
    stage(0, r0);
    load(k_begin + 2 * kSStep, r0);
  }
  for (int k0 = k_begin; k0 < k_end; k0 += 2 * kSStep) {
    step(0, k0, kBufs == 2 ? r1 : r0);
    if (k0 + kSStep < k_end) step(kBufs - 1, k0 + kSStep, kBufs == 2 ? r0 : r1);
  }
  if (kLow) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] += low[kLow ? i : 0][kLow ? j : 0];
  }
  // Lane: tokens 16 i + 4 (lane / 16) + q, expert 16 j + lane % 16.
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int t = tw + 16 * i + (lane >> 4) * 4 + q;
      if (t >= nt) continue;
      float* dst = p.partial + (static_cast<int64_t>(slice) * p.T + t0 + t) * p.E + e0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = ew + 16 * j + lr;
        if (e < ne) dst[e] = acc[i][j][q];
      }
    }
}

// Wave arg-max of (v, idx) pairs: larger v wins, equal v -> smaller idx.
// Each pair is one 64-bit key whose unsigned order is that order (the
// float's bits made monotonic above, the complemented index below; -0 is
// +0 first, so equal values tie), reduced over the wave with DPP row
// permutations and the permlane swaps (no LDS round trips).
__device__ __forceinline__ void wave_argmax(float& v, int& idx) {
  const uint32_t u = __float_as_uint(v + 0.0f);
  uint32_t hi = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  uint32_t lo = ~static_cast<uint32_t>(idx);
  auto take = [&](uint32_t ohi, uint32_t olo) __attribute__((always_inline)) {
    const bool gt = ohi > hi || (ohi == hi && olo > lo);
    hi = gt ? ohi : hi;
    lo = gt ? olo : lo;
  };
  auto dpp = [&](auto ctrl) __attribute__((always_inline)) {
    constexpr int c = decltype(ctrl)::value;
    take(static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(hi), c, 0xF, 0xF, false)),
         static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(lo), c, 0xF, 0xF, false)));
  };
  dpp(std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]: lane ^ 1
  dpp(std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]: lane ^ 2
  dpp(std::integral_constant<int, 0x124>{});  // row_ror:4
  dpp(std::integral_constant<int, 0x128>{});  // row_ror:8
  {  // rows r and r ^ 1
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const uint32_t h0 = h[0], h1 = h[1], l0 = l[0], l1 = l[1];
    hi = h0; lo = l0;
    take(h1, l1);
  }
  {  // lane halves
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const uint32_t h0 = h[0], h1 = h[1], l0 = l[0], l1 = l[1];
    hi = h0; lo = l0;
    take(h1, l1);
  }
  v = __uint_as_float((hi & 0x80000000u) ? (hi & 0x7FFFFFFFu) : ~hi);
  idx = static_cast<int>(~lo);
}

// Wave: top-k of the logits l[j] (expert j 64 + lane; -inf beyond E), weights
// and drop rule of token t.  NJ: experts per lane.
template <int NJ>
__device__ __forceinline__ void select_topk(const Params& p, int t, int lane, const float (&l)[NJ]) {
  const int nj = (p.E + kWave - 1) / kWave;
  // Top-k: k rounds of wave arg-max; a chosen expert is retired with a bit
  // of `taken`, so it cannot be chosen again even if every logit is -inf.
  // Lane s keeps the logit and id of slot s.
  uint32_t taken = 0;
  float my_l = -INFINITY;
  int my_e = -1;
  for (int s = 0; s < p.K; ++s) {
    float bv = -INFINITY;
    int bi = 0x7FFFFFFF;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if (j >= nj) break;  // wave-uniform: the layer's experts only
      const int e = j * kWave + lane;
      const bool ok = e < p.E && !((taken >> j) & 1u);
      if (ok && (l[j] > bv || bi == 0x7FFFFFFF)) {
        bv = l[j];
        bi = e;
      }
    }
    wave_argmax(bv, bi);
    if (lane == s) {
      my_l = bv;
      my_e = bi;
    }
    if (bi != 0x7FFFFFFF && (bi & (kWave - 1)) == lane) taken |= 1u << (bi / kWave);
  }
  // Renormalised softmax over the kept k (the full softmax denominator
  // cancels); sums run serially in slot order.
  const float m = __shfl(my_l, 0, kWave);
  float w = lane < p.K ? expf(my_l - m) : 0.f;
  float wsum = 0.f;
  for (int s = 0; s < p.K; ++s) wsum += __shfl(w, s, kWave);
  w = w / wsum;
  int keep = p.K;
  if (p.drop_rule == LATENT_DROP_INCLUSIVE) {
    // loader/adaptive_topk.py:29-55 on the descending top-k scores.
    float total = 0.f;
    for (int s = 0; s < p.K; ++s) total += __shfl(w, s, kWave);
    const float target = p.drop_param * total;
    float cum = 0.f;
    for (int s = 0; s < p.K; ++s) {
      const float ws = __shfl(w, s, kWave);
      if (cum + ws > target) {
        keep = s;
        break;
      }
      cum += ws;
    }
  }
  if (lane < p.K) {
    bool drop = lane >= keep;
    if (p.drop_rule == LATENT_DROP_BELOW && w < p.drop_param) drop = true;
    const int64_t o = static_cast<int64_t>(t) * p.K + lane;
    p.ids[o] = drop ? -1 : my_e;
    p.weights[o] = drop ? 0.f : w;
  }
}

// One token per 256-thread workgroup.  Thread e sums the slices of expert e
// (all loads in flight at once, added in slice order) into LDS; wave 0 then
// selects the top k.
__global__ void __launch_bounds__(kThreads) topk_kernel(Params p) {
  __shared__ float lg[kMaxE];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const int t = blockIdx.x;
  const int nj = (p.E + kWave - 1) / kWave;
  for (int e = threadIdx.x; e < p.E; e += kThreads) {
    float v;
    if (p.logits_in) {
      v = p.logits_in[static_cast<int64_t>(t) * p.E + e];
    } else {
      const float* src = p.partial + static_cast<int64_t>(t) * p.E + e;
      const int64_t stride = static_cast<int64_t>(p.T) * p.E;
      // Up to kSliceBatch slices in flight (d = 7168: all 112 in one round
      // trip), added in slice order.
      float part[kSliceBatch];
      v = 0.f;
      for (int s0 = 0; s0 < p.nslice; s0 += kSliceBatch) {
        // One pointer stepped by the slice stride (indexed loads kept one
        // scalar offset per slice and spilled them).
        typedef const __attribute__((address_space(1))) float* gptr;
        uintptr_t q = reinterpret_cast<uintptr_t>(src + s0 * stride);
#pragma unroll
        for (int i = 0; i < kSliceBatch; ++i) {
          part[i] = s0 + i < p.nslice ? *reinterpret_cast<gptr>(q) : 0.f;
          q += static_cast<uintptr_t>(stride) * sizeof(float);
          asm volatile("" : "+v"(q));
        }
#pragma unroll
        for (int i = 0; i < kSliceBatch; ++i) v += part[i];
      }
    }
    if (p.logits_out) p.logits_out[static_cast<int64_t>(t) * p.E + e] = v;
    lg[e] = v != v ? -INFINITY : v;  // NaN never wins a slot
  }
  __syncthreads();
  if (wave != 0) return;
  float l[kPerLane];
#pragma unroll
  for (int j = 0; j < kPerLane; ++j) {
    const int e = j * kWave + lane;
    l[j] = (j < nj && e < p.E) ? lg[e] : -INFINITY;
  }
  select_topk<kPerLane>(p, t, lane, l);
}

// The same for batches of the split kernel, one token per wave: lane l sums
// experts j 64 + l over the few slices.  4096 tokens, 256 experts, 8 slices:
// one token per workgroup (three of its four waves idle in the selection) took
// 36 us.
constexpr int kTopkWaves = 4;

// Workgroup: x . router of tokens t0 .. t0 + 3 in fp32 over 64-row slices, as
// logits_kernel sums it, into lg[token][expert].  A wave takes a quarter of the
// experts for all four tokens, a batch of router rows in flight.
template <int NJ, bool kWF32>
__device__ __forceinline__ void plain_logits(const Params& p, int t0, float (&xs)[kTopkWaves][kRows],
                                             float (&lg)[kTopkWaves][NJ * kWave]) {
  constexpr int kJ = NJ / kTopkWaves, kAhead = kSStep / kJ;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const int64_t xrow = static_cast<int64_t>(min(t0 + wave, p.T - 1)) * p.d;
  int e[kJ];
  float acc[kJ][kTopkWaves] = {};
#pragma unroll
  for (int j = 0; j < kJ; ++j) e[j] = min((wave * kJ + j) * kWave + lane, p.E - 1);
  for (int k0 = 0; k0 < p.d; k0 += kRows) {
    const int rows = min(kRows, p.d - k0);  // a multiple of kSStep
    __syncthreads();
    xs[wave][lane] = load_act(p.x, p.x_dtype, xrow + k0 + min(lane, rows - 1));
    __syncthreads();
    float s[kJ][kTopkWaves] = {};
    for (int r = 0; r < rows; r += kAhead) {
      float w[kAhead][kJ];
#pragma unroll
      for (int i = 0; i < kAhead; ++i)
#pragma unroll
        for (int j = 0; j < kJ; ++j)
          w[i][j] = load_act(p.router, kWF32 ? LATENT_F32 : LATENT_BF16, static_cast<int64_t>(k0 + r + i) * p.E + e[j]);
#pragma unroll
      for (int i = 0; i < kAhead; ++i)
#pragma unroll
        for (int t = 0; t < kTopkWaves; ++t) {
          const float x = xs[t][r + i];
#pragma unroll
          for (int j = 0; j < kJ; ++j) s[j][t] = fmaf(x, w[i][j], s[j][t]);
        }
    }
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
      for (int t = 0; t < kTopkWaves; ++t) acc[j][t] += s[j][t];
  }
#pragma unroll
  for (int j = 0; j < kJ; ++j)
#pragma unroll
    for (int t = 0; t < kTopkWaves; ++t) lg[t][(wave * kJ + j) * kWave + lane] = acc[j][t];
  __syncthreads();
}

template <int NJ>
__global__ void __launch_bounds__(kTopkWaves * kWave) topk_wave_kernel(Params p) {
  __shared__ float xs[kTopkWaves][kRows];
  __shared__ float lg[kTopkWaves][NJ * kWave];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const int t = blockIdx.x * kTopkWaves + wave;
  const int64_t stride = static_cast<int64_t>(p.T) * p.E;
  const float* row = p.partial + static_cast<int64_t>(min(t, p.T - 1)) * p.E;
  float l[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) l[j] = 0.f;
#pragma unroll 4
  for (int s = 0; s < p.nslice; ++s) {  // slice order
    const float* src = row + s * stride;
#pragma unroll
    for (int j = 0; j < NJ; ++j) l[j] += src[min(j * kWave + lane, p.E - 1)];
  }
  bool nan = false;
#pragma unroll
  for (int j = 0; j < NJ; ++j) nan = nan || l[j] != l[j];
  if (__syncthreads_or(nan)) {
    // NaN logits in fp32, the workgroup's four tokens together: 4096 tokens of
    // one NaN each, d 7168, 256 experts 0.48 ms a call, finite 59 us.  A lane
    // summing a token's d alone took 10 ms, and its call's stack made the finite
    // ones 66.
    if (p.router_dtype == LATENT_F32)
      plain_logits<NJ, true>(p, blockIdx.x * kTopkWaves, xs, lg);
    else
      plain_logits<NJ, false>(p, blockIdx.x * kTopkWaves, xs, lg);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      if (l[j] != l[j]) l[j] = lg[wave][j * kWave + lane];
  }
  if (t >= p.T) return;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int e = j * kWave + lane;
    if (e < p.E && p.logits_out) p.logits_out[static_cast<int64_t>(t) * p.E + e] = l[j];
    l[j] = e >= p.E || l[j] != l[j] ? -INFINITY : l[j];  // NaN never wins a slot
  }
  select_topk<NJ>(p, t, lane, l);
}

// split_logits_kernel from this many multiply-adds (T E d).  Both routes in us,
// MI355X, logits and top-k, split / 64-row slices, fp32 router:
//                   bf16 x                                fp32 x
//   E 256, d 7168:  T 128 23 / 25, 200 25 / 30,           128 28 / 26, 200 30 / 31,
//                   512 29 / 51, 4096 58 / 359            512 33 / 51, 4096 95 / 366
//   E 160, d 5120:  T 200 21 / 22, 350 22 / 27            256 24 / 23, 350 26 / 26, 512 27 / 31
//   E 64, d 2048:   T 1024 19 / 21, 2048 24 / 34          1024 21 / 21, 2048 27 / 33
//   E 1000, d 1408: T 100 30 / 33, 200 34 / 39            200 36 / 38
// Short batches have too few tiles to hide a workgroup's steps (three-part x has
// twice as many MFMAs in each); long ones pay the other route for ceil(d / 64)
// partials of every logit, written and read.
constexpr int64_t kSplitMacs = 250000000, kSplitMacsF32 = 400000000;
int64_t split_tokens(const latent_route_args& a) {
  const int64_t per = a.n_expert * a.n_embd, macs = a.x_dtype == LATENT_F32 ? kSplitMacsF32 : kSplitMacs;
  return per > 0 ? (macs + per - 1) / per : 0;
}
bool split_applies(const latent_route_args& a) {
  return a.n_tokens >= split_tokens(a) && a.n_embd % kSStep == 0;
}

int64_t split_tiles(const latent_route_args& a, int64_t tok) {
  return ((a.n_tokens + tok - 1) / tok) * ((a.n_expert + kSExp - 1) / kSExp);
}

// Slices of d (and, for the split kernel, their rows).
int64_t n_slices(const latent_route_args& a, int* slice_rows) {
  const int64_t slices = (a.n_embd + kRows - 1) / kRows;
  if (!split_applies(a)) return slices;
  // About two workgroups per CU, at most kFewSlices slices of whole steps, and
  // no more than the other route's (the workspace callers know).
  const int64_t tiles = split_tiles(a, kSTok);
  const int64_t want = std::max<int64_t>(1, std::min({int64_t{kFewSlices}, slices, 512 / tiles}));
  const int64_t rows = ((a.n_embd + want - 1) / want + kSStep - 1) / kSStep * kSStep;
  if (slice_rows) *slice_rows = static_cast<int>(rows);
  return (a.n_embd + rows - 1) / rows;
}

int validate(const latent_route_args& a) {
  if (a.n_tokens < 0 || a.n_expert <= 0 || a.n_expert_used <= 0) return LATENT_E_INVALID;
  if (a.n_expert_used > a.n_expert) return LATENT_E_INVALID;
  if (a.drop_rule < LATENT_DROP_NONE || a.drop_rule > LATENT_DROP_INCLUSIVE) return LATENT_E_INVALID;
  if (a.drop_rule == LATENT_DROP_INCLUSIVE && !(a.drop_param > 0.f && a.drop_param <= 1.f)) return LATENT_E_INVALID;
  if (!a.logits_in) {
    if (a.n_embd <= 0) return LATENT_E_INVALID;
    if (a.x_dtype < LATENT_F32 || a.x_dtype > LATENT_BF16) return LATENT_E_INVALID;
    if (a.router_dtype != LATENT_F32 && a.router_dtype != LATENT_BF16) return LATENT_E_INVALID;
  }
  if (a.n_expert > kMaxE || a.n_expert_used > kMaxK) return LATENT_E_UNSUPPORTED;
  if (a.n_tokens > (1 << 24) || a.n_embd > (1 << 20)) return LATENT_E_UNSUPPORTED;
  return LATENT_OK;
}

size_t workspace_bytes(const latent_route_args& a) {
  if (a.logits_in) return 0;
  // Partial rows: ceil(d / 64) a token, fewer for the split kernel's batches.  A
  // workspace sized for a batch also serves every smaller one: the split
  // kernel's slices x tokens are bounded by an expression that grows with the
  // tokens, and a batch just below its range needs ceil(d / 64) rows a token.
  const int64_t slices = (a.n_embd + kRows - 1) / kRows;
  if (a.n_embd % kSStep != 0) return static_cast<size_t>(slices * a.n_tokens) * a.n_expert * sizeof(float);
  int64_t rows = slices * std::min(a.n_tokens, split_tokens(a) - 1);
  if (split_applies(a)) {
    const int64_t neb = (a.n_expert + kSExp - 1) / kSExp;
    rows = std::max(rows, std::min(kFewSlices * a.n_tokens, std::max(a.n_tokens, 512 * kSTok / neb)));
    rows = std::min(rows, slices * a.n_tokens);
  }
  return static_cast<size_t>(rows) * a.n_expert * sizeof(float);
}

}  // namespace
}  // namespace route
}  // namespace latent

using namespace latent;

extern "C" int latent_route_workspace_size(const latent_route_args* args, size_t* bytes) {
  if (!args || !bytes) return LATENT_E_INVALID;
  const int st = route::validate(*args);
  if (st != LATENT_OK) return st;
  *bytes = route::workspace_bytes(*args);
  return LATENT_OK;
}

extern "C" int latent_route(const latent_route_args* args, latent_stream_t stream) {
  if (!args) return LATENT_E_INVALID;
  const latent_route_args& a = *args;
  const int st = route::validate(a);
  if (st != LATENT_OK) return st;
  if (a.n_tokens == 0) return LATENT_OK;
  if (!a.ids || !a.weights) return LATENT_E_INVALID;
  if (!a.logits_in && (!a.x || !a.router)) return LATENT_E_INVALID;
  const size_t need = route::workspace_bytes(a);
  if (need && (!a.workspace || a.workspace_bytes < need)) return LATENT_E_WORKSPACE;
  route::Params p{};
  p.x = a.x;
  p.x_dtype = a.x_dtype;
  p.router = a.router;
  p.router_dtype = a.router_dtype;
  p.logits_in = a.logits_in;
  p.logits_out = a.logits_out;
  p.ids = a.ids;
  p.weights = a.weights;
  p.partial = static_cast<float*>(a.workspace);
  p.T = static_cast<int>(a.n_tokens);
  p.d = static_cast<int>(a.n_embd);
  p.E = static_cast<int>(a.n_expert);
  p.K = static_cast<int>(a.n_expert_used);
  const bool split = !a.logits_in && route::split_applies(a);
  p.nslice = a.logits_in ? 0 : static_cast<int>(route::n_slices(a, &p.slice_rows));
  p.drop_rule = a.drop_rule;
  p.drop_param = a.drop_param;
  auto aligned = [](const void* q, int dtype) {
    return (reinterpret_cast<uintptr_t>(q) & (dtype == LATENT_F32 ? 15u : 7u)) == 0;
  };
  p.vec_router = a.router && a.n_expert % 4 == 0 && aligned(a.router, a.router_dtype);
  p.vec_x = a.x && a.n_embd % 4 == 0 && aligned(a.x, a.x_dtype);
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  const dim3 tok(static_cast<unsigned>(a.n_tokens)), block(route::kThreads);
  if (split) {
    const bool wf32 = a.router_dtype == LATENT_F32;
    const bool vec = (reinterpret_cast<uintptr_t>(a.x) & 15u) == 0;  // rows are multiples of 64 bytes
    const int64_t wide = route::split_tiles(a, 2 * route::kSTok) * p.nslice;
    // A workgroup on every CU; three-part x does not fit the LDS twice.
    const bool big = wide >= 256 && a.x_dtype != LATENT_F32;
    auto launch = [&](auto kernel, int tok) {
      hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(big ? wide : route::split_tiles(a, tok) * p.nslice)),
                         dim3(2 * tok), 0, s, p);
    };
    auto pick = [&](auto xt) {
      constexpr int kX = decltype(xt)::value;
      auto tile = [&](auto w, auto v) {
        constexpr bool kW = decltype(w)::value, kV = decltype(v)::value;
        constexpr int kBig = kX == LATENT_F32 ? route::kSTok : 2 * route::kSTok;
        if (big)
          launch(route::split_logits_kernel<kX, kW, kV, kBig>, kBig);
        else
          launch(route::split_logits_kernel<kX, kW, kV, route::kSTok>, route::kSTok);
      };
      if (wf32)
        vec ? tile(std::true_type{}, std::true_type{}) : tile(std::true_type{}, std::false_type{});
      else
        vec ? tile(std::false_type{}, std::true_type{}) : tile(std::false_type{}, std::false_type{});
    };
    if (a.x_dtype == LATENT_F32)
      pick(std::integral_constant<int, LATENT_F32>{});
    else if (a.x_dtype == LATENT_F16)
      pick(std::integral_constant<int, LATENT_F16>{});
    else
      pick(std::integral_constant<int, LATENT_BF16>{});
    if (hipGetLastError() != hipSuccess) return LATENT_E_HIP;
    const dim3 waves(static_cast<unsigned>((a.n_tokens + route::kTopkWaves - 1) / route::kTopkWaves));
    const dim3 wave_block(route::kTopkWaves * kWave);
    if (a.n_expert <= 4 * kWave)
      hipLaunchKernelGGL(route::topk_wave_kernel<4>, waves, wave_block, 0, s, p);
    else
      hipLaunchKernelGGL(route::topk_wave_kernel<route::kPerLane>, waves, wave_block, 0, s, p);
    return hipGetLastError() == hipSuccess ? LATENT_OK : LATENT_E_HIP;
  }
  if (!a.logits_in) {
    const dim3 grid(static_cast<unsigned>((a.n_expert + route::kCols - 1) / route::kCols), static_cast<unsigned>(p.nslice),
                    static_cast<unsigned>((a.n_tokens + route::kTok - 1) / route::kTok));
    hipLaunchKernelGGL(route::logits_kernel, grid, block, 0, s, p);
    if (hipGetLastError() != hipSuccess) return LATENT_E_HIP;
  }
  hipLaunchKernelGGL(route::topk_kernel, tok, block, 0, s, p);
  return hipGetLastError() == hipSuccess ? LATENT_OK : LATENT_E_HIP;
}
