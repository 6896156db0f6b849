// Single-expert LATENT SwiGLU FFN on the factor artifacts exactly as
// loader/latent_loader.py writes them (flat quantization groups).
//
// Replaces swiglu_expert / _load_factor of loader/latent_runtime.py:19-59 for
// one expert: the six factors stay in their packed artifact form on the device
// and are dequantized on the fly.  Unlike the stacked per-row layout of the
// MoE-layer path, an artifact quantizes each factor as one flat row-major
// array: group g covers flat elements [g*G, (g+1)*G) whatever the row length
// (quantize_nf4 / quantize_int8, loader/latent_loader.py:111-158), so groups
// straddle rows whenever cols % G != 0 (odd ranks such as 37 from the
// energy-based rank choice, or INT8 group 64 on any shape).  Element (k, n) of
// a [rows][cols] factor is flat index i = k*cols + n:
//   NF4   code = nibble (i & 1) of byte i >> 1 (low nibble = even index),
//         value = level[code] * f32(scale_f16[i / G])
//   INT8  value = f32(q[i]) * f32(scale_f16[i / G])
// one fp32 multiply each, as dequantize_nf4 / dequantize_int8
// (loader/latent_loader.py:133-145, 161-170) compute it.
//
// The chain (loader/latent_runtime.py:35-59), all fp32:
//   gl = x . A_g, ul = x . A_u            K = d
//   g  = gl . B_g, u = ul . B_u           K = rank
//   dl = (SiLU(g) * u [* w]) . A_d        K = ff   (SwiGLU folded into staging)
//   y  = dl . B_d                         K = rank
// An expert of moderate size (chain_applies) takes three launches, eight
// tokens a workgroup:
//   chain_a   x . [A_g | A_u] over (64-column tile, slice of d)
//   chain_bc  per range of ff: the latents (slices summed in order), g, u, h in
//             LDS, h . A_d
//   chain_d   per 64 columns of d: the down latent (ranges summed in order), y
// Others take one launch of proj_kernel per product, over (256-column tile, K
// slice, 8-token tile), and reduce_kernel where K has several slices.  Every
// sum runs in a fixed order, so results are reproducible call to call.
#include "common.hpp"

#include <algorithm>

namespace latent {
namespace expert {
namespace {

constexpr int kT = 256;      // threads = output columns per workgroup
constexpr int kMT = 8;       // tokens per workgroup
constexpr int kStage = 512;  // K rows of activations staged in LDS at a time
constexpr int kTargetBlocks = 2048;
constexpr int kMinKSlice = 64;

struct Flat {
  const uint8_t* data;
  const uint16_t* scales;
  int kind;    // LATENT_Q_NF4 | LATENT_Q_INT8
  int gshift;  // log2(group size)
};

struct Proj {
  Flat f;
  const float* act;   // [T][K] (the gate product g for the SwiGLU prologue)
  const float* act2;  // [T][K] the up product u (SwiGLU prologue only)
  float wmul;         // router weight applied before A_d (1 otherwise)
  float* dst;         // [S][T][N] partials, or the result when S == 1
  int T, K, N, ks;    // ks: K rows per slice
};

__device__ __forceinline__ float silu(float g) { return g / (1.0f + expf(-g)); }

template <bool kSwiGLU>
__global__ void __launch_bounds__(kT) proj_kernel(Proj p) {
  __shared__ float act[kMT][kStage];
  __shared__ float lv[16];
  const int tid = threadIdx.x;
  const int n = blockIdx.x * kT + tid;
  const int s = blockIdx.y;
  const int t0 = blockIdx.z * kMT;
  const int mt = min(kMT, p.T - t0);
  const int k0 = s * p.ks, k1 = min(p.K, k0 + p.ks);
  if (tid < 16) lv[tid] = nf4_level(tid);
  float acc[kMT];
#pragma unroll
  for (int t = 0; t < kMT; ++t) acc[t] = 0.f;
  int64_t idx = static_cast<int64_t>(k0) * p.N + n;
  for (int kc = k0; kc < k1; kc += kStage) {
    const int kn = min(kStage, k1 - kc);
    __syncthreads();  // the previous chunk's readers are done
    for (int i = tid; i < kMT * kStage; i += kT) {
      const int t = i / kStage, k = i - t * kStage;
      float v = 0.f;
      if (t < mt && k < kn) {
        const int64_t o = static_cast<int64_t>(t0 + t) * p.K + kc + k;
        v = p.act[o];
        if (kSwiGLU) v = silu(v) * p.act2[o] * p.wmul;
      }
      act[t][k] = v;
    }
    __syncthreads();
    if (n < p.N) {
      for (int k = 0; k < kn; ++k, idx += p.N) {
        const float sc = half_bits_to_float(p.f.scales[idx >> p.f.gshift]);
        float w;
        if (p.f.kind == LATENT_Q_NF4) {
          const uint32_t b = p.f.data[idx >> 1];
          w = __fmul_rn(lv[(idx & 1) ? (b >> 4) : (b & 15u)], sc);
        } else {
          w = __fmul_rn(static_cast<float>(reinterpret_cast<const int8_t*>(p.f.data)[idx]), sc);
        }
#pragma unroll
        for (int t = 0; t < kMT; ++t) acc[t] = fmaf(act[t][k], w, acc[t]);
      }
    }
  }
  if (n >= p.N) return;
  for (int t = 0; t < mt; ++t) p.dst[(static_cast<int64_t>(s) * p.T + t0 + t) * p.N + n] = acc[t];
}

// dst[t][n] = sum over slices s (in order) of part[s][t][n].
__global__ void __launch_bounds__(kT) reduce_kernel(const float* part, float* dst, int64_t tn, int S) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(kT) + threadIdx.x; i < tn; i += static_cast<int64_t>(gridDim.x) * kT) {
    float v = 0.f;
    for (int s = 0; s < S; ++s) v += part[s * tn + i];
    dst[i] = v;
  }
}

// ---- the three-launch chain -----------------------------------------------------
// Bound by latency: at d 512, ff 1408, rank 64 the six products and three sums
// took nine launches of 15-19 us and 5 us, each thread walking its rows one
// dependent element at a time.  Here a thread has 8 to 32 elements with eight
// rows' loads in flight, and the waves of a workgroup share K.
constexpr int kC = 64;        // columns per tile: one per lane
constexpr int kWaves = kT / kWave;
constexpr int kBT = 512, kBWaves = kBT / kWave;  // chain_bc: two products and their sums in one workgroup
constexpr int kMaxSlices = 16, kMaxRanges = 32;
constexpr int kRangeBlocks = 2048;  // chain_bc workgroups beyond which ranges only repeat the latents' sums
constexpr int kChainRank = 256, kChainD = 2048, kChainFf = 4096;
static_assert(kMT == 8 && kC == kWave, "activation rows of two float4, one column per lane");

struct Chain {
  Flat f[6];     // gate_a, up_a, gate_b, up_b, down_a, down_b
  const float* x;
  float* part_a;  // [n_slice][T][rg + ru]
  float* part_c;  // [n_range][T][rd]
  float* out;
  float wmul;
  int T, d, ff, rg, ru, rd;
  int ks, n_slice;   // rows of d per slice
  int sub, n_range;  // 64-column tiles of ff per range
};

// acc[t] += act[k][t] W[k][n] over rows [k0, k1) (act rows from row base).
__device__ __forceinline__ void gemv_rows(const Flat& f, int N, int n, int base, int k0, int k1, const float* act,
                                          const float* lv, float (&acc)[kMT]) {
  for (int k = k0; k < k1; k += 8) {
    uint32_t b[8];
    uint16_t sc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t idx = static_cast<int64_t>(min(k + i, k1 - 1)) * N + n;
      b[i] = f.kind == LATENT_Q_NF4 ? static_cast<uint32_t>(f.data[idx >> 1]) >> (4 * (idx & 1))
                                    : static_cast<uint32_t>(f.data[idx]);
      sc[i] = f.scales[idx >> f.gshift];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (k + i >= k1) break;
      const float v = f.kind == LATENT_Q_NF4 ? lv[b[i] & 15u] : static_cast<float>(static_cast<int8_t>(b[i]));
      const float w = __fmul_rn(v, half_bits_to_float(sc[i]));
      const float4* a = reinterpret_cast<const float4*>(act + (k + i - base) * kMT);
      const float4 a0 = a[0], a1 = a[1];
      acc[0] = fmaf(a0.x, w, acc[0]);
      acc[1] = fmaf(a0.y, w, acc[1]);
      acc[2] = fmaf(a0.z, w, acc[2]);
      acc[3] = fmaf(a0.w, w, acc[3]);
      acc[4] = fmaf(a1.x, w, acc[4]);
      acc[5] = fmaf(a1.y, w, acc[5]);
      acc[6] = fmaf(a1.z, w, acc[6]);
      acc[7] = fmaf(a1.w, w, acc[7]);
    }
  }
}

// One wave's share: rows [k0, k1) of W, column n (lanes past N sit out), into
// the wave's slot of red.
__device__ __forceinline__ void wave_rows(const Flat& f, int N, int n, int base, int k0, int k1, const float* act,
                                          const float* lv, float (*red)[kC]) {
  float acc[kMT];
#pragma unroll
  for (int t = 0; t < kMT; ++t) acc[t] = 0.f;
  if (n < N) gemv_rows(f, N, n, base, k0, k1, act, lv, acc);
#pragma unroll
  for (int t = 0; t < kMT; ++t) red[t][threadIdx.x & (kWave - 1)] = acc[t];
}

__global__ void __launch_bounds__(kT) chain_a(Chain p) {
  __shared__ __attribute__((aligned(16))) float act[kChainD / kMaxSlices * kMT];
  __shared__ float red[kWaves][kMT][kC];
  __shared__ float lv[16];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
  const int tg = (p.rg + kC - 1) / kC, up = static_cast<int>(blockIdx.x) >= tg;
  const int N = up ? p.ru : p.rg, n0 = (blockIdx.x - (up ? tg : 0)) * kC;
  const int s = blockIdx.y, t0 = blockIdx.z * kMT, mt = min(kMT, p.T - t0);
  const int k0 = s * p.ks, kn = min(p.ks, p.d - k0);
  if (tid < 16) lv[tid] = nf4_level(tid);
  for (int i = tid; i < kn * kMT; i += kT) {
    const int t = i / kn, k = i - t * kn;
    act[k * kMT + t] = t < mt ? p.x[static_cast<int64_t>(t0 + t) * p.d + k0 + k] : 0.f;
  }
  __syncthreads();
  wave_rows(p.f[up], N, n0 + lane, k0, k0 + wave * kn / kWaves, k0 + (wave + 1) * kn / kWaves, act, lv, red[wave]);
  __syncthreads();
  for (int i = tid; i < mt * kC; i += kT) {
    const int t = i / kC, n = i - t * kC;
    if (n0 + n < N)
      p.part_a[(static_cast<int64_t>(s) * p.T + t0 + t) * (p.rg + p.ru) + (up ? p.rg : 0) + n0 + n] =
          (red[0][t][n] + red[1][t][n]) + (red[2][t][n] + red[3][t][n]);
  }
}

// lat[c][t] = sum over n partials of [.][T][W] at (token t, column c), in
// order, sixteen loads in flight.
template <int kThreads>
__device__ __forceinline__ void sum_latents(const float* part, int n, int T, int W, int t0, int mt, float* lat) {
  const int64_t step = static_cast<int64_t>(T) * W;
  for (int i = threadIdx.x; i < W * kMT; i += kThreads) {
    const int t = i / W, c = i - t * W;
    float v = 0.f;
    if (t < mt) {
      const float* src = part + static_cast<int64_t>(t0 + t) * W + c;
      for (int s = 0; s < n; s += 16) {
        float l[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) l[j] = src[min(s + j, n - 1) * step];
#pragma unroll
        for (int j = 0; j < 16; ++j) v += s + j < n ? l[j] : 0.f;
      }
    }
    lat[c * kMT + t] = v;
  }
}

__global__ void __launch_bounds__(kBT) chain_bc(Chain p) {
  __shared__ __attribute__((aligned(16))) float lat[2 * kChainRank * kMT];
  __shared__ float dacc[kMT][kChainRank];
  __shared__ float red[kBWaves][kMT][kC];
  __shared__ __attribute__((aligned(16))) float hs[kC * kMT];
  __shared__ float lv[16];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
  const int t0 = blockIdx.z * kMT, mt = min(kMT, p.T - t0);
  if (tid < 16) lv[tid] = nf4_level(tid);
  sum_latents<kBT>(p.part_a, p.n_slice, p.T, p.rg + p.ru, t0, mt, lat);
  for (int i = tid; i < kMT * kChainRank; i += kBT) dacc[i / kChainRank][i % kChainRank] = 0.f;
  __syncthreads();
  const int up = wave & 1, share = wave >> 1, rk = up ? p.ru : p.rg;
  const int c_end = min(p.ff, static_cast<int>(blockIdx.x + 1) * p.sub * kC);
  for (int c0 = blockIdx.x * p.sub * kC; c0 < c_end; c0 += kC) {
    const int nc = min(kC, c_end - c0);
    // Waves: (gate, up) x quarters of the rank.
    wave_rows(p.f[2 + up], p.ff, c0 + lane, 0, share * rk / 4, (share + 1) * rk / 4, lat + (up ? p.rg * kMT : 0), lv,
              red[wave]);
    __syncthreads();
    for (int i = tid; i < kMT * kC; i += kBT) {
      const int t = i / kC, n = i - t * kC;
      const float g = (red[0][t][n] + red[2][t][n]) + (red[4][t][n] + red[6][t][n]);
      const float u = (red[1][t][n] + red[3][t][n]) + (red[5][t][n] + red[7][t][n]);
      hs[n * kMT + t] = silu(g) * u * p.wmul;
    }
    __syncthreads();
    for (int n0 = 0; n0 < p.rd; n0 += kC) {
      wave_rows(p.f[4], p.rd, n0 + lane, c0, c0 + wave * nc / kBWaves, c0 + (wave + 1) * nc / kBWaves, hs, lv, red[wave]);
      __syncthreads();
      for (int i = tid; i < kMT * kC; i += kBT) {
        const int t = i / kC, n = i - t * kC;
        if (n0 + n < p.rd) dacc[t][n0 + n] += ((red[0][t][n] + red[1][t][n]) + (red[2][t][n] + red[3][t][n])) +
                                           ((red[4][t][n] + red[5][t][n]) + (red[6][t][n] + red[7][t][n]));
      }
      __syncthreads();
    }
  }
  for (int i = tid; i < mt * p.rd; i += kBT) {
    const int t = i / p.rd, n = i - t * p.rd;
    p.part_c[(static_cast<int64_t>(blockIdx.x) * p.T + t0 + t) * p.rd + n] = dacc[t][n];
  }
}

__global__ void __launch_bounds__(kT) chain_d(Chain p) {
  __shared__ __attribute__((aligned(16))) float lat[kChainRank * kMT];
  __shared__ float red[kWaves][kMT][kC];
  __shared__ float lv[16];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid >> 6;
  const int n0 = blockIdx.x * kC, t0 = blockIdx.z * kMT, mt = min(kMT, p.T - t0);
  if (tid < 16) lv[tid] = nf4_level(tid);
  sum_latents<kT>(p.part_c, p.n_range, p.T, p.rd, t0, mt, lat);
  __syncthreads();
  wave_rows(p.f[5], p.d, n0 + lane, 0, wave * p.rd / kWaves, (wave + 1) * p.rd / kWaves, lat, lv, red[wave]);
  __syncthreads();
  for (int i = tid; i < mt * kC; i += kT) {
    const int t = i / kC, n = i - t * kC;
    if (n0 + n < p.d)
      p.out[static_cast<int64_t>(t0 + t) * p.d + n0 + n] =
          (red[0][t][n] + red[1][t][n]) + (red[2][t][n] + red[3][t][n]);
  }
}

struct Plan {
  int S, ks;
};

Plan plan_for(int64_t T, int64_t K, int64_t N) {
  const int64_t tiles = ((N + kT - 1) / kT) * ((T + kMT - 1) / kMT);
  int64_t S = std::max<int64_t>(1, (kTargetBlocks + tiles - 1) / tiles);
  S = std::min<int64_t>(S, std::max<int64_t>(1, K / kMinKSlice));
  S = std::min<int64_t>(S, 65535);
  const int64_t ks = (K + S - 1) / S;
  return {static_cast<int>((K + ks - 1) / ks), static_cast<int>(ks)};
}

int group_shift(int g) {
  if (g < 2 || (g & (g - 1))) return -1;
  int s = 0;
  while ((1 << s) < g) ++s;
  return s;
}

int check(const latent_flat_factor& f, int64_t rows, int64_t cols) {
  if (!f.data || !f.scales) return LATENT_E_INVALID;
  if (f.kind != LATENT_Q_NF4 && f.kind != LATENT_Q_INT8) return LATENT_E_INVALID;
  if (f.rows != rows || f.cols != cols || rows <= 0 || cols <= 0) return LATENT_E_INVALID;
  if (group_shift(f.group_size) < 0) return LATENT_E_UNSUPPORTED;  // power-of-two groups only
  if (rows > (1 << 24) || cols > (1 << 24) || rows * cols > (int64_t{1} << 40)) return LATENT_E_UNSUPPORTED;
  return LATENT_OK;
}

struct Dims {
  int64_t T, d, rg, ru, rd, ff;
};

int validate(const latent_expert_args& a, Dims& m) {
  m.T = a.n_tokens;
  m.d = a.gate_a.rows;
  m.rg = a.gate_a.cols;
  m.ff = a.gate_b.cols;
  m.ru = a.up_a.cols;
  m.rd = a.down_a.cols;
  if (m.T < 0 || m.T > (1 << 24)) return LATENT_E_INVALID;
  const struct {
    const latent_flat_factor* f;
    int64_t rows, cols;
  } want[6] = {{&a.gate_a, m.d, m.rg}, {&a.gate_b, m.rg, m.ff}, {&a.up_a, m.d, m.ru},
               {&a.up_b, m.ru, m.ff},   {&a.down_a, m.ff, m.rd}, {&a.down_b, m.rd, m.d}};
  for (const auto& w : want) {
    const int st = check(*w.f, w.rows, w.cols);
    if (st != LATENT_OK) return st;
  }
  return LATENT_OK;
}

size_t al(size_t v) { return (v + 255) / 256 * 256; }

struct Layout {
  size_t gl, ul, g, u, dl, part, part_a, part_c, total;
};

// The split of a chain.  chain_bc's workgroups each sum all slices' latents, so
// ranges of ff beyond what fills the chip only repeat that: d 2048, ff 4096, rank
// 256, 4096 tokens 2,356 us at 32 ranges, 2,119 at four (and 256 -> 144 MiB).
void chain_split(const Dims& m, Chain& c) {
  c.ks = static_cast<int>(std::max<int64_t>(32, (m.d + kMaxSlices - 1) / kMaxSlices));
  c.n_slice = static_cast<int>((m.d + c.ks - 1) / c.ks);
  const int64_t tiles = (m.ff + kC - 1) / kC, token_tiles = std::max<int64_t>(1, (m.T + kMT - 1) / kMT);
  const int64_t ranges = std::max<int64_t>(1, std::min<int64_t>(kMaxRanges, kRangeBlocks / token_tiles));
  c.sub = static_cast<int>((tiles + ranges - 1) / ranges);
  c.n_range = static_cast<int>((tiles + c.sub - 1) / c.sub);
}

// Experts whose latents fit the chain's LDS and whose factors do not want more
// than 16 slices of d and 32 ranges of ff.  Many tokens at a high rank keep a
// launch per product: their latents (n_slice x ranks a token) are most of the
// traffic.  Us, chain / products: d 2048, ff 4096, rank 256: 768 tokens 440 /
// 559, 1024 596 / 545, 4096 2,119 / 1,807; d 512, ff 4096, rank 256: 1024 462 /
// 451, 4096 1,612 / 1,363; d 2048, ff 4096, rank 192: 1024 308 / 421, 16,384
// 4,387 / 5,688; d 512, ff 1408, rank 64: 4 21 / 119, 16,384 706 / 1,010.
bool chain_applies(const Dims& m) {
  if (std::max({m.rg, m.ru, m.rd}) > kChainRank || m.d > kChainD || m.ff > kChainFf || m.T > 65535 * kMT) return false;
  Chain c{};
  chain_split(m, c);
  return m.T < 1024 || c.n_slice * (m.rg + m.ru) <= 16 * 2 * 192;
}

size_t part_floats(const Dims& m, int64_t K, int64_t N) {
  const Plan pl = plan_for(m.T, K, N);
  return pl.S > 1 ? static_cast<size_t>(pl.S) * m.T * N : 0;
}

Layout layout_for(const Dims& m) {
  Layout L{};
  size_t off = 0;
  if (chain_applies(m)) {
    Chain c{};
    chain_split(m, c);
    L.part_a = off; off = al(off + static_cast<size_t>(c.n_slice) * m.T * (m.rg + m.ru) * 4);
    L.part_c = off; off = al(off + static_cast<size_t>(c.n_range) * m.T * m.rd * 4);
    L.total = std::max<size_t>(off, 256);
    return L;
  }
  L.gl = off; off = al(off + m.T * m.rg * 4);
  L.ul = off; off = al(off + m.T * m.ru * 4);
  L.g = off;  off = al(off + m.T * m.ff * 4);
  L.u = off;  off = al(off + m.T * m.ff * 4);
  L.dl = off; off = al(off + m.T * m.rd * 4);
  size_t part = 0;
  part = std::max(part, part_floats(m, m.d, m.rg));
  part = std::max(part, part_floats(m, m.d, m.ru));
  part = std::max(part, part_floats(m, m.rg, m.ff));
  part = std::max(part, part_floats(m, m.ru, m.ff));
  part = std::max(part, part_floats(m, m.ff, m.rd));
  part = std::max(part, part_floats(m, m.rd, m.d));
  L.part = off; off = al(off + part * 4);
  L.total = std::max<size_t>(off, 256);
  return L;
}

Flat flat(const latent_flat_factor& f) {
  return {static_cast<const uint8_t*>(f.data), f.scales, f.kind, group_shift(f.group_size)};
}

// dst[T][N] = act[T][K] . W[K][N] (SwiGLU prologue: act = SiLU(act) * act2 * w).
int project(const Dims& m, const latent_flat_factor& f, const float* act, const float* act2, float wmul, bool swiglu,
            float* dst, float* part, hipStream_t s) {
  const int64_t K = f.rows, N = f.cols;
  const Plan pl = plan_for(m.T, K, N);
  Proj p{};
  p.f = flat(f);
  p.act = act;
  p.act2 = act2;
  p.wmul = wmul;
  p.dst = pl.S > 1 ? part : dst;
  p.T = static_cast<int>(m.T);
  p.K = static_cast<int>(K);
  p.N = static_cast<int>(N);
  p.ks = pl.ks;
  const dim3 grid(static_cast<unsigned>((N + kT - 1) / kT), static_cast<unsigned>(pl.S),
                  static_cast<unsigned>((m.T + kMT - 1) / kMT));
  if (grid.z > 65535) return LATENT_E_UNSUPPORTED;
  if (swiglu)
    hipLaunchKernelGGL(proj_kernel<true>, grid, dim3(kT), 0, s, p);
  else
    hipLaunchKernelGGL(proj_kernel<false>, grid, dim3(kT), 0, s, p);
  if (hipGetLastError() != hipSuccess) return LATENT_E_HIP;
  if (pl.S > 1) {
    const int64_t tn = m.T * N;
    const unsigned blocks = static_cast<unsigned>(std::min<int64_t>(4096, (tn + kT - 1) / kT));
    hipLaunchKernelGGL(reduce_kernel, dim3(blocks), dim3(kT), 0, s, part, dst, tn, pl.S);
    if (hipGetLastError() != hipSuccess) return LATENT_E_HIP;
  }
  return LATENT_OK;
}

}  // namespace
}  // namespace expert
}  // namespace latent

using namespace latent;

extern "C" int latent_expert_workspace_size(const latent_expert_args* args, size_t* bytes) {
  if (!args || !bytes) return LATENT_E_INVALID;
  expert::Dims m;
  const int st = expert::validate(*args, m);
  if (st != LATENT_OK) return st;
  *bytes = expert::layout_for(m).total;
  return LATENT_OK;
}

extern "C" int latent_expert_forward(const latent_expert_args* args, latent_stream_t stream) {
  if (!args) return LATENT_E_INVALID;
  const latent_expert_args& a = *args;
  expert::Dims m;
  int st = expert::validate(a, m);
  if (st != LATENT_OK) return st;
  if (m.T == 0) return LATENT_OK;
  if (!a.x || !a.out) return LATENT_E_INVALID;
  const expert::Layout L = expert::layout_for(m);
  if (!a.workspace || a.workspace_bytes < L.total) return LATENT_E_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(a.workspace) & 255u) return LATENT_E_WORKSPACE;
  const hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  (void)hipGetLastError();
  char* ws = static_cast<char*>(a.workspace);
  float* gl = reinterpret_cast<float*>(ws + L.gl);
  float* ul = reinterpret_cast<float*>(ws + L.ul);
  float* g = reinterpret_cast<float*>(ws + L.g);
  float* u = reinterpret_cast<float*>(ws + L.u);
  float* dl = reinterpret_cast<float*>(ws + L.dl);
  float* part = reinterpret_cast<float*>(ws + L.part);
  const float w = a.weight_before_down ? a.weight : 1.0f;
  if (expert::chain_applies(m)) {
    expert::Chain c{};
    expert::chain_split(m, c);
    const latent_flat_factor* fs[6] = {&a.gate_a, &a.up_a, &a.gate_b, &a.up_b, &a.down_a, &a.down_b};
    for (int i = 0; i < 6; ++i) c.f[i] = expert::flat(*fs[i]);
    c.x = a.x;
    c.part_a = reinterpret_cast<float*>(ws + L.part_a);
    c.part_c = reinterpret_cast<float*>(ws + L.part_c);
    c.out = a.out;
    c.wmul = w;
    c.T = static_cast<int>(m.T);
    c.d = static_cast<int>(m.d);
    c.ff = static_cast<int>(m.ff);
    c.rg = static_cast<int>(m.rg);
    c.ru = static_cast<int>(m.ru);
    c.rd = static_cast<int>(m.rd);
    const unsigned z = static_cast<unsigned>((m.T + expert::kMT - 1) / expert::kMT);
    auto tiles = [](int64_t n) { return static_cast<unsigned>((n + expert::kC - 1) / expert::kC); };
    hipLaunchKernelGGL(expert::chain_a, dim3(tiles(m.rg) + tiles(m.ru), c.n_slice, z), dim3(expert::kT), 0, s, c);
    hipLaunchKernelGGL(expert::chain_bc, dim3(c.n_range, 1, z), dim3(expert::kBT), 0, s, c);
    hipLaunchKernelGGL(expert::chain_d, dim3(tiles(m.d), 1, z), dim3(expert::kT), 0, s, c);
    return hipGetLastError() == hipSuccess ? LATENT_OK : LATENT_E_HIP;
  }
  if ((st = expert::project(m, a.gate_a, a.x, nullptr, 1.f, false, gl, part, s)) != LATENT_OK) return st;
  if ((st = expert::project(m, a.up_a, a.x, nullptr, 1.f, false, ul, part, s)) != LATENT_OK) return st;
  if ((st = expert::project(m, a.gate_b, gl, nullptr, 1.f, false, g, part, s)) != LATENT_OK) return st;
  if ((st = expert::project(m, a.up_b, ul, nullptr, 1.f, false, u, part, s)) != LATENT_OK) return st;
  if ((st = expert::project(m, a.down_a, g, u, w, true, dl, part, s)) != LATENT_OK) return st;
  return expert::project(m, a.down_b, dl, nullptr, 1.f, false, a.out, part, s);
}
