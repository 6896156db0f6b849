// MoE-layer LATENT expert FFN over the row layout with fp16 MFMA.
//
// The three phases of the multi-kernel path (moe.hip) for layers held in the
// row layout -- per-expert ranks up to 512, INT8 groups allowed -- with the
// products on v_mfma_f32_16x16x32_f16 instead of fp32 FMAs:
//   A   xh . A_g | A_u -> gu     items (expert, factor, range of d rows)
//   BC  g . B_g, u . B_u -> h = SiLU(g) u (in LDS); h . A_d -> dl
//                                items (expert, 256 columns of ff)
//   D   dl . B_d -> out          items (expert, 512 columns of d)
// Replaces, like moe.hip, the per-(token, slot) chain of
// kernels/latent_fused_expert_ffn.cu:27-108 for the routed pairs of each
// active expert; only an expert's true-rank rows and columns are read.
//
// The factors go from HBM to the matrix cores in rowblock.hpp's blocks of 32
// rows: a lane holds eight rows of CPL adjacent columns, and the eight values
// of a column are one operand.  Two rows' nibbles of a column meet in one byte
// (two shifts and two bit selects per eight columns), a byte table in LDS gives
// both levels as fp16, one packed product scales them.  An INT8 group's lanes
// take a zero NF4 scale and add q x scale (one rounding either way).  A lane
// reloads its rows from the next block as it uses them; the INT8 bytes of the
// next block are found through bitmap words loaded one block earlier still.
// No LDS round trip for a factor and no barrier in the loop: decoding chunks
// transposed through LDS, as this file once did, spent two barriers and 64
// scattered LDS stores a thread on every 8 KB.  DeepSeek-V3 shape, ranks 64 to
// 512, 10 % INT8 groups: batch 16 328 -> 219 us, batch 256 751 -> 509 us (198 and
// 484 with what came since).
//
// What bounds it with INT8 groups: the decode's VALU (about 390 instructions a
// block of 32 x 128, half of them for the INT8 bytes, which nearly every wave
// has some of) at three waves per SIMD.  Items of one expert are as long as its
// rank; the prep kernel lists the experts longest first and phase A cuts an
// expert's rows into pieces in proportion to its rank, which took batch 16 from
// 258 to 221 us (a late rank-512 item ran on alone).
//
// Activations (x rows, latents, h) enter the MFMA as fp16 rows scaled by a
// power of two per row (the row maximum into [2^14, 2^15)); products are
// scaled back in fp32 and summed into the fp32 accumulators of the
// multi-kernel path with atomics (gu, dl; out for the reduced output), which
// its prep kernel zeroes.  A pass takes MB blocks of 16 pairs of one expert;
// an expert with more pairs takes several passes.
//
// Ordered calls (row-layout prefill) repeat bit for bit: a range of d (phase
// A) or of ff (BC) stores its sums to a plane of its own, sum_planes_kernel
// adds the planes in order, and the reduced output comes from y rows.  E 64, d
// 2048, ff 1408, rank 128, 1999 tokens: 226 us with atomics, 224 so.
#include "common.hpp"
#include "rowblock.hpp"
#include "rows.hpp"

#include <algorithm>

namespace latent {
namespace rows {
namespace {

using namespace rowblock;

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

enum { F_GATE_A = 0, F_GATE_B, F_UP_A, F_UP_B, F_DOWN_A, F_DOWN_B };

constexpr int kT = 256;            // threads per workgroup (4 waves)
constexpr int kCB = 256;           // BC: ff columns per item
constexpr int kCD = 512;           // D: d columns per item
constexpr int kHStr = kCB + 8;     // halves per h row
constexpr int kTileStr = 128 + 4;  // floats per row of a wave's products
constexpr int kHalfSlot = 8 * kTileStr * 4;  // LDS bytes of eight rows of them
constexpr int kRedBytes = 4 * kHalfSlot;     // of every wave
constexpr int kCopies = 16;               // of the level table, by lane
constexpr int kLutBytes = 256 * kCopies * 4;
constexpr int kMetaSlot = 256 + 256;         // a block's scales [group][row]; its INT8 words, then offsets
constexpr int kMetaBytes = 2 * kMetaSlot;    // per wave
constexpr int kFixBytes = kLutBytes + 4 * kMetaBytes;  // the table, then the waves' meta slots

__device__ __forceinline__ int rank_of(const Params& p, int e, int kind) {
  if (!p.ranks) return p.R;
  const int r = p.ranks[e * 3 + kind];
  return r < 0 ? 0 : (r > p.R ? p.R : r);
}

// Workgroup b -> (active expert a, item i): an expert's items on one XCD
// (workgroups go to the 8 XCDs round robin), so its activations stay in one L2.
__device__ __forceinline__ bool map_item(int b, int n_items, int n_active, int& a, int& i) {
  const int x = b & 7, j = b >> 3;
  a = x + 8 * (j / n_items);
  i = j - (j / n_items) * n_items;
  return a < n_active;
}

// Level-pair table: entry b = (level(b & 15), level(b >> 4)) as two fp16, in
// kCopies copies so that a wave's random lookups spread over the banks.
__device__ __forceinline__ void lut_fill(uint32_t lut, int tid) {
  const half2v lv = {static_cast<_Float16>(nf4_level(tid & 15)), static_cast<_Float16>(nf4_level(tid >> 4))};
  const uint32_t v = __builtin_bit_cast(uint32_t, lv);
#pragma unroll
  for (int i = 0; i < kCopies / 4; ++i) lds_st<u32x4>(lut + tid * (kCopies * 4) + i * 16, u32x4{v, v, v, v});
}

// A wave's walk over blocks [b0, b1) of 32 rows from `row0` of a factor and
// 16 CPL columns from col0, times MB blocks of 16 pairs.  start() issues the
// first loads (as early as the caller can), run() does the rest.
// act.load(b) issues the loads of block b's activations, act.get(b, mb) gives
// the lane's eight of pair block mb (zero for rows that do not count).
//
// Per block a lane loads the codes of its eight rows and, for INT8 factors,
// the bytes of its flagged rows; the scales, bitmap words and word offsets,
// which lanes share, are loaded once per wave, two blocks ahead, and go
// through wave-private LDS slots (a lane then reads its eight rows' scales as
// one 16-byte word): loading them per lane and row made two thirds of all
// load instructions.
template <int CPL, int MB, bool kInt8, class Act>
struct Walk {
  static constexpr int kG = CPL / 4;  // groups a lane loads the scale of
  static constexpr int kQ = kInt8 ? CPL / 4 : 1;
  int row0, b0, b1, lane;
  uint32_t meta;  // LDS address of the wave's meta slots
  Src<CPL> src;
  __amdgpu_buffer_rsrc_t rb, ro, rd;  // INT8 bitmap words, word offsets, bytes
  uint32_t vm, vw, bit, byte, gsc;
  int wstride;
  Act act;
  uint32_t c[8];  // codes of the block
  uint32_t q[kInt8 ? 8 : 1][kQ];  // its INT8 bytes
  uint32_t flags;                 // bit i: row i is INT8
  uint32_t msc[kG], mw, mo;       // meta of the block after the next
  __device__ __forceinline__ Walk(const Factor& f, int e, int col0, int row0_, int b0_, int b1_, int lane_,
                                  uint32_t meta_, const Act& act_)
      : row0(row0_), b0(b0_), b1(b1_), lane(lane_), meta(meta_), src(make_src<CPL>(f, e, col0, lane_)), act(act_),
        flags(0u) {
    // Scales: lane -> row lane / 2, half lane & 1 of the tile's groups (groups
    // past the factor's last belong to columns that are not stored).
    const int g0 = col0 / kGroup;
    vm = static_cast<uint32_t>((lane >> 1) * src.ss + (g0 + (lane & 1) * kG) * 2);
    gsc = static_cast<uint32_t>(src.group - g0) * 64u + static_cast<uint32_t>(lane >> 4) * 16u;
    if (kInt8) {
      const int words = f.words();
      const int64_t er = static_cast<int64_t>(e) * f.rows * words;
      const bool has = f.ext.bitmap != nullptr;
      const uint32_t bytes = has ? static_cast<uint32_t>(f.rows) * words * 4u : 0u;
      rb = buffer_rsrc(has ? f.ext.bitmap + er : nullptr, bytes);
      ro = buffer_rsrc(has ? f.ext.word_offset + er : nullptr, bytes);
      rd = buffer_rsrc(f.ext.data, has ? 0x7FFFFFF0u : 0u);
      wstride = words * 4;
      vw = static_cast<uint32_t>((lane & 31) * wstride + (g0 >> 5) * 4);
      bit = 1u << (src.group & 31);
      byte = static_cast<uint32_t>(min(col0 + CPL * (lane & 15), static_cast<int>(f.cols) - CPL) % kGroup);
    }
  }
  __device__ __forceinline__ int row_of(int b) const { return row0 + 32 * max(0, min(b, b1 - 1)); }  // the same loads on every path
  __device__ __forceinline__ void load_codes(int row, int h) {
    const int oc = row * src.cs;
#pragma unroll
    for (int i = 2 * h; i < 2 * h + 2; ++i) {
      if (CPL == 8)
        c[i] = __builtin_amdgcn_raw_buffer_load_b32(src.rc, src.vc, oc + i * src.cs, 0);
      else
        c[i] = __builtin_amdgcn_raw_buffer_load_b16(src.rc, src.vc, oc + i * src.cs, 0);
    }
  }
  __device__ __forceinline__ void load_meta(int row) {
#pragma unroll
    for (int j = 0; j < kG; ++j) msc[j] = __builtin_amdgcn_raw_buffer_load_b16(src.rs, vm + 2 * j, row * src.ss, 0);
    if (kInt8) {
      mw = __builtin_amdgcn_raw_buffer_load_b32(rb, vw, row * wstride, 0);
      mo = __builtin_amdgcn_raw_buffer_load_b32(ro, vw, row * wstride, 0);
    }
  }
  // Slot of block b: scales [group][row], then 32 words, 32 offsets.
  __device__ __forceinline__ void store_meta(int b) {
    const uint32_t slot = meta + static_cast<uint32_t>(b & 1) * kMetaSlot;
#pragma unroll
    for (int j = 0; j < kG; ++j)
      lds_st<uint16_t>(slot + static_cast<uint32_t>(((lane & 1) * kG + j) * 64 + (lane >> 1) * 2),
                       static_cast<uint16_t>(msc[j]));
    if (kInt8) lds_st<uint32_t>(slot + 256u + 4u * lane, lane < 32 ? mw : mo);
    __builtin_amdgcn_wave_barrier();
  }
  // The INT8 bytes of rows 2 h, 2 h + 1 of block b (its meta stored); an NF4
  // row reads past the range and gets zeros.
  __device__ __forceinline__ void load_int8(int b, int h, uint32_t& fl) {
    if (!kInt8) return;
    const uint32_t at = meta + static_cast<uint32_t>(b & 1) * kMetaSlot + 256u + 32u * (lane >> 4) + 8u * h;
    const u32x2 w = lds_ld<u32x2>(at), o = lds_ld<u32x2>(at + 128u);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = kInt8 ? 2 * h + j : 0;
      const bool is8 = (w[j] & bit) != 0u;
      const uint32_t off = is8 ? (o[j] + popc(w[j] & (bit - 1u))) * kGroup + byte : 0x80000000u;
      fl |= is8 ? 1u << (2 * h + j) : 0u;
      if (CPL == 8) {
        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rd, off, 0, 0));
#pragma unroll
        for (int t = 0; t < kQ; ++t) q[i][t] = v[t & 1];
      } else {
        q[i][0] = __builtin_amdgcn_raw_buffer_load_b32(rd, off, 0, 0);
      }
    }
  }
  __device__ __forceinline__ void start() {
    load_meta(row_of(b0));
    act.load(max(0, min(b0, b1 - 1)));
#pragma unroll
    for (int h = 0; h < 4; ++h) load_codes(row_of(b0), h);
    store_meta(b0);
    load_meta(row_of(b0 + 1));
#pragma unroll
    for (int h = 0; h < 4; ++h) load_int8(b0, h, flags);
  }
  __device__ __forceinline__ void run(uint32_t lut, float4v (&acc)[MB][CPL]) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int j = 0; j < CPL; ++j) acc[mb][j] = float4v{0.f, 0.f, 0.f, 0.f};
    for (int b = b0; b < b1; ++b) {
      store_meta(b + 1);
      load_meta(row_of(b + 2));
      const u32x4 sc = lds_ld<u32x4>(meta + static_cast<uint32_t>(b & 1) * kMetaSlot + gsc);
      half8 a[MB];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) a[mb] = act.get(b, mb);
      act.load(max(0, min(b + 1, b1 - 1)));
      uint32_t fl = 0u;
      // Every level pair of the block first (the scheduling fence keeps the
      // reads together: left alone, the compiler waited for each one).
      uint32_t v[4][CPL];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const uint32_t d0 = c[2 * h], d1 = c[2 * h + 1];
        // Bytes of (row 2h, row 2h + 1) nibbles: even columns, odd columns.
        const uint32_t even = (d0 & 0x0F0F0F0Fu) | ((d1 << 4) & 0xF0F0F0F0u);
        const uint32_t odd = ((d0 >> 4) & 0x0F0F0F0Fu) | (d1 & 0xF0F0F0F0u);
#pragma unroll
        for (int j = 0; j < CPL; ++j)
          v[h][j] = lds_ld<uint32_t>(lut + ((((j & 1) ? odd : even) >> (8 * (j >> 1))) & 0xFFu) * (kCopies * 4));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        half2v s = __builtin_bit_cast(half2v, static_cast<uint32_t>(sc[h])), s8 = {};
        if (kInt8) {
          const uint32_t m = ((flags >> (2 * h)) & 1u ? 0xFFFFu : 0u) | ((flags >> (2 * h)) & 2u ? 0xFFFF0000u : 0u);
          s8 = __builtin_bit_cast(half2v, __builtin_bit_cast(uint32_t, s) & m);
          s = __builtin_bit_cast(half2v, __builtin_bit_cast(uint32_t, s) & ~m);
        }
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
          half2v x = __builtin_bit_cast(half2v, v[h][j]);
          if (kInt8) {
            // q ^ 0x80 under 0x64: 1024 + q + 128 as fp16, exactly.
            const int t = kInt8 ? j >> 2 : 0;
            const uint32_t q0 = q[kInt8 ? 2 * h : 0][t] ^ 0x80808080u;
            const uint32_t q1 = q[kInt8 ? 2 * h + 1 : 0][t] ^ 0x80808080u;
            const uint32_t pr = __builtin_amdgcn_perm(q1, q0, (j & 2) ? 0x07030602u : 0x05010400u);
            const half2v bias = {static_cast<_Float16>(-1152.f), static_cast<_Float16>(-1152.f)};
            const half2v y = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, pr, (j & 1) ? 0x04030402u : 0x04010400u));
            x = __builtin_elementwise_fma(x, s, (y + bias) * s8);  // one of the two is zero
          } else {
            x = x * s;
          }
          v[h][j] = __builtin_bit_cast(uint32_t, x);
        }
        load_codes(row_of(b + 1), h);  // the rows are used: reload them from the next block
        load_int8(b + 1, h, fl);
      }
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        const half8 bv = __builtin_bit_cast(half8, u32x4{v[0][j], v[1][j], v[2][j], v[3][j]});
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          acc[mb][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[mb], bv, acc[mb][j], 0, 0, 0);
      }
      flags = fl;
    }
  }
};

// x rows (fp16, global): the lane's row of each pair block at the item's first
// column + 8 kq.
template <int MB>
struct ActX {
  const _Float16* src[MB];
  half8 r[MB];
  __device__ __forceinline__ void load(int b) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) r[mb] = *reinterpret_cast<const half8*>(src[mb] + 32 * b);
  }
  __device__ __forceinline__ half8 get(int, int mb) const { return r[mb]; }
};
// fp16 rows in LDS, `block` bytes between pair blocks: at = the lane's row of
// the first, column 8 kq.
struct ActLds {
  uint32_t at, block;
  __device__ __forceinline__ void load(int) const {}
  __device__ __forceinline__ half8 get(int b, int mb) const { return lds_ld<half8>(at + mb * block + b * 64); }
};

// f(columns per lane, column tiles) for N columns.
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

// A lane's products of a 16 x 16 CPL tile in LDS (at: its first row, column CPL n).
template <int CPL>
__device__ __forceinline__ void store_tile(uint32_t at, const float4v (&acc)[CPL]) {
#pragma unroll
  for (int v = 0; v < 4; ++v)
#pragma unroll
    for (int c = 0; c < CPL; c += 4)
      lds_st<float4v>(at + static_cast<uint32_t>(v * kTileStr + c) * 4u,
                      float4v{acc[c][v], acc[c + 1][v], acc[c + 2][v], acc[c + 3][v]});
}
// Products of 32 nblk rows (from row0 of the factor) with `cols` columns for
// m pairs, times 2^-exp of their rows, added to (kStore: stored to)
// dst[row][0 .. cols) (rows `stride` floats apart).  The waves share K where
// the columns are fewer than four tiles.  ready(): the level table and the
// activations are in LDS (the first factor loads are issued before it).  red:
// LDS address of kRedBytes the table, the meta slots and the activations may
// overlap.
template <int MB, bool kInt8, bool kStore, class Act, typename Ready>
__device__ __forceinline__ void rank_gemm(const Factor& f, int e, int row0, int nblk, int cols, int m, uint32_t lut,
                                          uint32_t meta, uint32_t red, const int* rexp, const Act& act, Ready&& ready,
                                          float* dst, int stride) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid >> 6);
  const int n = lane & 15, kq = lane >> 4;
  with_columns(cols, [&](auto cpl, auto nt) __attribute__((always_inline)) {
    constexpr int CPL = decltype(cpl)::value, NT = decltype(nt)::value, KP = 4 / NT;
    const int tile = wave % NT, kp = wave / NT;
    Walk<CPL, MB, kInt8, Act> walk(f, e, tile * 16 * CPL, row0, kp * nblk / KP, (kp + 1) * nblk / KP, lane, meta, act);
    walk.start();
    ready();
    float4v acc[MB][CPL];
    walk.run(lut, acc);
    const uint32_t at = red + wave * kHalfSlot + static_cast<uint32_t>((kq & 1) * 4 * kTileStr + n * CPL) * 4u;
#pragma unroll
    for (int half = 0; half < 2 * MB; ++half) {
      if (half * 8 >= m) break;
      lds_barrier();  // every wave is done with the activations, or with the last rows' sums
      if ((kq >> 1) == (half & 1)) store_tile(at, acc[half >> 1]);
      lds_barrier();
      const int rows = min(8, m - half * 8);
      if constexpr (kStore) {
        for (int i = tid; i < rows * cols / 4; i += kT) {
          const int r = i * 4 / cols, c = i * 4 - r * cols, t = c / (16 * CPL);
          const uint32_t src = red + t * kHalfSlot + static_cast<uint32_t>(r * kTileStr + c - t * 16 * CPL) * 4u;
          float* to = dst + static_cast<int64_t>(half * 8 + r) * stride + c;
          const int ex = -rexp[half * 8 + r];
          float4v s = lds_ld<float4v>(src);
#pragma unroll
          for (int k = 1; k < KP; ++k) s += lds_ld<float4v>(src + k * NT * kHalfSlot);
#pragma unroll
          for (int q = 0; q < 4; ++q) s[q] = ldexpf(s[q], ex);
          *reinterpret_cast<float4v*>(to) = s;
        }
      } else {
        for (int i = tid; i < rows * cols; i += kT) {
          const int r = i / cols, c = i - r * cols, t = c / (16 * CPL);
          const uint32_t src = red + t * kHalfSlot + static_cast<uint32_t>(r * kTileStr + c - t * 16 * CPL) * 4u;
          float s = lds_ld<float>(src);
#pragma unroll
          for (int k = 1; k < KP; ++k) s += lds_ld<float>(src + k * NT * kHalfSlot);
          atomic_add_f32(dst + static_cast<int64_t>(half * 8 + r) * stride + c, ldexpf(s, -rexp[half * 8 + r]));
        }
      }
    }
  });
}

// fp32 latent rows [m][.] (rank values of each, `stride` floats apart) as fp16
// rows times a power of two in LDS (dst, dst_str bytes apart), zero past the
// rank (to `width`) and past m up to 16 MB rows; the exponents to rexp.  16
// lanes per row; a row's values stay in registers between its maximum and the
// conversion, and up to 16 loads of a lane are in flight (a second pass over
// the rows, one row at a time, was half of phase BC's time at 64 pairs).
template <int MB, int NV>
__device__ __forceinline__ void stage_rows_n(const float* src, int stride, int m, int rank, int width,
                                             uint32_t dst, uint32_t dst_str, int* rexp) {
  typedef _Float16 half4 __attribute__((ext_vector_type(4)));
  constexpr int kRows = NV * MB <= 16 ? MB : 16 / NV;  // rows at a time
  const int t = threadIdx.x & 15;
  // Loads past row m read zeros: no branch and no mask per load.
  const __amdgpu_buffer_rsrc_t rows = buffer_rsrc(src, static_cast<uint32_t>(m * stride - (stride - width)) * 4u);
#pragma unroll
  for (int i0 = 0; i0 < MB; i0 += kRows) {
    float4v v[kRows][NV];
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      const int r = (threadIdx.x >> 4) + 16 * (i0 + i);
#pragma unroll
      for (int j = 0; j < NV; ++j)
        v[i][j] = __builtin_bit_cast(float4v, __builtin_amdgcn_raw_buffer_load_b128(
                                                  rows, static_cast<uint32_t>(r * stride + 4 * t) * 4u, 256 * j, 0));
    }
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      const int r = (threadIdx.x >> 4) + 16 * (i0 + i);
      float mx = 0.f;
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[i][j][q] = 4 * (t + 16 * j) + q < rank ? v[i][j][q] : 0.f;
          mx = fmaxf(mx, fabsf(v[i][j][q]));
        }
      mx = op_over(mx, 1, 16, OpMax{});
      const int ex = pow2_row_exponent(mx);
      if (t == 0) rexp[r] = ex;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        if (4 * (t + 16 * j) >= width) continue;
        half4 h;
#pragma unroll
        for (int q = 0; q < 4; ++q) h[q] = static_cast<_Float16>(ldexpf(v[i][j][q], ex));
        lds_st<half4>(dst + r * dst_str + (t + 16 * j) * 8, h);
      }
    }
  }
}
template <int MB>
__device__ __forceinline__ void stage_rows(const float* src, int stride, int m, int rank, int width, uint32_t dst,
                                           uint32_t dst_str, int* rexp) {
  if (width <= 128)
    stage_rows_n<MB, 2>(src, stride, m, rank, width, dst, dst_str, rexp);
  else if (width <= 256)
    stage_rows_n<MB, 4>(src, stride, m, rank, width, dst, dst_str, rexp);
  else
    stage_rows_n<MB, 8>(src, stride, m, rank, width, dst, dst_str, rexp);
}

// Waves per SIMD the kernels are compiled for (four pair blocks take 128
// accumulators).
constexpr int waves_for(int mb) { return mb == 1 ? 3 : 2; }

// ---------------------------------------------------------------------------
// Phase A: x . A_g, x . A_u over a range of d rows
// ---------------------------------------------------------------------------
template <int MB, bool kInt8, bool kOrdered>
__global__ void __launch_bounds__(kT, waves_for(MB)) a_kernel(Params p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int rexp[16 * MB];
  int a, item;
  if (!map_item(blockIdx.x, p.n_a * p.n_pass, p.meta[0], a, item)) return;
  const int pass = item / p.n_a;
  item -= pass * p.n_a;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int kind = item & 1, split = item >> 1;
  const int e = p.act_expert[a], s0 = p.act_start[a], mtot = p.act_count[a];
  const int cols = (rank_of(p, e, kind) + kGroup - 1) / kGroup * kGroup;
  // Ranges of d in proportion to the expert's rank, so that items are alike;
  // every plane of an ordered call is written.
  const int pieces = kOrdered ? p.na_split : (p.na_split * max(cols, 128) + p.R - 1) / max(p.R, 128), nblk = p.d / 32;
  if (split >= pieces) return;
  const int blk0 = split * nblk / pieces, blk1 = (split + 1) * nblk / pieces;
  if (blk0 == blk1) return;
  const uint32_t lut0 = lds_addr(smem), lut = lut0 + (lane & (kCopies - 1)) * 4;
  const uint32_t meta = lut0 + kLutBytes + uniform(tid >> 6) * kMetaBytes;
  float* gu = kOrdered && p.na_split > 1 ? p.sums + static_cast<int64_t>(split) * p.T * p.K * (2 * p.R) : p.gu;
  for (int tb = 16 * MB * pass; tb < mtot; tb += 16 * MB * p.n_pass) {
    const int m = min(16 * MB, mtot - tb);
    ActX<MB> act;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {  // rows past m repeat the last: their results are not stored
      const int tok = p.pair_tok[s0 + tb + min(16 * mb + (lane & 15), m - 1)];
      act.src[mb] = p.xh + static_cast<int64_t>(tok) * p.d + 32 * blk0 + 8 * (lane >> 4);
    }
    auto ready = [&]() __attribute__((always_inline)) {
      if (tid < 16 * MB) rexp[tid] = p.xexp[p.pair_tok[s0 + tb + min(tid, m - 1)]];
      lut_fill(lut0, tid);  // the sums take the table's place
      lds_barrier();
    };
    rank_gemm<MB, kInt8, kOrdered>(p.fac[kind ? F_UP_A : F_GATE_A], e, 32 * blk0, blk1 - blk0, cols, m, lut, meta, lut0,
                                   rexp, act, ready, gu + static_cast<int64_t>(s0 + tb) * (2 * p.R) + kind * p.R, 2 * p.R);
    lds_barrier();  // the sums and exponents are read
  }
}

// ---------------------------------------------------------------------------
// Phase BC: g . B_g and u . B_u over 256 columns of ff, h = SiLU(g) u in
// LDS, then h . A_d (those 256 rows of A_d)
// ---------------------------------------------------------------------------
template <int MB, bool kInt8, bool kOrdered>
__global__ void __launch_bounds__(kT, waves_for(MB)) bc_kernel(Params p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int rexp[2][16 * MB], hexp[16 * MB];
  int a, item;
  if (!map_item(blockIdx.x, p.n_bc * p.n_pass, p.meta[0], a, item)) return;
  const int pass = item / p.n_bc;
  item -= pass * p.n_bc;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid >> 6);
  const int n = lane & 15, kq = lane >> 4;
  const int e = p.act_expert[a], s0 = p.act_start[a], mtot = p.act_count[a];
  const int rg = rank_of(p, e, 0), ru = rank_of(p, e, 1), rd = rank_of(p, e, 2);
  const int c0 = item * kCB, ncol = min(kCB, p.ff - c0);
  // LDS: level table and meta slots, then the latents (gate and up halves of a
  // row); their place the h rows take, and behind those the waves' products,
  // eight rows at a time (three workgroups per CU at any rank).
  const uint32_t lstr = (2 * p.R + 8) * 2;
  const uint32_t lut0 = lds_addr(smem), L_lat = lut0 + kFixBytes, L_h = L_lat, L_red = L_h + 16 * MB * kHStr * 2;
  const uint32_t lut = lut0 + (lane & (kCopies - 1)) * 4, meta = lut0 + kLutBytes + wave * kMetaBytes;
  lut_fill(lut0, tid);
  // Waves: (gate, up) x (columns 0-127, 128-255).
  const int kind = wave & 1, tile = wave >> 1;
  const int nb = tile * 128 < ncol ? ((kind ? ru : rg) + 31) / 32 : 0;
  const int cols = (rd + kGroup - 1) / kGroup * kGroup;
  float* dl = kOrdered && p.n_bc > 1 ? p.sums + static_cast<int64_t>(item) * p.T * p.K * p.R : p.dl;
  for (int tb = 16 * MB * pass; tb < mtot; tb += 16 * MB * p.n_pass) {
    const int m = min(16 * MB, mtot - tb);
    Walk<8, MB, kInt8, ActLds> walk(
        p.fac[kind ? F_UP_B : F_GATE_B], e, min(c0 + tile * 128, p.ff - 32), 0, 0, nb, lane, meta,
        ActLds{L_lat + n * lstr + static_cast<uint32_t>(kind * p.R + 8 * kq) * 2u, 16u * lstr});
    walk.start();
    const float* gu = p.gu + static_cast<int64_t>(s0 + tb) * (2 * p.R);
    stage_rows<MB>(gu, 2 * p.R, m, rg, p.R, L_lat, lstr, rexp[0]);
    stage_rows<MB>(gu + p.R, 2 * p.R, m, ru, p.R, L_lat + 2u * p.R, lstr, rexp[1]);
    lds_barrier();
    float4v acc[MB][8];
    walk.run(lut, acc);
    const uint32_t at = L_red + (2 * kind + tile) * kHalfSlot + static_cast<uint32_t>((kq & 1) * 4 * kTileStr + n * 8) * 4u;
#pragma unroll
    for (int half = 0; half < 2 * MB; ++half) {
      lds_barrier();  // the latents (or the last rows' products) are read
      if ((kq >> 1) == (half & 1)) store_tile(at, acc[half >> 1]);
      lds_barrier();
      // h = SiLU(g) u (x router weight before down), fp16 with one exponent
      // per row (the maximum over the item's columns); 32 lanes per row.
      const int r = half * 8 + (tid >> 5), t = tid & 31;
      const float sg = ldexpf(1.0f, -rexp[0][r]), su = ldexpf(1.0f, -rexp[1][r]);
      const float wr = p.wbd && r < m ? p.pair_w[s0 + tb + r] : 1.0f;
      float4v h[2];
      float mx = 0.f;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int col = 128 * j + 4 * t;
        const uint32_t src = L_red + j * kHalfSlot + static_cast<uint32_t>((tid >> 5) * kTileStr + 4 * t) * 4u;
        const float4v g = lds_ld<float4v>(src) * sg, u = lds_ld<float4v>(src + 2 * kHalfSlot) * su;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          h[j][q] = col < ncol && r < m ? g[q] / (1.0f + expf(-g[q])) * u[q] * wr : 0.f;
          mx = fmaxf(mx, fabsf(h[j][q]));
        }
      }
      mx = op_over(mx, 1, 32, OpMax{});
      const int ex = pow2_row_exponent(mx);
      if (t == 0) hexp[r] = ex;
      typedef _Float16 half4 __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        half4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = static_cast<_Float16>(ldexpf(h[j][q], ex));
        lds_st<half4>(L_h + static_cast<uint32_t>(r * kHStr + 128 * j + 4 * t) * 2u, v);
      }
    }
    if (cols != 0)
      rank_gemm<MB, kInt8, kOrdered>(p.fac[F_DOWN_A], e, c0, ncol / 32, cols, m, lut, meta, L_red, hexp,
                                     ActLds{L_h + static_cast<uint32_t>(n * kHStr + 8 * kq) * 2u, 16u * kHStr * 2},
                                     [] { lds_barrier(); }, dl + static_cast<int64_t>(s0 + tb) * p.R, p.R);
    lds_barrier();
  }
}

// ---------------------------------------------------------------------------
// Phase D: d_lat . B_d over 512 columns of d, weighted into out
// ---------------------------------------------------------------------------
// kAdd: weighted into the reduced output by atomics.  Otherwise into rows of
// their own (y, or the per-slot output), each lane its eight columns: through
// LDS, a row at a time like the atomics, the stores of 98 MB of y rows (11,994
// pairs, d 2048) took the phase 67 us, from the registers 38 (with 10 % INT8
// groups, one pair block a pass, both ways level).
template <int MB, bool kInt8, bool kAdd>
__global__ void __launch_bounds__(kT, waves_for(MB)) d_kernel(Params p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  __shared__ int rexp[16 * MB];
  int a, item;
  if (!map_item(blockIdx.x, p.n_d * p.n_pass, p.meta[0], a, item)) return;
  const int pass = item / p.n_d;
  item -= pass * p.n_d;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid >> 6);
  const int n = lane & 15, kq = lane >> 4;
  const int e = p.act_expert[a], s0 = p.act_start[a], mtot = p.act_count[a];
  const int rd = rank_of(p, e, 2);
  const int c0 = item * kCD, ct = c0 + wave * 128;  // a tile of 128 columns per wave
  const int nb = ct < p.d ? (rd + 31) / 32 : 0;
  const uint32_t lstr = (p.R + 8) * 2;
  const uint32_t lut0 = lds_addr(smem), L_lat = lut0 + kFixBytes, lut = lut0 + (lane & (kCopies - 1)) * 4;
  const uint32_t meta = lut0 + kLutBytes + wave * kMetaBytes;
  lut_fill(lut0, tid);
  for (int tb = 16 * MB * pass; tb < mtot; tb += 16 * MB * p.n_pass) {
    const int m = min(16 * MB, mtot - tb);
    Walk<8, MB, kInt8, ActLds> walk(p.fac[F_DOWN_B], e, min(ct, p.d - 32), 0, 0, nb, lane, meta,
                                    ActLds{L_lat + n * lstr + 16u * kq, 16u * lstr});
    walk.start();
    stage_rows<MB>(p.dl + static_cast<int64_t>(s0 + tb) * p.R, p.R, m, rd, p.R, L_lat, lstr, rexp);
    lds_barrier();
    float4v acc[MB][8];
    walk.run(lut, acc);
    if constexpr (!kAdd) {
      const int col = ct + n * 8;
#pragma unroll
      for (int b = 0; b < MB; ++b) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * b + 4 * kq + v;
          if (row >= m || col >= p.d) continue;
          const int pair = s0 + tb + row;
          const int64_t orow = p.y ? pair : static_cast<int64_t>(p.pair_tok[pair]) * p.K + p.pair_slot[pair];
          float4v* dst = reinterpret_cast<float4v*>((p.y ? p.y : p.out) + orow * p.d + col);
          const float sc = ldexpf(1.0f, -rexp[row]);
          dst[0] = sc * float4v{acc[b][0][v], acc[b][1][v], acc[b][2][v], acc[b][3][v]};
          dst[1] = sc * float4v{acc[b][4][v], acc[b][5][v], acc[b][6][v], acc[b][7][v]};
        }
      }
      lds_barrier();  // the latents are read
      continue;
    }
    // Eight rows of every wave's products at a time, one row at a time over the
    // workgroup: a wave's atomics cover consecutive columns.
    const uint32_t at = L_lat + wave * kHalfSlot + static_cast<uint32_t>((kq & 1) * 4 * kTileStr + n * 8) * 4u;
#pragma unroll
    for (int half = 0; half < 2 * MB; ++half) {
      if (half * 8 >= m) break;
      lds_barrier();  // the latents (or the last rows' products) are read
      if ((kq >> 1) == (half & 1)) store_tile(at, acc[half >> 1]);
      lds_barrier();
      const int rows = min(8, m - half * 8);
      for (int r = 0; r < rows; ++r) {
        const int pair = s0 + tb + half * 8 + r;
        const float sc = ldexpf(1.0f, -rexp[half * 8 + r]);
        const float w = p.wbd ? sc : p.pair_w[pair] * sc;
        float* dst = p.out + static_cast<int64_t>(p.pair_tok[pair]) * p.d;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int col = c0 + t * 256 + tid;
          if (col < p.d)
            atomic_add_f32(dst + col, w * lds_ld<float>(L_lat + (2 * t + (tid >> 7)) * kHalfSlot +
                                                        static_cast<uint32_t>(r * kTileStr + (tid & 127)) * 4u));
        }
      }
    }
    lds_barrier();  // the products are read
  }
}

// dst = the planes' sum, in plane order; one float4 per thread.  Columns past an
// expert's rank and rows past the routed pairs were never written: no one
// reads their sums.
__global__ void __launch_bounds__(kT) sum_planes_kernel(const float* planes, int n, int64_t n4, float* dst) {
  const int64_t i = blockIdx.x * static_cast<int64_t>(kT) + threadIdx.x;
  if (i >= n4) return;
  const float4v* src = reinterpret_cast<const float4v*>(planes) + i;
  float4v s = src[0];
#pragma unroll 8
  for (int k = 1; k < n; ++k) s += src[k * n4];
  reinterpret_cast<float4v*>(dst)[i] = s;
}

// Reduced output from y rows: the weighted sum over a token's slots in slot
// order, one float4 per thread.  One grid dimension: a call may have more tokens
// than the 65,535 workgroups of another.
__global__ void __launch_bounds__(kT) combine_kernel(Params p) {
  const int d4 = p.d / 4, per = (d4 + kT - 1) / kT;
  const int t = blockIdx.x / per, c = (blockIdx.x - t * per) * kT + threadIdx.x;
  if (c >= d4) return;
  float4v s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int k = 0; k < p.K; ++k) {
    const int slot = t * p.K + k, e = p.ids[slot];
    if (e < 0 || e >= p.E) continue;
    const float w = p.wbd ? 1.0f : load_act(p.weights, p.w_dtype, slot);
    s += w * reinterpret_cast<const float4v*>(p.y + static_cast<int64_t>(p.pos_of[slot]) * p.d)[c];
  }
  reinterpret_cast<float4v*>(p.out + static_cast<int64_t>(t) * p.d)[c] = s;
}

// Dynamic LDS bytes of the phases.
constexpr size_t lds_a() { return std::max(kFixBytes, kRedBytes); }
template <int MB>
size_t lds_bc(int R) {
  return static_cast<size_t>(kFixBytes + std::max(16 * MB * (2 * R + 8) * 2, 16 * MB * kHStr * 2 + kRedBytes));
}
template <int MB>
size_t lds_d(int R) {
  return static_cast<size_t>(kFixBytes + std::max(16 * MB * (R + 8) * 2, kRedBytes));
}

template <int MB, bool kInt8, bool kOrdered = false>
int launch_phases(const Params& p, hipStream_t s) {
  const unsigned groups = static_cast<unsigned>((p.a_max + 7) / 8 * p.n_pass);
  const int64_t P = static_cast<int64_t>(p.T) * p.K;
  auto sum_planes = [&](int n, int64_t width, float* dst) {
    if (!kOrdered || n == 1) return;
    const int64_t n4 = P * width / 4;
    hipLaunchKernelGGL(sum_planes_kernel, dim3(static_cast<unsigned>((n4 + kT - 1) / kT)), dim3(kT), 0, s, p.sums, n, n4,
                       dst);
  };
  hipLaunchKernelGGL((a_kernel<MB, kInt8, kOrdered>), dim3(8 * groups * p.n_a), dim3(kT), lds_a(), s, p);
  sum_planes(p.na_split, 2 * p.R, p.gu);
  hipLaunchKernelGGL((bc_kernel<MB, kInt8, kOrdered>), dim3(8 * groups * p.n_bc), dim3(kT), lds_bc<MB>(p.R), s, p);
  sum_planes(p.n_bc, p.R, p.dl);
  if (!p.y && p.out_mode == LATENT_OUT_REDUCED)
    hipLaunchKernelGGL((d_kernel<MB, kInt8, true>), dim3(8 * groups * p.n_d), dim3(kT), lds_d<MB>(p.R), s, p);
  else
    hipLaunchKernelGGL((d_kernel<MB, kInt8, false>), dim3(8 * groups * p.n_d), dim3(kT), lds_d<MB>(p.R), s, p);
  const unsigned per_token = (p.d / 4 + kT - 1) / kT;
  if (p.y) hipLaunchKernelGGL(combine_kernel, dim3(per_token * p.T), dim3(kT), 0, s, p);
  return hipGetLastError() == hipSuccess ? LATENT_OK : LATENT_E_HIP;
}

}  // namespace

bool supported(const latent_moe_args& a) {
  if (a.layout != LATENT_LAYOUT_ROWS || a.max_rank > 512) return false;
  if ((reinterpret_cast<uintptr_t>(a.x) & 15u) != 0) return false;  // 16-byte loads of x (prep's fp16 rows)
  // INT8 bytes are read through 32-bit buffer offsets: even an all-INT8 side
  // buffer of a factor must stay below 2^31 bytes.
  const latent_factor* fs[6] = {&a.gate_a, &a.gate_b, &a.up_a, &a.up_b, &a.down_a, &a.down_b};
  for (const latent_factor* f : fs) {
    if (!f->int8_bitmap) continue;
    if (a.n_expert * f->rows * f->cols >= (int64_t{1} << 31)) return false;
  }
  return true;
}

// Pair blocks a decoded block of the factor is multiplied with: an expert of
// many pairs then decodes its factors once per 64 (or 32) of them.  E 128, d
// 4096, ff 1408, rank 64, top-8: 200 tokens (12 pairs an expert) 99 us at one
// block and 110 at two, 2000 tokens 674 at one and 568 at four; E 64, d 2048,
// rank 192, 200 tokens (19 pairs): 124 at one, 116 at two.
// Above rank 256, four blocks' latents leave LDS for one workgroup per CU, which
// pays from some 64 pairs an expert (E 64, d 4096, ff 1408, top-8, us at one / two
// / four blocks): rank 480 50 pairs 328 / 439 / 415, 87 pairs 512 / - / 526, 125
// pairs 691 / 730 / 706; rank 416 302 / 357 / 341, 478 / - / 441, 645 / 588 / 601.
// Ordered calls (ff 2048): rank 384 50 pairs 308 / 292 / 339, 81 pairs - / 389 /
// 416; rank 512 348 / 377 / 392, 125 pairs 707 / 745 / 652.
int pair_blocks(const Params& p, bool int8) {
  const int64_t per = static_cast<int64_t>(p.T) * p.K / p.a_max;
  if (!int8 && p.R > 256 && per < (p.ordered ? 96 : 64)) return p.ordered ? 2 : 1;
  return int8 || per < 16 ? 1 : per < 24 ? 2 : 4;
}

void plan(Params& p, bool int8) {
  // Workgroups that share an expert's passes, up to four rounds of phase D's items.
  const int64_t step = 16 * pair_blocks(p, int8);
  const int64_t passes = (3 * static_cast<int64_t>(p.T) * p.K / (2 * p.a_max) + step - 1) / step;  // half over the mean
  p.n_bc = (p.ff + kCB - 1) / kCB;
  p.n_d = (p.d + kCD - 1) / kCD;
  p.n_pass = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(passes, 2048 / (static_cast<int64_t>(p.a_max) * p.n_d))));
  // Phase A ranges per expert and factor at the full rank (a smaller rank has
  // fewer): about 4096 items in all, of eight blocks of 32 rows or more; with
  // 64 pairs a pass the items are eight times as long, and their sums cost as
  // many atomics per range.  Ordered calls, one plane per range: some 512 items
  // and at most four ranges (E 256, d 7168, rank 256, 512 tokens: 417 us at one,
  // 433 at four; E 64, d 4096, rank 256, 150 tokens 121 and 98).
  const bool few = step == 64 || p.ordered;
  const int64_t want = few ? 512 : 4096;
  int s = few ? 1 : 4;
  while (s < (p.ordered ? 4 : 32) && 2ll * p.a_max * p.n_pass * s < want && p.d / 32 >= 16 * s) s *= 2;
  p.na_split = s;
  p.n_a = 2 * s;
}

size_t sums_bytes(const Params& p) {
  const size_t P = static_cast<size_t>(p.T) * p.K;
  size_t n = p.out_mode == LATENT_OUT_REDUCED ? P * p.d : 0;
  if (p.na_split > 1) n = std::max(n, P * 2 * p.R * p.na_split);
  if (p.n_bc > 1) n = std::max(n, P * p.R * p.n_bc);
  return n * sizeof(float);
}

int launch(const Params& p, bool int8, hipStream_t s) {
  if (p.ordered)  // at least 16 pairs an expert, no INT8 groups
    return pair_blocks(p, false) == 4 ? launch_phases<4, false, true>(p, s) : launch_phases<2, false, true>(p, s);
  if (int8) return launch_phases<1, true>(p, s);
  switch (pair_blocks(p, false)) {
    case 4: return launch_phases<4, false>(p, s);
    case 2: return launch_phases<2, false>(p, s);
    default: return launch_phases<1, false>(p, s);
  }
}

}  // namespace rows
}  // namespace latent
