// Blocks of a row-layout factor as MFMA B operands, without a transpose.
//
// A row-layout factor [K][N] stores 32-column groups along N (16 bytes of NF4
// codes, low nibble first, and one fp16 scale).  A wave takes a block of 32
// rows by 16 CPL columns: lane (n = lane & 15, kq = lane >> 4) loads CPL / 2
// bytes of each of the rows 8 kq .. 8 kq + 7, columns CPL n .. CPL n + CPL - 1.
// Column c of those of every lane is one 16-column MFMA operand (a column
// order that only the store of the result sees), and the lane's eight rows are
// its K values: no LDS round trip and no barrier between HBM and the matrix
// cores.
#pragma once

#include "common.hpp"

namespace latent {
namespace rowblock {

typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// LDS byte address of a __shared__ array and raw LDS accesses.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) char*)(p)));
}
template <typename T>
__device__ __forceinline__ T lds_ld(uint32_t addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>(static_cast<uintptr_t>(addr));
}
template <typename T>
__device__ __forceinline__ void lds_st(uint32_t addr, const T& v) {
  *reinterpret_cast<__attribute__((address_space(3))) T*>(static_cast<uintptr_t>(addr)) = v;
}

// Workgroup barrier over LDS only (__syncthreads() would also wait for the
// global loads issued ahead).
__device__ __forceinline__ void lds_barrier() {
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt left at their maxima
  __builtin_amdgcn_s_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Raw buffer resource over `bytes` bytes (loads beyond them return zero).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0), static_cast<int>(bytes),
                                           0x00020000);
}

// One lane's codes and scales of a block (rows 8 kq + i).
template <int CPL>
struct Block {
  uint32_t c[8];
  u16x2 s[4];  // rows 2 i, 2 i + 1
};

// One lane's view of 16 CPL columns of an expert's factor, from column col0
// (a multiple of 16 CPL).  Lanes past the factor's last column read its last
// group: their results are never stored.  Every factor has a multiple of 32
// rows, so a block never ends early.
template <int CPL>
struct Src {
  __amdgpu_buffer_rsrc_t rc, rs;
  uint32_t vc, vs;  // the lane's offsets at row 8 kq
  int cs, ss;       // bytes per row of codes and scales
  int group;
};
template <int CPL>
__device__ __forceinline__ Src<CPL> make_src(const Factor& f, int e, int col0, int lane) {
  const int n = lane & 15, kq = lane >> 4;
  const int64_t er = static_cast<int64_t>(e) * f.rows;
  Src<CPL> s;
  s.cs = static_cast<int>(f.code_stride());
  s.ss = static_cast<int>(f.scale_stride()) * 2;
  s.rc = buffer_rsrc(f.codes + er * s.cs, static_cast<uint32_t>(f.rows) * s.cs);
  s.rs = buffer_rsrc(reinterpret_cast<const char*>(f.scales) + er * s.ss, static_cast<uint32_t>(f.rows) * s.ss);
  const int col = min(col0 + CPL * n, static_cast<int>(f.cols) - CPL);
  s.group = col / kGroup;
  s.vc = static_cast<uint32_t>(8 * kq * s.cs + col / 2);
  s.vs = static_cast<uint32_t>(8 * kq * s.ss + s.group * 2);
  return s;
}
// Rows 2 h and 2 h + 1 of the lane in the block whose first row is `row` (uniform).
template <int CPL>
__device__ __forceinline__ void load_rows(const Src<CPL>& s, int row, int h, Block<CPL>& b) {
  static_assert(CPL == 4 || CPL == 8, "columns per lane");
  const int oc = row * s.cs, os = row * s.ss;
#pragma unroll
  for (int i = 2 * h; i < 2 * h + 2; ++i) {
    if (CPL == 8)
      b.c[i] = __builtin_amdgcn_raw_buffer_load_b32(s.rc, s.vc, oc + i * s.cs, 0);
    else
      b.c[i] = __builtin_amdgcn_raw_buffer_load_b16(s.rc, s.vc, oc + i * s.cs, 0);
    b.s[i >> 1][i & 1] = __builtin_amdgcn_raw_buffer_load_b16(s.rs, s.vs, os + i * s.ss, 0);
  }
}

// INT8 groups: the lane's bytes of row `row` (absolute) of expert e.  Returns
// whether the group is INT8; q holds CPL bytes then.
template <int CPL>
__device__ __forceinline__ bool int8_row(const Factor& f, int e, int row, int col, uint32_t (&q)[(CPL + 3) / 4]) {
  const int64_t er = static_cast<int64_t>(e) * f.rows + row;
  const int g = col / kGroup;
  const int64_t wi = er * f.words() + (g >> 5);
  const uint32_t word = f.ext.bitmap[wi], bit = 1u << (g & 31);
  if (!(word & bit)) return false;
  const int64_t idx = f.ext.word_offset[wi] + popc(word & (bit - 1u));
  const int8_t* src = f.ext.data + idx * kGroup + col % kGroup;
#pragma unroll
  for (int i = 0; i < (CPL + 3) / 4; ++i) q[i] = reinterpret_cast<const uint32_t*>(src)[i];
  return true;
}

}  // namespace rowblock
}  // namespace latent
