// gfx950 matrix-core and LDS helpers shared by the attention kernels.
#pragma once

#include "pkv_common.h"

namespace pkv {

typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

template <typename T> struct Mma;
template <> struct Mma<_Float16> {
  typedef f16x8 vec8;
  typedef f16x4 vec4;
  __device__ static f32x4 qk(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
  __device__ static f32x4 pv(vec4 a, vec4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<__bf16> {
  typedef bf16x8 vec8;
  typedef bf16x4 vec4;
  __device__ static f32x4 qk(vec8 a, vec8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  __device__ static f32x4 pv(vec4 a, vec4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(i16x4, a),
                                                    __builtin_bit_cast(i16x4, b), c, 0, 0, 0);
  }
};

// MFMA operand layouts used here (16x16 tiles, 64 lanes, lane l = 16 g + n):
//   16x16x32: A: lane holds A[n][8g .. 8g+7]; B: lane holds B[8g .. 8g+7][n];
//   16x16x16: A: lane holds A[n][4g .. 4g+3]; B: lane holds B[4g .. 4g+3][n];
//   C/D (both): lane holds D[4g + i][n], i = 0..3.
// ds_read_b64_tr_b16: within each 16-lane block, lane i receives element i
// of each of the 4 rows x 16 columns (16-bit) that the block's lanes point
// at (4 consecutive elements each) -- i.e. a transposed 4x16 tile.
// Orders this wave's LDS writes before its own (cross-lane) LDS reads. A
// wave's LDS operations execute in order, so a compiler-level barrier with
// wavefront-scope fences is all that is needed (no s_barrier).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Buffer resource over [base, base + bytes): raw (untyped) records with a
// hardware range check (out-of-range loads read 0, stores are dropped). The
// base lives in scalar registers, so per-lane addresses are 32-bit offsets.
// Cache-policy bits of a buffer load/store: kSc1 = agent-scope coherent
// access (through to the memory-side coherence point), kNt = streaming.
constexpr int kNt = 2;
constexpr int kSc1 = 16;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ws_rsrc(void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(base, (short)0, (int)bytes, 0x00020000);
}

// Row `row` of a tile stores its 16-byte chunk c at chunk position
// c ^ xr(row), xr a permutation of row & 7. Eight consecutive rows reading
// the same chunk (the K operand reads) then hit eight different chunk
// positions, and so do four consecutive rows reading chunks 2j and 2j + 1
// (the transposed V reads): both are free of bank conflicts.
__device__ __forceinline__ int xr(int row) { return ((row & 3) << 1) | ((row >> 2) & 1); }
// Byte offset of element `e` (of 2-byte elements) in row `row` of a tile.
template <int RB>
__device__ __forceinline__ int swz(int row, int e) {
  return row * RB + ((((e >> 3) ^ xr(row)) & 7) | ((e >> 3) & ~7)) * 16 + (e & 7) * 2;
}

// NL loads of 16 bytes a lane straight to LDS: load k from range `rs` at byte
// offset v[k] to LDS bytes lds + 1024 k + 16 * lane .. + 15. The whole offset
// is the lane's: a scalar offset is documented as outside the range check.
// Written in asm so that only the kernel's own waits cover them: where the
// compiler cannot tell an LDS ring's tiles apart, it waits for every load in
// flight before each tile read. No vector register is written; the no-ops cover
// scalar registers written just before; m0, which the compiler may use, is put
// back.
template <int NL>
__device__ __forceinline__ void load_to_lds(u32x4 rs, const uint32_t* v, uint32_t lds) {
  static_assert(NL == 2 || NL == 4, "a page of 2 or 4 KiB");
  uint32_t m0;
  if constexpr (NL == 2)
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %4\n\ts_nop 4\n\t"
                 "buffer_load_dwordx4 %1, %3, 0 offen lds\n\ts_mov_b32 m0, %5\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %2, %3, 0 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(m0)
                 : "v"(v[0]), "v"(v[1]), "s"(rs), "s"(lds), "s"(lds + 1024)
                 : "memory");
  else
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %6\n\ts_nop 4\n\t"
                 "buffer_load_dwordx4 %1, %5, 0 offen lds\n\ts_mov_b32 m0, %7\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %2, %5, 0 offen lds\n\ts_mov_b32 m0, %8\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %3, %5, 0 offen lds\n\ts_mov_b32 m0, %9\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %4, %5, 0 offen lds\n\ts_mov_b32 m0, %0"
                 : "=&s"(m0)
                 : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "s"(rs), "s"(lds),
                   "s"(lds + 1024), "s"(lds + 2048), "s"(lds + 3072)
                 : "memory");
}
// The buffer resource of ws_rsrc as the four words load_to_lds takes.
__device__ __forceinline__ u32x4 raw_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes, 0x00020000u};
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)p);
}

}  // namespace pkv
