// bf16 matrix-core helpers of the attention kernels.
#pragma once
#include "models.h"
#include <math.h>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef zp_u32x4 u32x4;
typedef zp_f32x4 f32x4;

__device__ __forceinline__ f32x4 mfma_bf16(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// 32 x 32 x 16: lane (half, l32) gives row or column l32 at elements 8 half .., and ends with rows 8 (i / 4) + 4 half + i % 4 of
// column l32.  Half the operand reads of 16 x 16 x 32 for the same products, and a quarter of its cycles at the vector issue
// instead of a half.
typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f32x16 mfma32_bf16(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const zp_f32x2 f = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, zp_bf16x2));
}
// key of operand element i (0..7) held by lane group g, within a step of 32 keys
__device__ __forceinline__ int step_key(int g, int i) { return i < 4 ? 4 * g + i : 12 + 4 * g + i; }

// A 4 x 16 block of 16-bit values in LDS, transposed: lane i of a group of sixteen names row i / 4, values 4 (i % 4) on,
// and receives the four of column i.
typedef short zp_s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint2 read_transposed(const uint16_t* p) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) zp_s16x4*)p));
}

// A load straight into LDS: lane l's 16 bytes from `rows` + lane_at (+ at) to `lds` + 16 l.  Written out, because the compiler,
// which cannot tell the stage being filled from the stage being read, would wait for it at the next LDS read; what
// waits is the code that meets the other waves.
typedef __attribute__((address_space(3))) void* lds_ptr_t;
// PAST: past the last-level cache, where more is read once than that holds
template <bool PAST> __device__ __forceinline__ u32x4 load_piece(const void* p) {
  if constexpr (PAST) return __builtin_nontemporal_load((const u32x4*)p);
  return *(const u32x4*)p;
}
__host__ __device__ inline bool past_cache(int64_t bytes) { return bytes >= 320ll << 20; }
template <bool PAST = false>
__device__ __forceinline__ void load_to_lds(const u32x4& rows, void* lds, int lane_at, int at) {
  const uint32_t to = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(uintptr_t)(lds_ptr_t)lds);
  const int so = __builtin_amdgcn_readfirstlane(at);
  if constexpr (PAST)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :: "s"(to), "v"(lane_at), "s"(rows), "s"(so) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(to), "v"(lane_at), "s"(rows), "s"(so) : "memory", "m0");
}
// What such loads read: `bytes` from `base` on, zeros behind them.
__device__ __forceinline__ u32x4 rows_from(const void* base, uint32_t bytes) {
  const uint64_t p = (uint64_t)base;
  return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)p),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(p >> 32) & 0xffffu)),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}

// Eight rows (keys) of eight bf16 columns -> for column t the four dwords of its eight keys.
__device__ __forceinline__ u32x4 column_of(const u32x4* rows, int t) {
  const uint32_t sel = (t & 1) ? 0x07060302u : 0x05040100u;
  u32x4 o;
#pragma unroll
  for (int d = 0; d < 4; ++d)
    o[d] = __builtin_amdgcn_perm(rows[2 * d + 1][t >> 1], rows[2 * d][t >> 1], sel);
  return o;
}

}  // namespace
