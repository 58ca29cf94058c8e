// What the 16-bit kernels with loads that write LDS directly share (gemm_dma.hip, gemm_ring.hip): MFMA, explicit waits, the load, and
// the layouts of an operand's tile in LDS.
#pragma once
#include <hip/hip_runtime.h>

#include "gemm.h"

namespace ughip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

typedef float floatx4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ floatx4 mma16(__bf16, const u32x4& a, const u32x4& b, const floatx4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ floatx4 mma16(_Float16, const u32x4& a, const u32x4& b, const floatx4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// s_waitcnt vmcnt(n) alone (gfx9 encoding: vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 15) | (((N >> 4) & 3) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(0xc07f); }

// Every lane's 16 bytes at base + voff go to LDS at lds_byte_addr + lane * 16.  The compiler does not see the load
// (it would wait for all of them before any LDS read): the waits are explicit.
__device__ __forceinline__ void dma16(const void* base, unsigned voff, unsigned lds_byte_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_byte_addr), "v"(voff), "s"(base) : "memory", "m0");
}
constexpr int BK = 64;

// k-contiguous operand tile ([rows][64] 16-bit): 128-byte rows of 8 chunks, chunk' = chunk ^ ((row / 2) & 7)
__device__ __forceinline__ int kc_idx(int row, int chunk) { return row * 8 + (chunk ^ ((row >> 1) & 7)); }  // in 16-byte units

// n-contiguous rhs tile ([64 k][BN n] 16-bit): rows of BN / 16 pieces of 32 bytes, piece' = piece ^ h(k) with
// h(k) = (k & 3) | ((k >> 3) & 1) << 2.  A transposing read names, per half wave, 8 rows (k = 8 g + e: e = 0..3 and two values
// of g) and 32 bytes of each; h sends those rows to 8 different pieces, i.e. to all 64 banks once.  (With 64-byte segments
// swizzled by k & 7 the two g of a half wave met in the same banks: 4096^3 95.5 -> 94.2 us on one box.)
__device__ __forceinline__ int kn_h(int k) { return (k & 3) | (((k >> 3) & 1) << 2); }
template <int BN>
__device__ __forceinline__ int kn_byte(int k, int n) {
  return k * (BN * 2) + (((n >> 4) ^ kn_h(k)) << 5) + (n & 15) * 2;
}

// Which K tile of the lhs and of the rhs in memory K tile `tile` of the loop reads (scalar arithmetic); BDIV as in gemm_dma4.
template <int BDIV>
__device__ __forceinline__ int lhs_k_tile(int tile) {
  if constexpr (BDIV == 6) {
    const int g = tile / 6, r = tile - 6 * g;
    return 3 * g + ((0x010120 >> (4 * r)) & 3);  // planes 0, 2, 1, 0, 1, 0
  } else {
    return tile;
  }
}
template <int BDIV>
__device__ __forceinline__ int rhs_k_tile(int tile) {
  if constexpr (BDIV == 6) {
    const int g = tile / 6, r = tile - 6 * g;
    return 3 * g + ((0x001102 >> (4 * r)) & 3);  // planes 2, 0, 1, 1, 0, 0
  } else {
    return tile / BDIV;
  }
}

// The products those kernels take, besides plain ones: see gemm_dma4.
enum class DmaForm { PLAIN, PLANES3, ROWS, ROWS_GLU, ROWS_LOOKUP };
// gemm_ring.hip: one of its tiles (codes 129, 97, 65, 48, 32: 256 x 128, 192 x 192, 128 x 128, 64 x 128, 64 x 64), operands as the _supported functions of gemm_dma.hip check them.
hipError_t gemm_ring_launch(hipStream_t stream, int dtype, DmaForm form, const MMArgs& p, size_t batch, int tile, const float* residual, const DmaRows& rw);

}  // namespace ughip
