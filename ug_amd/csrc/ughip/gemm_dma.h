// What the 16-bit kernels with loads that write LDS directly share (gemm_dma.hip, gemm_ring.hip): MFMA, explicit waits, the load, and
// the layouts of an operand's tile in LDS.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm.h"
#include "layers.h"

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

// Inclusive scans over the lanes of a wave, all active; of values from 0 up.
template <int CTRL, int ROWS>
__device__ __forceinline__ int scan_move(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, false);  // 0 where there is no lane to read from
}
template <typename F>
__device__ __forceinline__ int wave_scan(int v, F f) {
  v = f(v, scan_move<0x111, 0xf>(v));  // within rows of 16 lanes: from 1, 2, 4 and 8 lanes below
  v = f(v, scan_move<0x112, 0xf>(v));
  v = f(v, scan_move<0x114, 0xf>(v));
  v = f(v, scan_move<0x118, 0xf>(v));
  v = f(v, scan_move<0x142, 0xa>(v));  // the last lane of rows 0 and 2 to rows 1 and 3
  return f(v, scan_move<0x143, 0xc>(v));  // lane 31 to rows 2 and 3
}

// Rows sorted by group, ceil(rows / BM) tile rows to each: a lane per group, 64 at a time.  Every workgroup asks for it before its first load, one
// that finds no tile of its own too, and mostly has its CU to itself: read one after the other by scalar loads the ends took it 0.1-0.15 us each
// (64 groups, n = 2 x 552, k = 128, 1638 rows: 49 us so, on 64 x 128 tiles, 12.8 with a lane per group; 18.9 in rows_product).
// EVEN: a group's rows in shares of equal size, whole 16s (BM % 16 == 0: no share is larger than BM, and as rows are more than (tiles - 1) BM, none is empty).
template <int BM, bool EVEN = false>
struct GroupTiles {
  const int* group_end;
  int groups, m, lane;
  int begin = 0, end = 0, upto = 0;  // lane's group: its rows, and the tile rows of all groups up to it
  int rows = 0, tiles = 0;           // of the groups read so far

  __device__ __forceinline__ void read(int base) {
    int e = base + lane < groups ? group_end[base + lane] : 0;
    e = wave_scan(max(min(e, m), rows), [](int a, int b) { return max(a, b); });  // (an end in front of its predecessor's: an empty group)
    begin = __builtin_amdgcn_update_dpp(rows, e, 0x138, 0xf, 0xf, false);         // from one lane below, lane 0 the groups in front
    end = e;
    upto = tiles + wave_scan((e - begin + BM - 1) / BM, [](int a, int b) { return a + b; });
    rows = __builtin_amdgcn_readlane(e, 63), tiles = __builtin_amdgcn_readlane(upto, 63);
  }
  __device__ __forceinline__ int count() {
    rows = tiles = 0;
    for (int base = 0; base < groups; base += 64) read(base);
    return tiles;
  }
  // behind count(): group and rows [m0, m_end) of a tile row below it
  __device__ __forceinline__ bool find(int tile, int& group, int& m0, int& m_end) {
    if (groups > 64) rows = tiles = 0;
    for (int base = 0; base < groups; base += 64) {
      if (groups > 64) read(base);
      const unsigned long long behind = __ballot(upto > tile);
      if (!behind) continue;
      const int l = __builtin_ctzll(behind), first = __builtin_amdgcn_readlane(begin, l);
      group = base + l, m_end = __builtin_amdgcn_readlane(end, l);
      const int n = (m_end - first + BM - 1) / BM, at = tile - __builtin_amdgcn_readlane(upto, l) + n;
      if constexpr (EVEN) {
        const int share = ((m_end - first + n - 1) / n + 15) / 16 * 16;
        m0 = first + at * share, m_end = min(m_end, m0 + share);
      } else {
        m0 = first + at * BM;
      }
      return true;
    }
    return false;
  }
};

// The products those kernels take, besides plain ones: see gemm_dma4.
enum class DmaForm { PLAIN, PLANES3, ROWS, ROWS_GLU, ROWS_LOOKUP };
// How a wave's NI x NJ fragments of rows leave (ROWS as in gemm_dma4, 3 as in gemm_ring): register e of fragment (i, j) is row row0 + 16 i of the tile's, column col0 + 16 j + e.
// First everything that has to be loaded, then stores alone: a wait for a load behind a store is a wait for that store's way to memory as well, and with a bias or a table looked at
// fragment by fragment each store was waited for before the next one went out, a lone wave per SIMD with nothing to do meanwhile: 256 x 256 tiles spent 26700 cycles here, gated ones
// 23200; 20700 and 11800 so (2048 x 2 of 5632 x 2048 104 -> 94 us on them, 93 -> 92 on the ring's 256 x 128; 2048 x 8192 x 2048 62 -> 59).
// A store takes a CU's address unit a cycle for each lane that does not follow its neighbour in memory, and a lane of a fragment has a row to itself: 70 to 80 cycles where 16 would do.  So 16
// rows at a time go through the wave's own piece of LDS (nobody reads operands any more; a wave's LDS instructions keep their order, so there is no barrier) and leave in 16-byte
// pieces of whole rows, the next 16 on their way into a second piece: us, 2048 rows, weights from memory: f32 3072 x 2048
// 47.8 -> 45.2 (256 x 256 tiles), 43.4 -> 41.8 (128 x 128); bf16 8192 x 2048 69.3 -> 66.5 (256 x 128), 86.3 -> 81.3 (128 x 128); gated 2 x 5632 92.2 -> 90.9, 116 -> 112.5.
template <typename T, int ROWS, int NI, int NJ>
__device__ __forceinline__ void rows_out(floatx4 (&acc)[NI][NJ], const DmaRows& rw, int m0, int m_last, int row_base, int col_base, int wave, u32x4* lds) {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));  // (not worked out in front of the products, where there is no register to keep it in)
  const int row0 = row_base + (lane & 15), col0 = col_base + (lane >> 4) * 4;
  typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
  constexpr int NC = ROWS == 2 ? NJ / 2 : NJ;
  floatx4 b[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) b[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (rw.bias) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) b[j] = *reinterpret_cast<const floatx4*>(rw.bias + (j < NC ? 0 : rw.n_out) + min(col0 + j % NC * 16, rw.n_out - 4));
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) asm volatile("" : "+v"(b[j]));  // they are here from now on
  if constexpr (ROWS == 3) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int id = rw.ids[m0 + min(row0 + i * 16, m_last)];
      const bool known = id >= 0 && id < rw.table_rows;
      const size_t at = (size_t)(known ? id : 0) * rw.table_stride + rw.table_col;
      // 16 rows' table elements at a time (all of them at once are more than the registers hold), the table's type asked for once: asked for each, every load was waited for by itself and the gates stayed, in
      // part in scratch memory, until the last of them
      float f[NJ][4];
      auto load = [&](auto* table) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const auto v = table[at + min(col0 + j * 16, rw.n_out - 4) + e];
            if constexpr (sizeof(v) == 2) f[j][e] = bf16_to_f32(v);
            else f[j][e] = v;
          }
      };
      if (rw.table_bf16) load(static_cast<const uint16_t*>(rw.table));
      else load(static_cast<const float*>(rw.table));
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[i][j][e] = gelu_tanh_f(acc[i][j][e] + b[j][e]) * (known ? f[j][e] : __uint_as_float(0x7fc00000u));
          asm volatile("" : "+v"(acc[i][j][e]));
        }
      asm volatile("" ::: "memory");
    }
  }
  auto value = [&](int i, int j) {
    if constexpr (ROWS == 3) return acc[i][j];
    floatx4 v = acc[i][j] + b[j];
    if constexpr (ROWS == 2) {
      floatx4 u = acc[i][j + NC] + b[j + NC];
      if (rw.glu_limit > 0.f) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = v[e] > rw.glu_limit ? rw.glu_limit : v[e];
          u[e] = u[e] > rw.glu_limit ? rw.glu_limit : u[e] < -rw.glu_limit ? -rw.glu_limit : u[e];
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = v[e] * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * rw.glu_alpha * v[e])) * (u[e] + rw.glu_shift);
    }
    return v;
  };
  auto out = [&](auto* dst) {
    constexpr int E = sizeof(*dst), PER = 16 / E, CPR = NC * 16 / PER, RP = 64 / CPR, PITCH = NC * 16 * E + 16, PIECE = 16 * PITCH, PIECES = NI > 1 ? 2 : 1;  // elements of 16 bytes, those of a row, rows of a pass
    typedef char __attribute__((address_space(3))) lds_char;
    if (CPR >= 4 && (E == 4 || ((rw.n_out | rw.dst_stride) % 8 == 0 && ((size_t)rw.dst & 15) == 0))) {
      lds_char* mine = (lds_char*)lds + wave * PIECES * PIECE;
      auto put = [&](int i) {
        lds_char* to = mine + (i & 1) * PIECE + (lane & 15) * PITCH + (lane >> 4) * 4 * E;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
          const floatx4 v = value(i, j);
          if constexpr (E == 2) *(u32x2 __attribute__((address_space(3)))*)(to + j * 32) = __builtin_bit_cast(u32x2, __builtin_convertvector(v, bf16x4));
          else *(floatx4 __attribute__((address_space(3)))*)(to + j * 64) = v;
        }
        asm volatile("" ::: "memory");
      };
      put(0);
      const int c = lane % CPR, r0 = lane / CPR, row = row_base + r0, col = col_base + c * PER;
      const bool there = r0 < RP && col < rw.n_out;  // n_out % PER == 0: a piece exists whole or not at all
      auto* to = dst + (size_t)(m0 + row) * rw.dst_stride + col;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if (i + 1 < NI) put(i + 1);
#pragma unroll
        for (int r = 0; r < 16; r += RP) {
          if (there && r + r0 < 16 && row + i * 16 + r <= m_last)
            *reinterpret_cast<u32x4*>(to + (i * 16 + r) * (size_t)rw.dst_stride) = *(const u32x4 __attribute__((address_space(3)))*)(mine + (i & 1) * PIECE + (r + r0) * PITCH + c * 16);
        }
        asm volatile("" ::: "memory");
      }
      return;
    }
    auto* to = dst + (size_t)(m0 + row0) * rw.dst_stride + col0;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (row0 + i * 16 <= m_last) {
#pragma unroll
        for (int j = 0; j < NC; ++j)
          if (col0 + j * 16 < rw.n_out) {  // n_out % 4 == 0: a group of 4 columns exists whole or not at all
            const floatx4 v = value(i, j);
            if constexpr (E == 2) *reinterpret_cast<u32x2*>(to + j * 16) = __builtin_bit_cast(u32x2, __builtin_convertvector(v, bf16x4));
            else *reinterpret_cast<floatx4*>(to + j * 16) = v;
          }
      }
      to += 16 * (size_t)rw.dst_stride;
    }
  };
  if (rw.dst_bf16) out(static_cast<T*>(rw.dst));
  else out(static_cast<float*>(rw.dst));
}

// How f32 sums leave, N % 8 == 0: rows of n from c on, by the same way.  A residual is added to them first, all of it loaded before the first store (but for
// the tile whose sums leave no registers for that).
template <int NI, int NJ>
__device__ __forceinline__ void sums_out(floatx4 (&acc)[NI][NJ], float* __restrict__ c, const float* __restrict__ residual, int n, int m_last, int n_left, int row_base, int col_base,
                                         int wave, u32x4* lds) {
  constexpr int CPR = NJ * 4, RP = 64 / CPR, PITCH = NJ * 64 + 16, PIECE = 16 * PITCH, PIECES = NI > 1 ? 2 : 1;
  typedef char __attribute__((address_space(3))) lds_char;
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  if (NI * NJ < 64 && residual) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const float* from = residual + (size_t)min(row_base + i * 16 + (lane & 15), m_last) * n;
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] += *reinterpret_cast<const floatx4*>(from + min(col_base + j * 16 + (lane >> 4) * 4, n_left - 4));
    }
  }
  const int r0 = lane / CPR, row = row_base + r0, col = col_base + lane % CPR * 4;
  const bool there = r0 < RP && col < n_left;  // a piece exists whole or not at all
  lds_char* mine = (lds_char*)lds + wave * PIECES * PIECE;
  auto put = [&](int i) {
    lds_char* to = mine + (i & 1) * PIECE + (lane & 15) * PITCH + (lane >> 4) * 16;
#pragma unroll
    for (int j = 0; j < NJ; ++j) *(floatx4 __attribute__((address_space(3)))*)(to + j * 64) = acc[i][j];
    asm volatile("" ::: "memory");
  };
  float* to = c + (size_t)row * n + col;
  put(0);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (i + 1 < NI) put(i + 1);
#pragma unroll
    for (int r = 0; r < 16; r += RP)
      if (there && r + r0 < 16 && row + i * 16 + r <= m_last) {
        floatx4 v = *(const floatx4 __attribute__((address_space(3)))*)(mine + (i & 1) * PIECE + (r + r0) * PITCH + lane % CPR * 16);
        if (NI * NJ == 64 && residual) v += *reinterpret_cast<const floatx4*>(residual + (size_t)(row + i * 16 + r) * n + col);
        *reinterpret_cast<floatx4*>(to + (size_t)(i * 16 + r) * n) = v;
      }
    asm volatile("" ::: "memory");
  }
}

// gemm_ring.hip: one of its tiles (codes 129, 97, 65, 48, 32, 16: 256 x 128, 192 x 192, 128 x 128, 64 x 128, 64 x 64, 32 x 32; 193, 130: rows by group, tiles by height with 192 and 128 columns), operands as the _supported functions of gemm_dma.hip check them.
hipError_t gemm_ring_launch(hipStream_t stream, int dtype, DmaForm form, const MMArgs& p, size_t batch, int tile, const float* residual, const DmaRows& rw);

}  // namespace ughip
