// Attention of many positions over keys and values in memory, the scores never leaving registers; shared by the kinds of attention
// that bring their operands into this form.
//   A wave owns 32 queries and, of every tile of 64 keys that comes through LDS, all of them or a half.  The scores are computed transposed, S^T = K Q^T
//   (32 x 32 tiles), which leaves lane l with query l % 32 as its column: the running maximum and sum are one exchange with lane
//   l ^ 32, and the weights sit where the second product, O^T = V^T P^T, wants its right operand (the order in which keys take
//   part in it is the order the accumulator layout gives; V is read in the same order).  Values come transposed for that.  Waves with
//   the same queries and other keys meet at the end.
//   bf16 operands: v_mfma_f32_32x32x16_bf16, a weight as two bf16 terms (16 bits of it); f32: v_mfma_f32_32x32x2_f32.
// bf16 heads of up to 192 elements: two groups of waves take every second tile of keys, by blocks of 128 queries, however many queries a workgroup has: a rounding in front of a product may turn a
// router's choice or a bf16 row's last bit, so the order of these sums stays.  Otherwise a wave has a half of every tile (or, f32 in one round of workgroups, a tile).
// What bounds it (bf16, 128 elements): the vector instructions of a wave's softmax and splits, 240 for 32 x 32 scores and 27 of 63 thousand cycles, 19 thousand of MFMA, and a wave's steps
// one behind the other.  us with the launch that places queries and keys (11 to 16), 128 queries to a workgroup, then 64 queries and two workgroups to a CU: 16 heads of 128 on 4, 509 / 1024 / 2048 positions 25.3 / 39.0 /
// 67.7 -> 21.6 / 33.3 / 59.9, 2048 behind a window of 1024 50.4 -> 50.9; 16 heads of 64 18.8 / 27.8 / 46.6 -> 16.8 / 24.3 / 42.6.  At 192 elements LDS has no room for two: 16 heads, 64 queries 30.6 / 46.3 / 86.5, 128 queries 33.3 /
// 50.1 / 83.9 and behind a window 64.6 for 84.8, so the larger blocks come where they leave no CU without one.
// Heads of 256 and f32, a whole tile to a wave (128 queries) and halves of it (64 queries): 8 heads of 256 in bf16, 509 / 2048 positions 50.4 / 151 -> 40.2 / 111, f32 176 / 634 -> 114 / 388; f32 16 heads
// of 128 85 / 301 -> 56 / 200, of 192 106 / 374 -> 70 / 251.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "bf16_split.h"
#include "layers.h"

namespace ughip {
namespace {  // every file that launches the kernel has its own

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Queries come times scale * log2(e): the weights are powers of two of the scores.  q [heads][q_rows][DQ], k [kv_heads][k_rows][DQ],
// v [kv_heads vdim][v_stride] (one row per value element, position along it); zeros past a query's and a key's last element and past
// the last query.
struct AttRowsArgs {
  const void* q;
  const void* k;
  const void* v;
  void* dst;
  size_t v_stride, dst_stride;
  int t, pos, vdim, q_rows, k_rows;
  int kv_heads;  // key head of query head h: h / (heads / kv_heads)
  int window;    // > 0: a position sees itself and the window - 1 positions in front of it
  bool dst_bf16;
  bool paired = false, whole = false;  // set by the launch; whole: vdim is DV, and four elements of a result's row lie aligned
};

template <typename T>
__device__ __forceinline__ T to_elem(float v) {
  if constexpr (sizeof(T) == 2) return bf16_rne(v);
  else return v;
}

template <typename T>
__device__ __forceinline__ void mfma_chunk(const u32x4_t& a, const u32x4_t& b, f32x16& acc) {
  if constexpr (sizeof(T) == 2) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
  } else {
    const f32x4_t x = __builtin_bit_cast(f32x4_t, a), y = __builtin_bit_cast(f32x4_t, b);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, y.x, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, y.y, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, y.z, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, y.w, acc, 0, 0, 0);
  }
}

constexpr int ATT_KT = 64, ATT_QT = 64;  // caches hold whole tiles of keys, queries' rows whole blocks of 64
template <typename T, int DQ, int DV>
constexpr int attention_rows_tile_bytes() {
  return ATT_KT * (DQ * (int)sizeof(T) + 16) + DV * (ATT_KT * (int)sizeof(T) + 16);
}
// How a workgroup's waves share its work.  QW of them have 32 queries each; with PARTS == 2 as many again have the same queries and the other part of the keys: every second tile (GROUPS == 2,
// a tile in LDS for either group), or the other half of every tile (HALVES).
template <typename T, int DQ, int DV, int GROUPS, int HALVES, int QW>
struct AttShape {
  static constexpr int PARTS = GROUPS * HALVES, THREADS = 64 * QW * PARTS, TILE = attention_rows_tile_bytes<T, DQ, DV>();
  // two to a CU where their waves' registers and their tiles' LDS allow it: one multiplies while the other has its softmax, and a long row may have a short one beside it
  static constexpr int PER_CU = THREADS <= 256 && (sizeof(T) == 2 ? DQ <= 192 && DV <= 128 : DQ <= 64) && 2 * GROUPS * TILE <= 160 * 1024 ? 2 : 1;
  static constexpr int WAVES = PER_CU * THREADS <= 256 ? 1 : 2;           // of a SIMD
  static constexpr bool TWICE = PER_CU * 2 * GROUPS * TILE <= 160 * 1024;  // a tile is there twice: the next one goes in while this one is multiplied
  static constexpr int LDS_BYTES = (TWICE ? 2 : 1) * GROUPS * TILE;
  static_assert(PARTS <= 2 && LDS_BYTES <= 160 * 1024, "the tiles fit LDS");
};

// o / sum of query i_mine: element e of block i of the lane's column lies at value element 32 i + 8 (e / 4) + 4 hf + e % 4
template <int DV>
__device__ __forceinline__ void attention_rows_out(const AttRowsArgs& a, int i_mine, int head, int hf, float sum, const f32x16 (&o)[DV / 32]) {
  if (i_mine >= a.t) return;
  const float inv = 1.f / sum;
  const size_t at = (size_t)i_mine * a.dst_stride + (size_t)head * a.vdim + 4 * hf;
  if (a.whole) {  // four elements of a row at a time (one by one, with a branch and two bytes each, a workgroup's result takes as long as three tiles of keys)
#pragma unroll
    for (int i = 0; i < DV / 32; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t v = f32x4_t{o[i][4 * q], o[i][4 * q + 1], o[i][4 * q + 2], o[i][4 * q + 3]} * inv;
        typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
        if (a.dst_bf16) *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.dst) + at + i * 32 + 8 * q) = __builtin_bit_cast(uint2, __builtin_convertvector(v, bf16x4));
        else *reinterpret_cast<f32x4_t*>(static_cast<float*>(a.dst) + at + i * 32 + 8 * q) = v;
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < DV / 32; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int vc = i * 32 + 8 * (e >> 2) + (e & 3);
      if (vc + 4 * hf < a.vdim) {
        if (a.dst_bf16) static_cast<uint16_t*>(a.dst)[at + vc] = bf16_rne(o[i][e] * inv);
        else static_cast<float*>(a.dst)[at + vc] = o[i][e] * inv;
      }
    }
}

// DQ >= dim + rot and DV >= vdim, the surplus is zeros.  T: uint16_t (bf16) or float.
template <typename T, int DQ, int DV, int GROUPS, int HALVES, int QW>
__global__ void __launch_bounds__((AttShape<T, DQ, DV, GROUPS, HALVES, QW>::THREADS), (AttShape<T, DQ, DV, GROUPS, HALVES, QW>::WAVES)) attention_rows_kernel(AttRowsArgs a) {
  typedef AttShape<T, DQ, DV, GROUPS, HALVES, QW> Shape;
  constexpr int E = 16 / sizeof(T), QC = DQ / E, K_ROW = DQ * sizeof(T) + 16, V_ROW = ATT_KT * sizeof(T) + 16, VC = ATT_KT / E;
  constexpr int GT = 64 * QW * HALVES, QT = 32 * QW, NK = ATT_KT * QC / GT, NV = DV * VC / GT;  // threads of a group, queries, 16-byte pieces of a tile per thread
  constexpr int STEP = GROUPS * ATT_KT, NB = 2 / HALVES, KW = 32 * NB;  // a wave's share of a tile: KW keys in blocks of 32
  constexpr bool TWICE = Shape::TWICE;
  // The next tile waits in registers while this one is multiplied.  With two waves to a SIMD they have to have room for it (16 heads of 128, 64 queries, 2048 positions: 79.7 us so, with spills, 59.9 without).
  constexpr bool AHEAD = Shape::WAVES == 2 ? 2 * QC + DV / 2 + 16 * NB + 4 * (NK + NV) < 192 : NK + NV <= 16 || GROUPS == 2;
  static_assert(ATT_KT * QC % GT == 0 && DV * VC % GT == 0, "whole pieces per thread");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int group = GROUPS == 1 ? 0 : threadIdx.x / GT, tid = threadIdx.x % GT;
  constexpr int TILE = Shape::TILE;
  char* const tiles = lds + group * (TWICE ? 2 : 1) * TILE;
  char* Ks = tiles;                // [ATT_KT][DQ]
  char* Vs = Ks + ATT_KT * K_ROW;  // [DV][ATT_KT]
  // consecutive workgroups (dealt round robin to the chip's eight parts) take different key heads: those that share one meet in a cache
  const int per = gridDim.x / a.kv_heads, kv = blockIdx.x % a.kv_heads, head = kv * per + blockIdx.x / a.kv_heads;
  // The longest rows first.  Where all workgroups are there at once, two to a CU, the second half of them goes from the shortest up: a long one has a short one beside it.
  const int ny = gridDim.y, half_y = (ny + 1) / 2, y = blockIdx.y, qb = a.paired && y >= half_y ? y - half_y : ny - 1 - y;
  const int lane = tid & 63, wave = tid >> 6, col = lane & 31, hf = lane >> 5, q_wave = wave % QW, half = HALVES == 1 ? 0 : wave / QW, part = GROUPS == 2 ? group : half;
  const int i_mine = qb * QT + q_wave * 32 + col, p_mine = a.pos + min(i_mine, a.t - 1);
  // the wave's queries as the right operand of S^T: chunk 2 c + hf of query `col` (past t any: nobody stores what comes of it)
  u32x4_t qf[QC / 2];
  {
    const char* qr = static_cast<const char*>(a.q) + ((size_t)head * a.q_rows + min(i_mine, a.q_rows - 1)) * DQ * sizeof(T) + hf * 16;
#pragma unroll
    for (int c = 0; c < QC / 2; ++c) qf[c] = *reinterpret_cast<const u32x4_t*>(qr + c * 32);
  }
  f32x16 o[DV / 32];
#pragma unroll
  for (int i = 0; i < DV / 32; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[i][e] = 0.f;
  float mx = -INFINITY, sum = 0.f;
  const int s_all = a.pos + a.t, last_q = min(a.t, (qb + 1) * QT), keys = a.pos + last_q, first_p = a.pos + qb * QT + q_wave * 32;
  auto window_begin = [&](int block) { return a.window ? max(0, a.pos + block - a.window + 1) / ATT_KT * ATT_KT : 0; };  // the first tile that a block of queries from there on sees
  const int k_begin = window_begin(qb * QT), oldest = a.window ? p_mine - a.window : -1;  // keys > oldest are seen
  // which of two tiles is a group's goes by blocks of 128 queries, so that the order of the sums does not depend on QW
  const int second = GROUPS == 1 ? 0 : (group ^ ((k_begin - window_begin(qb * QT / 128 * 128)) / ATT_KT & 1)) * ATT_KT;
  const char* k_head = static_cast<const char*>(a.k) + (size_t)kv * a.k_rows * DQ * sizeof(T);
  const T* v_head = static_cast<const T*>(a.v) + (size_t)kv * a.vdim * a.v_stride;
  u32x4_t kr[NK], vr[NV];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < NK; ++u) kr[u] = *reinterpret_cast<const u32x4_t*>(k_head + (size_t)k0 * DQ * sizeof(T) + (tid + u * GT) * 16);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      // rows are padded to whole tiles and 16-byte aligned; every lane loads (no branches between loads)
      const int x = tid + u * GT, vc = x / VC;
      vr[u] = *reinterpret_cast<const u32x4_t*>(v_head + (size_t)(vc < a.vdim ? vc : 0) * a.v_stride + k0 + x % VC * E);
    }
  };
  // what of a piece of values is none: columns past the last one, positions past the last one (never written)
  auto value_piece = [&](const u32x4_t& piece, int vc, int kp) {
    T v[E];
    __builtin_memcpy(v, &piece, 16);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = vc < a.vdim && kp + e < s_all ? v[e] : T(0);
    u32x4_t out;
    __builtin_memcpy(&out, v, 16);
    return out;
  };
  // (bf16: values are read by eight bytes of 32 rows at once, and the rows of a pitch of 36 banks meet every 16: the pieces of every second 16 rows lie with their halves swapped)
  constexpr bool SWAP = sizeof(T) == 2;
  auto place = [&](int k0, char* kt) {
    char* vt = kt + ATT_KT * K_ROW;
#pragma unroll
    for (int u = 0; u < NK; ++u) {
      const int x = tid + u * GT;
      *reinterpret_cast<u32x4_t*>(kt + x / QC * K_ROW + x % QC * 16) = kr[u];
    }
    const bool whole = k0 + ATT_KT <= s_all && DV == a.vdim;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int x = tid + u * GT;
      const u32x4_t piece = whole ? vr[u] : value_piece(vr[u], x / VC, k0 + x % VC * E);
      *reinterpret_cast<u32x4_t*>(vt + x / VC * V_ROW + x % VC * 16) = SWAP && (x / VC & 16) ? u32x4_t{piece.z, piece.w, piece.x, piece.y} : piece;
    }
  };
  if (AHEAD && k_begin + second < keys) fetch(k_begin + second);
  if constexpr (TWICE) {
    if (!AHEAD && k_begin + second < keys) fetch(k_begin + second);
    if (k_begin + second < keys) place(k_begin + second, tiles);
    if (AHEAD && k_begin + second + STEP < keys) fetch(k_begin + second + STEP);
  }
  for (int k0 = k_begin + second; k0 - second < keys; k0 += STEP) {
    const bool there = GROUPS == 1 || k0 < keys;  // (the last tile of an odd number is one group's alone)
    const int k_next = k0 + STEP;
    __syncthreads();  // (twice: this tile is there; either: the one before has been read)
    if constexpr (TWICE) {
      if (k_next < keys) {
        if (!AHEAD) fetch(k_next);
        place(k_next, tiles + (Ks == tiles ? TILE : 0));
        if (AHEAD && k_next + STEP < keys) fetch(k_next + STEP);
      }
    } else {
      if (there) {
        if (!AHEAD) fetch(k0);
        place(k0, tiles);
      }
      __syncthreads();
      if (AHEAD && k_next < keys) fetch(k_next);
    }
    const char* const Kc = Ks + half * KW * K_ROW;
    const char* const Vc = Vs + half * KW * sizeof(T);
    if constexpr (TWICE) Ks = Ks == tiles ? tiles + TILE : tiles, Vs = Ks + ATT_KT * K_ROW;
    if (!there) continue;
    const int kw = k0 + half * KW;
    if ((HALVES == 2 && kw >= keys) || kw > first_p + 31 || (a.window && kw + KW - 1 <= first_p - a.window)) continue;  // nothing in it is visible to the wave's queries
    f32x16 s[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[b][e] = 0.f;
#pragma unroll
    for (int c = 0; c < QC / 2; ++c)
#pragma unroll
      for (int b = 0; b < NB; ++b) mfma_chunk<T>(*reinterpret_cast<const u32x4_t*>(Kc + (b * 32 + col) * K_ROW + hf * 16 + c * 32), qf[c], s[b]);
    // element e of s[b]: key kw + 32 b + 8 (e / 4) + 4 hf + e % 4, query `col`
    float top = mx;
    if (kw + KW - 1 > first_p || (a.window && kw <= first_p + 31 - a.window)) {  // some keys are not visible to some of the wave's queries
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = kw + 32 * b + 8 * (e >> 2) + 4 * hf + (e & 3);
          s[b][e] = key <= p_mine && key > oldest ? s[b][e] : -INFINITY;
        }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) top = fmaxf(top, s[b][e]);
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    // the weights' base follows the maximum only when that has left it well behind: up to 2^8 they lose nothing
    const bool behind = top > mx + 8.f;
    if (__any(behind)) {
      const float alpha = !behind ? 1.f : HALVES == 2 ? __builtin_amdgcn_exp2f(mx - top) : exp2f(mx - top);
      sum *= alpha;
#pragma unroll
      for (int i = 0; i < DV / 32; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] *= alpha;
      mx = behind ? top : mx;
    }
    const float base = mx == -INFINITY ? 0.f : mx;
    float part_sum = 0.f;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[b][e] = __builtin_amdgcn_exp2f(s[b][e] - base);
        part_sum += s[b][e];
      }
    sum += HALVES == 2 ? part_sum : part_sum + __shfl_xor(part_sum, 32, 64);  // (of halves the half-waves' sums meet at the end)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if constexpr (sizeof(T) == 2) {
        const int swap = (col & 16) >> 1;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          u32x4_t h, l;  // two terms of every weight, two at a time
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float w0 = s[b][8 * u + 2 * e], w1 = s[b][8 * u + 2 * e + 1];
            h[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(split_f32x2{w0, w1}, split_bf16x2));
            l[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(split_f32x2{w0 - __uint_as_float(h[e] << 16), w1 - __uint_as_float(h[e] & 0xffff0000u)}, split_bf16x2));
          }
          const bf16x8 hi = __builtin_bit_cast(bf16x8, h), lo = __builtin_bit_cast(bf16x8, l);
          bf16x8 vf[DV / 32];
#pragma unroll
          for (int i = 0; i < DV / 32; ++i) {
            const char* at = Vc + (i * 32 + col) * V_ROW + b * 64 + u * 32;
            const uint2 v0 = *reinterpret_cast<const uint2*>(at + ((8 * hf) ^ swap)), v1 = *reinterpret_cast<const uint2*>(at + 16 + ((8 * hf) ^ swap));
            vf[i] = __builtin_bit_cast(bf16x8, u32x4_t{v0.x, v0.y, v1.x, v1.y});
          }
#pragma unroll
          for (int i = 0; i < DV / 32; ++i) o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i], hi, o[i], 0, 0, 0);
#pragma unroll
          for (int i = 0; i < DV / 32; ++i) o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i], lo, o[i], 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < DV / 32; ++i) {
            const f32x4_t v = *reinterpret_cast<const f32x4_t*>(Vc + (i * 32 + col) * V_ROW + (b * 32 + 8 * u + 4 * hf) * 4);
            o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.x, s[b][4 * u], o[i], 0, 0, 0);
            o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.y, s[b][4 * u + 1], o[i], 0, 0, 0);
            o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.z, s[b][4 * u + 2], o[i], 0, 0, 0);
            o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.w, s[b][4 * u + 3], o[i], 0, 0, 0);
          }
      }
    }
  }
  if constexpr (HALVES == 2) sum += __shfl_xor(sum, 32, 64);
  if constexpr (Shape::PARTS == 2) {  // the two parts of the keys meet
    constexpr int N = DV / 32 * 4;
    static_assert(QW * 64 * (N * 16 + 8) <= Shape::LDS_BYTES, "a part's results fit where the tiles were");
    f32x4_t* other = reinterpret_cast<f32x4_t*>(lds) + q_wave * N * 64 + lane;
    float* ms = reinterpret_cast<float*>(lds + QW * 64 * N * 16) + (q_wave * 64 + lane) * 2;
    __syncthreads();
    if (part == 1) {
#pragma unroll
      for (int i = 0; i < DV / 32; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) other[(i * 4 + q) * 64] = f32x4_t{o[i][4 * q], o[i][4 * q + 1], o[i][4 * q + 2], o[i][4 * q + 3]};
      ms[0] = mx, ms[1] = sum;
    }
    __syncthreads();
    if (part == 1) return;
    const float m2 = ms[0], s2 = ms[1], top = fmaxf(mx, m2), base = top == -INFINITY ? 0.f : top, f1 = exp2f(mx - base), f2 = exp2f(m2 - base);
    sum = f1 * sum + f2 * s2;
#pragma unroll
    for (int i = 0; i < DV / 32; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t v = other[(i * 4 + q) * 64];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[i][4 * q + e] = f1 * o[i][4 * q + e] + f2 * v[e];
      }
  }
  attention_rows_out<DV>(a, i_mine, head, hf, sum, o);
}

template <typename T, int DQ, int DV, int GROUPS, int HALVES, int QW>
hipError_t attention_rows_launch_as(ughip_device* dev, AttRowsArgs a, int heads) {
  typedef AttShape<T, DQ, DV, GROUPS, HALVES, QW> Shape;
  auto kernel = attention_rows_kernel<T, DQ, DV, GROUPS, HALVES, QW>;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, Shape::LDS_BYTES);
  if (attr != hipSuccess) return attr;
  const int blocks = (a.t + 32 * QW - 1) / (32 * QW);
  const size_t all = (size_t)heads * blocks, cus = (size_t)dev->num_cus;
  a.paired = Shape::PER_CU == 2 && all <= 2 * cus && all > cus && !a.window;
  kernel<<<dim3((unsigned)heads, (unsigned)blocks), Shape::THREADS, Shape::LDS_BYTES, dev->stream>>>(a);
  return hipGetLastError();
}

// Tiles of keys that the workgroup of the last but n-th block of queries goes through
inline int attention_rows_tiles(const AttRowsArgs& a, int block, int n) {
  const int q0 = std::max(0, (a.t + block - 1) / block - 1 - n) * block, last = a.pos + std::min(a.t, q0 + block);
  return (last + ATT_KT - 1) / ATT_KT - (a.window ? std::max(0, a.pos + q0 - a.window + 1) / ATT_KT : 0);
}
// What the busiest CU of up to two rounds goes through, the longest rows first: the longest by itself, or the shortest of the first round and the longest of the second
inline int attention_rows_busiest(const AttRowsArgs& a, int block, int heads, int cus) {
  const int longest = attention_rows_tiles(a, block, 0);
  if ((size_t)heads * ((a.t + block - 1) / block) <= (size_t)cus) return longest;
  return std::max(longest, attention_rows_tiles(a, block, (cus - 1) / heads) + attention_rows_tiles(a, block, cus / heads));
}

// heads x blocks of queries; q_rows a multiple of ATT_QT
template <typename T, int DQ, int DV>
hipError_t attention_rows_launch(ughip_device* dev, AttRowsArgs a, int heads) {
  a.whole = a.vdim == DV && a.dst_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(a.dst) & (a.dst_bf16 ? 7 : 15)) == 0;
  const size_t blocks = ((size_t)a.t + 127) / 128, cus = (size_t)dev->num_cus;
  if constexpr (sizeof(T) == 2 && DQ <= 192 && DV <= 128) {
    if constexpr (DQ == 192)
      if (heads * blocks >= cus) return attention_rows_launch_as<T, DQ, DV, 2, 1, 4>(dev, a, heads);
    return attention_rows_launch_as<T, DQ, DV, 2, 1, 2>(dev, a, heads);
  } else {
    // Halves of tiles and 64 queries, at 0.59 of the time of a whole tile with 128, unless those are one round and a window makes most rows as long: 16 heads over 2048 positions behind a window of 1024, 18 tiles against 17 + 16
    // halves, us on halves and on whole tiles: f32 of 128 / 192 / 256 elements 193 / 243 / 432 and 183 / 228 / 395, bf16 of 256 133 and 113.  Over 1900 positions 178 and 184, without a window 199 and 302.
    if constexpr (DQ >= 128)
      if (heads * blocks <= cus && attention_rows_busiest(a, 128, heads, dev->num_cus) < 0.59 * attention_rows_busiest(a, 64, heads, dev->num_cus))
        return attention_rows_launch_as<T, DQ, DV, 1, 1, 4>(dev, a, heads);
    return attention_rows_launch_as<T, DQ, DV, 1, 2, 2>(dev, a, heads);
  }
}
}  // namespace
}  // namespace ughip
