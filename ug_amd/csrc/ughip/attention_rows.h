// Attention of many positions over keys and values in memory, the scores never leaving registers; shared by the kinds of attention
// that bring their operands into this form.
//   A workgroup owns 64 queries, a wave 32 of them and half of the keys of every tile of 64, which come through LDS.  The scores are computed transposed, S^T = K Q^T
//   (32 x 32 tiles), which leaves lane l with query l % 32 as its column: the running maximum and sum are one exchange with lane
//   l ^ 32, and the weights sit where the second product, O^T = V^T P^T, wants its right operand (the order in which keys take
//   part in it is the order the accumulator layout gives; V is read in the same order).  Values come transposed for that.  The
//   halves of the keys meet at the end.
//   bf16 operands: v_mfma_f32_32x32x16_bf16, a weight as two bf16 terms (16 bits of it); f32: v_mfma_f32_32x32x2_f32.
// What bounds it (bf16, 128 elements): the vector instructions of a wave's softmax and splits, 240 for 32 x 32 scores and 27 of 63 thousand cycles, 19 thousand of MFMA, and a wave's steps
// one behind the other.  Workgroups of 128 queries and two groups of waves in step (one to a CU) had long rows on CUs of their own and left their results two bytes at a time:
// us, then and now: 16 heads of 128 on 4 over 2048 positions, mean of a full one and two windows of 1024, 49.1 -> 43.1, 509 positions 23.1 -> 15.9, f32 77 -> 46; 16 heads of 192 / 128
// over 2048 / 509 positions 69 -> 58 / 25.8 -> 17.2, f32 93.6 -> 55.8.  Tiles of 128 keys, 64 to a wave (as many registers as there are): 43.4 and 18.6 for the first two.
#pragma once
#include <hip/hip_runtime.h>

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

constexpr int ATT_KT = 64, ATT_QT = 64;  // caches hold whole tiles of keys
// A tile's bytes, and whether it is there twice: the next one goes in while this one is multiplied.  Two workgroups to a CU come first: their waves are at different
// places, so that one multiplies while the other has its softmax.
template <typename T, int DQ, int DV>
constexpr int attention_rows_tile_bytes() {
  return ATT_KT * (DQ * (int)sizeof(T) + 16) + DV * (ATT_KT * (int)sizeof(T) + 16);
}
template <typename T, int DQ, int DV>
constexpr int attention_rows_per_cu() {  // as the registers of a wave allow
  return (sizeof(T) == 2 ? DQ <= 192 && DV <= 128 : DQ <= 64) ? 2 : 1;
}
template <typename T, int DQ, int DV>
constexpr bool attention_rows_twice() {
  return attention_rows_per_cu<T, DQ, DV>() * 2 * attention_rows_tile_bytes<T, DQ, DV>() <= 160 * 1024;
}
template <typename T, int DQ, int DV>
constexpr int attention_rows_lds_bytes() {
  return (attention_rows_twice<T, DQ, DV>() ? 2 : 1) * attention_rows_tile_bytes<T, DQ, DV>();
}

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
template <typename T, int DQ, int DV>
__global__ void __launch_bounds__(256, (attention_rows_per_cu<T, DQ, DV>())) attention_rows_kernel(AttRowsArgs a) {
  constexpr int E = 16 / sizeof(T), QC = DQ / E, K_ROW = DQ * sizeof(T) + 16, V_ROW = ATT_KT * sizeof(T) + 16, VC = ATT_KT / E;
  constexpr int NK = ATT_KT * QC / 256, NV = DV * VC / 256;  // 16-byte pieces of a tile per thread
  constexpr bool AHEAD = NK + NV <= 16;                  // the next tile waits in registers while this one is multiplied
  static_assert(ATT_KT * QC % 256 == 0 && DV * VC % 256 == 0, "whole pieces per thread");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x;
  constexpr int TILE = attention_rows_tile_bytes<T, DQ, DV>();
  constexpr bool TWICE = attention_rows_twice<T, DQ, DV>();
  char* Ks = lds;                  // [ATT_KT][DQ]
  char* Vs = Ks + ATT_KT * K_ROW;  // [DV][ATT_KT]
  // consecutive workgroups (dealt round robin to the chip's eight parts) take different key heads: those that share one meet in a cache
  const int per = gridDim.x / a.kv_heads, kv = blockIdx.x % a.kv_heads, head = kv * per + blockIdx.x / a.kv_heads;
  // The longest rows first.  Where all workgroups are there at once, two to a CU, the second half of them goes from the shortest up: a long one has a short one beside it.
  const int ny = gridDim.y, half = (ny + 1) / 2, y = blockIdx.y, qb = a.paired && y >= half ? y - half : ny - 1 - y;
  const int lane = tid & 63, wave = tid >> 6, col = lane & 31, hf = lane >> 5, q_half = wave & 1, k_half = wave >> 1;
  const int i_mine = qb * ATT_QT + q_half * 32 + col, p_mine = a.pos + min(i_mine, a.t - 1);
  // the wave's queries as the right operand of S^T: chunk 2 c + hf of query `col` (rows up to q_rows exist, zeros past t)
  u32x4_t qf[QC / 2];
  {
    const char* qr = static_cast<const char*>(a.q) + ((size_t)head * a.q_rows + i_mine) * DQ * sizeof(T) + hf * 16;
#pragma unroll
    for (int c = 0; c < QC / 2; ++c) qf[c] = *reinterpret_cast<const u32x4_t*>(qr + c * 32);
  }
  f32x16 o[DV / 32];
#pragma unroll
  for (int i = 0; i < DV / 32; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[i][e] = 0.f;
  float mx = -INFINITY, sum = 0.f;
  const int s_all = a.pos + a.t, last_q = min(a.t, (qb + 1) * ATT_QT), keys = a.pos + last_q, first_p = a.pos + qb * ATT_QT + q_half * 32;
  const int k_begin = a.window ? max(0, a.pos + qb * ATT_QT - a.window + 1) / ATT_KT * ATT_KT : 0, oldest = a.window ? p_mine - a.window : -1;  // keys > oldest are seen
  const char* k_head = static_cast<const char*>(a.k) + (size_t)kv * a.k_rows * DQ * sizeof(T);
  const T* v_head = static_cast<const T*>(a.v) + (size_t)kv * a.vdim * a.v_stride;
  u32x4_t kr[NK], vr[NV];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < NK; ++u) kr[u] = *reinterpret_cast<const u32x4_t*>(k_head + (size_t)k0 * DQ * sizeof(T) + (tid + u * 256) * 16);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      // rows are padded to whole tiles and 16-byte aligned; every lane loads (no branches between loads)
      const int x = tid + u * 256, vc = x / VC;
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
      const int x = tid + u * 256;
      *reinterpret_cast<u32x4_t*>(kt + x / QC * K_ROW + x % QC * 16) = kr[u];
    }
    const bool whole = k0 + ATT_KT <= s_all && DV == a.vdim;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int x = tid + u * 256;
      const u32x4_t piece = whole ? vr[u] : value_piece(vr[u], x / VC, k0 + x % VC * E);
      *reinterpret_cast<u32x4_t*>(vt + x / VC * V_ROW + x % VC * 16) = SWAP && (x / VC & 16) ? u32x4_t{piece.z, piece.w, piece.x, piece.y} : piece;
    }
  };
  if (AHEAD) fetch(k_begin);
  if constexpr (TWICE) {
    if (!AHEAD) fetch(k_begin);
    place(k_begin, lds);
    if (AHEAD && k_begin + ATT_KT < keys) fetch(k_begin + ATT_KT);
  }
  constexpr int KW = ATT_KT / 2;  // a wave's share of a tile
  for (int k0 = k_begin; k0 < keys; k0 += ATT_KT) {
    const int k_next = k0 + ATT_KT;
    __syncthreads();  // (twice: this tile is there; either: the one before has been read)
    if constexpr (TWICE) {
      if (k_next < keys) {
        if (!AHEAD) fetch(k_next);
        place(k_next, lds + (Ks == lds ? TILE : 0));
        if (AHEAD && k_next + ATT_KT < keys) fetch(k_next + ATT_KT);
      }
    } else {
      if (!AHEAD) fetch(k0);
      place(k0, lds);
      __syncthreads();
      if (AHEAD && k_next < keys) fetch(k_next);
    }
    const char* const Kc = Ks + k_half * KW * K_ROW;
    const char* const Vc = Vs;
    if constexpr (TWICE) Ks = Ks == lds ? lds + TILE : lds, Vs = Ks + ATT_KT * K_ROW;
    const int kw = k0 + k_half * KW;
    if (kw >= keys || kw > first_p + 31 || (a.window && kw + KW - 1 <= first_p - a.window)) continue;  // nothing in it is visible to the wave's queries
    // bf16: the sums start at minus the weights' base (a subtraction less for every score; in f32 that would round them at the base's size)
    constexpr bool FROM_BASE = sizeof(T) == 2;
    float base = mx == -INFINITY ? 0.f : mx;
    const float start = FROM_BASE ? -base : 0.f;
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = start;
#pragma unroll
    for (int c = 0; c < QC / 2; ++c) mfma_chunk<T>(*reinterpret_cast<const u32x4_t*>(Kc + col * K_ROW + hf * 16 + c * 32), qf[c], s);
    // element e: key kw + 8 (e / 4) + 4 hf + e % 4, query `col`
    if (kw + KW - 1 > first_p || (a.window && kw <= first_p + 31 - a.window)) {  // some keys are not visible to some of the wave's queries
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int key = kw + 8 * (e >> 2) + 4 * hf + (e & 3);
        s[e] = key <= p_mine && key > oldest ? s[e] : -INFINITY;
      }
    }
    float top = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; ++e) top = fmaxf(top, s[e]);
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    if (!FROM_BASE) top -= base;
    // the weights' base follows the maximum only when that has left it well behind: up to 2^8 they lose nothing
    const bool behind = top > (mx == -INFINITY ? -INFINITY : 8.f);
    if (__any(behind)) {
      const float now = behind ? base + top : base, by = now - base, alpha = mx == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(-by);
      sum *= alpha;
#pragma unroll
      for (int i = 0; i < DV / 32; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] *= alpha;
      if constexpr (FROM_BASE) {
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] -= by;
      }
      base = now;
      mx = behind ? now : mx;
    }
    float part = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s[e] = __builtin_amdgcn_exp2f(FROM_BASE ? s[e] : s[e] - base);
      part += s[e];
    }
    sum += part;  // (the half-waves' parts meet at the end)
    if constexpr (sizeof(T) == 2) {
      const char* const p = Vc + col * V_ROW + k_half * KW * 2;
      const int swap = (col & 16) >> 1;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        u32x4_t h, l;  // two terms of every weight, two at a time
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float w0 = s[8 * u + 2 * e], w1 = s[8 * u + 2 * e + 1];
          h[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(split_f32x2{w0, w1}, split_bf16x2));
          l[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(split_f32x2{w0 - __uint_as_float(h[e] << 16), w1 - __uint_as_float(h[e] & 0xffff0000u)}, split_bf16x2));
        }
        const bf16x8 hi = __builtin_bit_cast(bf16x8, h), lo = __builtin_bit_cast(bf16x8, l);
        bf16x8 vf[DV / 32];
#pragma unroll
        for (int i = 0; i < DV / 32; ++i) {
          const char* at = p + i * 32 * V_ROW + u * 32;
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
          const f32x4_t v = *reinterpret_cast<const f32x4_t*>(Vc + (i * 32 + col) * V_ROW + (k_half * KW + 8 * u + 4 * hf) * 4);
          o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.x, s[4 * u], o[i], 0, 0, 0);
          o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.y, s[4 * u + 1], o[i], 0, 0, 0);
          o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.z, s[4 * u + 2], o[i], 0, 0, 0);
          o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v.w, s[4 * u + 3], o[i], 0, 0, 0);
        }
    }
  }
  sum += __shfl_xor(sum, 32, 64);
  // the two halves of the keys meet
  constexpr int N = DV / 32 * 4;
  static_assert(2 * 64 * (N * 16 + 8) <= attention_rows_lds_bytes<T, DQ, DV>(), "the results of two waves fit where the tiles were");
  f32x4_t* other = reinterpret_cast<f32x4_t*>(lds) + q_half * N * 64 + lane;
  float* ms = reinterpret_cast<float*>(lds + 2 * 64 * N * 16) + (q_half * 64 + lane) * 2;
  __syncthreads();
  if (k_half == 1) {
#pragma unroll
    for (int i = 0; i < DV / 32; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) other[(i * 4 + q) * 64] = f32x4_t{o[i][4 * q], o[i][4 * q + 1], o[i][4 * q + 2], o[i][4 * q + 3]};
    ms[0] = mx, ms[1] = sum;
  }
  __syncthreads();
  if (k_half == 1) return;
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
  attention_rows_out<DV>(a, i_mine, head, hf, sum, o);
}

// bf16 keys of 192 elements, as routed models have them: two groups of QW waves with 32 queries each take every second tile of keys.  Their sums stay in this order, whatever QW: a rounding
// in front of a router may turn a choice of experts.  LDS holds a tile for each group once, so that a CU has one workgroup: of 128 queries, or of 64 where those would leave CUs without one
// (16 heads, us with results two bytes at a time and so: 509 positions 25.8 -> 18.7, 1200 positions 43.7 -> 37.9, 2048 on 128 queries 69 -> 65; sums in the other kernel's order would be 17.3 and 57).
template <typename T, int DQ, int DV, int QW>
__global__ void __launch_bounds__(128 * QW) attention_rows_pairs_kernel(AttRowsArgs a) {
  constexpr int E = 16 / sizeof(T), QC = DQ / E, K_ROW = DQ * sizeof(T) + 16, V_ROW = ATT_KT * sizeof(T) + 16, VC = ATT_KT / E;
  constexpr int GT = 64 * QW, QT = 32 * QW, NK = ATT_KT * QC / GT, NV = DV * VC / GT;  // threads of a group, queries, 16-byte pieces of a tile per thread
  static_assert(ATT_KT * QC % GT == 0 && DV * VC % GT == 0 && sizeof(T) == 2, "whole pieces per thread");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int GROUPS = 2, TILE = attention_rows_tile_bytes<T, DQ, DV>();
  const int group = threadIdx.x / GT, tid = threadIdx.x % GT;
  char* const Ks = lds + group * TILE;   // [ATT_KT][DQ]
  char* const Vs = Ks + ATT_KT * K_ROW;  // [DV][ATT_KT]
  // consecutive workgroups (dealt round robin to the chip's eight parts) take different key heads: those that share one meet in a cache
  const int per = gridDim.x / a.kv_heads, kv = blockIdx.x % a.kv_heads, head = kv * per + blockIdx.x / a.kv_heads;
  const int qb = gridDim.y - 1 - blockIdx.y;  // the longest rows first
  const int lane = tid & 63, wave = tid >> 6, col = lane & 31, hf = lane >> 5;
  const int i_mine = qb * QT + wave * 32 + col, p_mine = a.pos + min(i_mine, a.t - 1);
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
  const int s_all = a.pos + a.t, last_q = min(a.t, (qb + 1) * QT), keys = a.pos + last_q, first_p = a.pos + qb * QT + wave * 32;
  const int k_begin = a.window ? max(0, a.pos + qb * QT - a.window + 1) / ATT_KT * ATT_KT : 0, oldest = a.window ? p_mine - a.window : -1;  // keys > oldest are seen
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
  const int k_mine = k_begin + group * ATT_KT;
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
      *reinterpret_cast<u32x4_t*>(vt + x / VC * V_ROW + x % VC * 16) = x / VC & 16 ? u32x4_t{piece.z, piece.w, piece.x, piece.y} : piece;  // (as in attention_rows_kernel)
    }
  };
  if (k_mine < keys) fetch(k_mine);
  for (int k0 = k_mine; k0 - group * ATT_KT < keys; k0 += GROUPS * ATT_KT) {
    const bool there = k0 < keys;  // (the last tile of an odd number is the first group's alone)
    const int k_next = k0 + GROUPS * ATT_KT;
    __syncthreads();
    if (there) place(k0, Ks);
    __syncthreads();
    if (k_next < keys) fetch(k_next);
    if (!there) continue;
    if (k0 > first_p + 31 || (a.window && k0 + ATT_KT - 1 <= first_p - a.window)) continue;  // nothing in this tile is visible to the wave's queries
    f32x16 s[2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) s[b][e] = 0.f;
#pragma unroll
    for (int c = 0; c < QC / 2; ++c)
#pragma unroll
      for (int b = 0; b < 2; ++b) mfma_chunk<T>(*reinterpret_cast<const u32x4_t*>(Ks + (b * 32 + col) * K_ROW + hf * 16 + c * 32), qf[c], s[b]);
    // element e of s[b]: key k0 + 32 b + 8 (e / 4) + 4 hf + e % 4, query `col`
    float top = mx;
    if (k0 + ATT_KT - 1 > first_p || (a.window && k0 <= first_p + 31 - a.window)) {  // some keys of the tile are not visible to some of the wave's queries
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = k0 + 32 * b + 8 * (e >> 2) + 4 * hf + (e & 3);
          s[b][e] = key <= p_mine && key > oldest ? s[b][e] : -INFINITY;
        }
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) top = fmaxf(top, s[b][e]);
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    // the weights' base follows the maximum only when that has left it well behind: up to 2^8 they lose nothing
    const bool behind = top > mx + 8.f;
    if (__any(behind)) {
      const float alpha = behind ? exp2f(mx - top) : 1.f;
      sum *= alpha;
#pragma unroll
      for (int i = 0; i < DV / 32; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[i][e] *= alpha;
      mx = behind ? top : mx;
    }
    const float base = mx == -INFINITY ? 0.f : mx;
    float part = 0.f;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        s[b][e] = __builtin_amdgcn_exp2f(s[b][e] - base);
        part += s[b][e];
      }
    sum += part + __shfl_xor(part, 32, 64);
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int swap = (col & 16) >> 1;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        u32x4_t h, l;
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
          const char* at = Vs + (i * 32 + col) * V_ROW + b * 64 + u * 32;
          const uint2 v0 = *reinterpret_cast<const uint2*>(at + ((8 * hf) ^ swap)), v1 = *reinterpret_cast<const uint2*>(at + 16 + ((8 * hf) ^ swap));
          vf[i] = __builtin_bit_cast(bf16x8, u32x4_t{v0.x, v0.y, v1.x, v1.y});
        }
#pragma unroll
        for (int i = 0; i < DV / 32; ++i) o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i], hi, o[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < DV / 32; ++i) o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i], lo, o[i], 0, 0, 0);
      }
    }
  }
  constexpr int N = DV / 32 * 4;
  static_assert(QW * 64 * (N * 16 + 8) <= 2 * TILE, "a group's results fit where the tiles were");
  f32x4_t* other = reinterpret_cast<f32x4_t*>(lds) + wave * N * 64 + lane;
  float* ms = reinterpret_cast<float*>(lds + QW * 64 * N * 16) + (wave * 64 + lane) * 2;
  __syncthreads();
  if (group == 1) {
#pragma unroll
    for (int i = 0; i < DV / 32; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) other[(i * 4 + q) * 64] = f32x4_t{o[i][4 * q], o[i][4 * q + 1], o[i][4 * q + 2], o[i][4 * q + 3]};
    ms[0] = mx, ms[1] = sum;
  }
  __syncthreads();
  if (group == 1) return;
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
  attention_rows_out<DV>(a, i_mine, head, hf, sum, o);
}

// heads x blocks of queries; q_rows a multiple of ATT_QT
template <typename T, int DQ, int DV>
hipError_t attention_rows_single_launch(ughip_device* dev, AttRowsArgs a, int heads) {
  constexpr int bytes = attention_rows_lds_bytes<T, DQ, DV>();
  static_assert(bytes <= 160 * 1024, "tile does not fit LDS");
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_rows_kernel<T, DQ, DV>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (attr != hipSuccess) return attr;
  const int blocks = a.q_rows / ATT_QT;
  a.paired = attention_rows_per_cu<T, DQ, DV>() == 2 && (size_t)heads * blocks <= 2 * (size_t)dev->num_cus && (size_t)heads * blocks > (size_t)dev->num_cus && !a.window;
  attention_rows_kernel<T, DQ, DV><<<dim3((unsigned)heads, (unsigned)blocks), 256, bytes, dev->stream>>>(a);
  return hipGetLastError();
}
template <typename T, int DQ, int DV, int QW>
hipError_t attention_rows_pairs_launch(ughip_device* dev, const AttRowsArgs& a, int heads) {
  constexpr int bytes = 2 * attention_rows_tile_bytes<T, DQ, DV>();
  static_assert(bytes <= 160 * 1024, "tiles do not fit LDS");
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_rows_pairs_kernel<T, DQ, DV, QW>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (attr != hipSuccess) return attr;
  attention_rows_pairs_kernel<T, DQ, DV, QW><<<dim3((unsigned)heads, (unsigned)((a.t + 32 * QW - 1) / (32 * QW))), 128 * QW, bytes, dev->stream>>>(a);
  return hipGetLastError();
}
template <typename T, int DQ, int DV>
hipError_t attention_rows_launch(ughip_device* dev, AttRowsArgs a, int heads) {
  a.whole = a.vdim == DV && a.dst_stride % 4 == 0 && (reinterpret_cast<uintptr_t>(a.dst) & (a.dst_bf16 ? 7 : 15)) == 0;
  if constexpr (sizeof(T) == 2 && DQ == 192)
    return (size_t)heads * ((a.t + 127) / 128) < (size_t)dev->num_cus ? attention_rows_pairs_launch<T, DQ, DV, 2>(dev, a, heads) : attention_rows_pairs_launch<T, DQ, DV, 4>(dev, a, heads);
  else return attention_rows_single_launch<T, DQ, DV>(dev, a, heads);
}
}  // namespace
}  // namespace ughip
