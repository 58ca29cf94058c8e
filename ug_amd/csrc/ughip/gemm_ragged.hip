// MFMA GEMM for operands that no tuned kernel takes -- any M, N and K, rows that start at any element -- with f32 accumulate: f32, f16, bf16;
// each operand contiguous along k or along its other dimension.
//
//   64 x 64 or 128 x 128 tiles, four waves 2 x 2, 32 x 32 MFMA blocks (and 32 x 32 tiles: gemm_ragged32).  A K step is 128 bytes of a k-contiguous row, 8 chunks of 16 bytes,
//   fetched by 16-byte loads at whatever address the row has (the hardware takes any) two steps ahead into registers, then written to one of
//   two LDS buffers: k-contiguous operands as rows of k, the others as they lie, and the waves read those back transposed
//   (ds_read_b64_tr_b16; f32 element by element).  The last step, K's remainder or a whole one, comes first, under the way of the next ones: the
//   elements in front of K's end by vectors, with zeros for those that belong to the step before (a K of less than one step: element by element). It
//   holds the only row of a [k, n]-major operand behind which nothing may be read.
//
// What bounds it: the steps of K on few tiles (0.2 us each in 16 bits with operands in L2 and 0.3 past it, a CU's share of the caches; 0.6 in f32, the f32 matrix pipe two thirds of that; four steps ahead, or a
// tile's waves each on a part of K, change nothing), LDS and the f32
// matrix pipe on many.  Against element-by-element
// loads between two barriers per 32 k (f32: 16), one box: 1000 x 777 x 1531 f16 196 -> 11.9 us (11.2 with chunks put together from words, Side), f32 256 -> 32; 2001^3 f16 270 -> 33, f32 340 -> 139; 3999^2 x
// 2000 f16 1204 -> 103, f32 1014 -> 520; 100^3 9.4 -> 6.0.  Which tile takes what and where K is split: gemm_ragged_plan.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "gemm.h"
#include "ughip.h"

namespace ughip {
namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// vectors at the address of any element
typedef u32x4 u32x4_at2 __attribute__((aligned(2)));
typedef u32x4 u32x4_at4 __attribute__((aligned(4)));
typedef u32x2 u32x2_at2 __attribute__((aligned(2)));
typedef f32x4 f32x4_at4 __attribute__((aligned(4)));
__device__ __forceinline__ u32x4 load16(const float* p) { return *reinterpret_cast<const u32x4_at4*>(p); }
template <typename T>
__device__ __forceinline__ u32x4 load16(const T* p) {
  return *reinterpret_cast<const u32x4_at2*>(p);
}
__device__ __forceinline__ void store4(float* p, const f32x4& v) { *reinterpret_cast<f32x4_at4*>(p) = v; }
template <typename T>
__device__ __forceinline__ void store4(T* p, const f32x4& v) {
  typedef T tx4 __attribute__((ext_vector_type(4)));
  *reinterpret_cast<u32x2_at2*>(p) = __builtin_bit_cast(u32x2, __builtin_convertvector(v, tx4));
}

__device__ __forceinline__ void mma(__bf16, const u32x4& a, const u32x4& b, f32x16& c) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ void mma(_Float16, const u32x4& a, const u32x4& b, f32x16& c) {
  c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ void mma(float, const u32x4& a, const u32x4& b, f32x16& c) {
  const f32x4 fa = __builtin_bit_cast(f32x4, a), fb = __builtin_bit_cast(f32x4, b);
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], c, 0, 0, 0);  // lanes 0-31 the even chunk's k, 32-63 the odd one's
}

// One operand's share of a workgroup's tile: `rows` (M or N) times k.  KC: contiguous along k.
// ODD (16 bits, KC): rows may start in the middle of a 4-byte word.  A 16-byte load there keeps a CU's address unit busy for 67 cycles, 44 in the mean where every
// second row does, and 27 at any word (22 at 16 bytes; 256 workgroups, tiles in L2).  So chunks are loaded from the word behind a row's start on and put together
// from two words each: the element in front is the last one of the chunk before, the lane below's or, for a row's first chunk, of the step before (`carry`).  A step
// reads one element past its end, which is there: K's last elements are load_end's.  f16 1000 x 776 x 2057, both operands so, 15.3 -> 13.4 us.
template <typename T, int B, bool KC, int THREADS = 256, bool ODD = false>
struct Side {
  static_assert(!ODD || (KC && sizeof(T) == 2));
  static constexpr int E = 16 / sizeof(T), KE = 8 * E;           // elements per chunk, k per step
  static constexpr int CPR = KC ? 8 : B / E;                     // chunks per row in LDS (a row: of k, or of the operand's rows at one k)
  static constexpr int PITCH = CPR * 16 + 16, LDS_ROWS = KC ? B : KE, BYTES = LDS_ROWS * PITCH;
  static constexpr int N = LDS_ROWS * CPR / THREADS;             // chunks per thread
  const T* at[N];
  long long step;  // elements from one K step to the next
  int lds_at[N];
  unsigned odd[ODD ? N : 1], carry[ODD ? N : 1];

  __device__ void place(const T* base, int r0, int rows, long long rs, long long cs, int tid) {
    step = KC ? KE : KE * cs;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int id = tid + THREADS * i, row = id / CPR, c = id % CPR;
      lds_at[i] = row * PITCH + c * 16;
      // past the last row: any row (its results are not stored); a chunk that straddles the end runs on into the next k's row
      if (KC) at[i] = base + min(r0 + row, rows - 1) * rs + c * E;
      else at[i] = base + (long long)row * cs + (r0 + c * E < rows ? r0 + c * E : 0);
      if constexpr (ODD) odd[i] = (unsigned)(reinterpret_cast<uintptr_t>(at[i]) >> 1) & 1u, at[i] += odd[i];  // (every step's: a step is 128 bytes)
    }
  }
  __device__ u32x4 load(int i, int s) const {
    if constexpr (ODD) return *reinterpret_cast<const u32x4_at4*>(at[i] + s * step);
    else return load16(at[i] + s * step);
  }
  // ODD: chunks from step s on; the word that a row's first one wants of the step before
  __device__ void begin_at(int s, int tid) {
    if constexpr (ODD)
#pragma unroll
      for (int i = 0; i < N; ++i) carry[i] = *reinterpret_cast<const unsigned*>(at[i] - (tid & 7) * E + s * step - 2 * (int)odd[i]);
  }
  // The chunk that load's result stands for; ODD: step by step.
  __device__ u32x4 chunk(u32x4 v, int i, int tid) {
    if constexpr (!ODD) return v;
    const unsigned below = __builtin_amdgcn_update_dpp(0u, v[3], 0x111, 0xf, 0xf, true);  // lane - 1's
    const unsigned before = (tid & 7) == 0 ? carry[i] : below, pick = odd[i] ? 0x05040302u : 0x07060504u;
    carry[i] = __builtin_amdgcn_update_dpp(0u, v[3], 0x107, 0xf, 0xf, true);              // lane + 7's
    return u32x4{__builtin_amdgcn_perm(v[0], before, pick), __builtin_amdgcn_perm(v[1], v[0], pick), __builtin_amdgcn_perm(v[2], v[1], pick),
                 __builtin_amdgcn_perm(v[3], v[2], pick)};
  }
  // step s with `left` elements of k, by element; rows: of the operand behind r0
  __device__ u32x4 load_last(int i, int s, int left, int r0, int rows, int tid) const {
    const int id = tid + THREADS * i, row = id / CPR, c = id % CPR;
    T v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int k = KC ? c * E + e : row;
      long long off = s * step;
      if (KC) off += k < left ? e : -c * E;
      else off += (r0 + c * E < rows ? min(e, rows - 1 - r0 - c * E) : 0);
      const bool there = k < left;
      const T* p = at[i] + off;
      if (!KC && !there) p = at[i] - row * (step / KE);  // something that exists: the operand's first k
      v[e] = there ? *p : (T)0.f;
    }
    return __builtin_bit_cast(u32x4, v);
  }
  // The same for K >= KE, by vectors: the KE elements of k in front of K's end, of which `trimmed` keeps those that step s - 1 has not had.  (32 loads of
  // an element per thread kept a CU's address unit busy for a microsecond: f16 1000 x 777 x 1531 12.8 -> 12.2 us.)
  __device__ u32x4 load_end(int i, int s, int left, int r0, int rows, int tid) const {
    const int id = tid + THREADS * i, row = id / CPR, c = id % CPR, x = r0 + c * E < rows ? r0 + c * E : 0;
    if (KC) return load16(at[i] + s * step - (KE - left) - (ODD ? (int)odd[i] : 0));
    const T* q = at[i] + s * step - (KE - left) * (step / KE);
    if (row < KE - 1 || x + E <= rows) return load16(q);
    T t[E];  // behind the last row nothing may be read
#pragma unroll
    for (int e = 0; e < E; ++e) t[e] = q[min(e, rows - 1 - x)];
    return __builtin_bit_cast(u32x4, t);
  }
  __device__ static u32x4 trimmed(u32x4 v, int i, int left, int tid) {
    const int id = tid + THREADS * i, row = id / CPR, c = id % CPR, had = KE - left;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const int n = KC ? had - c * E - w * (E / 4) : row < had ? 2 : 0;  // of this word's elements and those behind it
      v[w] = n >= E / 4 ? 0u : n > 0 ? v[w] & 0xffff0000u : v[w];
    }
    return v;
  }
  // lane's fragment of block b0 .. b0 + 31, chunk pair c2 (chunks 2 c2 and 2 c2 + 1)
  __device__ static u32x4 frag(const char* lds, int b0, int c2, int lane) {
    if constexpr (KC) {
      return *reinterpret_cast<const u32x4*>(lds + (b0 + (lane & 31)) * PITCH + (2 * c2 + (lane >> 5)) * 16);
    } else if constexpr (sizeof(T) == 4) {
      u32x4 v;
      const char* q = lds + (2 * c2 + (lane >> 5)) * 4 * PITCH + (b0 + (lane & 31)) * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const unsigned*>(q + e * PITCH);
      return v;
    } else {
      // lane q + 4 e of a 16-lane group names row k0 + e and four columns from 4 q; lane i receives k0 .. k0 + 3 of column i
      typedef __attribute__((address_space(3))) s16x4 lds_v4;
      const int g = lane >> 4, li = lane & 15, k0 = c2 * 16 + 8 * (g >> 1) + (li >> 2);
      const char* q = lds + k0 * PITCH + (b0 + (g & 1) * 16 + 4 * (li & 3)) * 2;
      const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)q));
      const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(q + 4 * PITCH)));
      return u32x4{lo.x, lo.y, hi.x, hi.y};
    }
  }
};

template <typename T, bool SPLIT>
struct Result { typedef T type; };
template <typename T>
struct Result<T, true> { typedef float type; };

// ONE: K is one step or less: loaded by element, one multiplication, no loop.  What bounds it: the launch.  (Going through the code for more steps, us before / so: f16
// 777 x 1001 x 33 4.7 / 4.3, x 63 5.2 / 4.7, 40 of 130 x 130 x 40 5.7 / 5.2, 2001^2 x 33 9.3 / 8.5; f32 777 x 1001 x 30 5.0 / 4.7.)
// SPLIT: slab s of nsplit has the steps per * s .. per * (s + 1) - 1 of K, the last one the remainder, and leaves its sums in ws, slab_elems apart.
enum Form { ONE, WHOLE, SPLIT_K };
template <typename T, int BT, bool A_KC, bool B_KC, Form FORM, bool ODD>
__global__ void __launch_bounds__(256) gemm_ragged(MMArgs p, int batches, int tiles_m, int tiles_n, int nsplit, int per, float* __restrict__ ws, size_t slab_elems) {
  typedef Side<T, BT, A_KC, 256, ODD && A_KC> SA;
  typedef Side<T, BT, B_KC, 256, ODD && B_KC> SB;
  constexpr bool SPLIT = FORM == SPLIT_K;
  constexpr int MI = BT / 64, KE = SA::KE;
  __shared__ __attribute__((aligned(16))) char lds[2][SA::BYTES + SB::BYTES];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // each XCD a contiguous run of all products' tiles (block ids go round-robin over the 8): with the runs dealt product by product a batch
  // of products of one tile would be one XCD's work (300 of 33 x 17 x 129 in f32: 32 us that way, 8.9 so, 16 in the kernel by element)
  const int tpb = tiles_m * tiles_n, tiles = batches * tpb * (SPLIT ? nsplit : 1), run = (tiles + 7) >> 3;
  int bid = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
  if (bid >= tiles) return;
  const int slab = SPLIT ? bid / (batches * tpb) : 0;  // (slab by slab: tiles of one slab that share rows are neighbours)
  if (SPLIT) bid -= slab * batches * tpb;
  const int batch = bid / tpb, in_batch = bid - batch * tpb, tm = in_batch / tiles_n, tn = in_batch - tm * tiles_n, m0 = tm * BT, n0 = tn * BT;
  SA a;
  SB b;
  a.place(static_cast<const T*>(p.a) + (size_t)batch * p.a_bs, m0, p.M, p.a_rs, p.a_cs, tid);
  b.place(static_cast<const T*>(p.b) + (size_t)batch * p.b_bs, n0, p.N, p.b_cs, p.b_rs, tid);
  const int full = (p.K - 1) / KE, left = p.K - full * KE;  // whole steps, and 1 .. KE elements of k behind them
  // the steps behind the first one: that is K's remainder, or in front of the last slab the slab's first
  const bool with_left = !SPLIT || slab == nsplit - 1;
  const int begin = SPLIT ? slab * per + (with_left ? 0 : 1) : 0, end = with_left ? full : (slab + 1) * per;
  f32x16 acc[MI][MI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  const int wm = (wave >> 1) * 32 * MI, wn = (wave & 1) * 32 * MI;

  u32x4 ra[2][SA::N], rb[2][SB::N], la[SA::N], lb[SB::N];
  auto fetch = [&](int d, int s) {
#pragma unroll
    for (int i = 0; i < SA::N; ++i) ra[d][i] = a.load(i, s);
#pragma unroll
    for (int i = 0; i < SB::N; ++i) rb[d][i] = b.load(i, s);
  };
  auto put = [&](char* buf, const u32x4* va, const u32x4* vb, bool whole) {  // whole: chunks as they are
#pragma unroll
    for (int i = 0; i < SA::N; ++i) *reinterpret_cast<u32x4*>(buf + a.lds_at[i]) = whole ? va[i] : a.chunk(va[i], i, tid);
#pragma unroll
    for (int i = 0; i < SB::N; ++i) *reinterpret_cast<u32x4*>(buf + SA::BYTES + b.lds_at[i]) = whole ? vb[i] : b.chunk(vb[i], i, tid);
  };
  auto multiply = [&](const char* buf) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      u32x4 fa[MI], fb[MI];
#pragma unroll
      for (int i = 0; i < MI; ++i) fa[i] = SA::frag(buf, wm + 32 * i, c, lane), fb[i] = SB::frag(buf + SA::BYTES, wn + 32 * i, c, lane);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j) mma(T(), fb[j], fa[i], acc[i][j]);  // swapped: a lane holds columns of one row
    }
  };
  if constexpr (FORM == ONE) {
#pragma unroll
    for (int i = 0; i < SA::N; ++i) la[i] = a.load_last(i, 0, left, m0, p.M, tid);
#pragma unroll
    for (int i = 0; i < SB::N; ++i) lb[i] = b.load_last(i, 0, left, n0, p.N, tid);
    put(lds[0], la, lb, true);
    __syncthreads();
    multiply(lds[0]);
  } else {
    a.begin_at(with_left ? begin : begin - 1, tid);
    b.begin_at(with_left ? begin : begin - 1, tid);
    if (with_left) {
#pragma unroll
      for (int i = 0; i < SA::N; ++i) la[i] = a.load_end(i, full, left, m0, p.M, tid);
#pragma unroll
      for (int i = 0; i < SB::N; ++i) lb[i] = b.load_end(i, full, left, n0, p.N, tid);
    } else {
#pragma unroll
      for (int i = 0; i < SA::N; ++i) la[i] = a.load(i, begin - 1);
#pragma unroll
      for (int i = 0; i < SB::N; ++i) lb[i] = b.load(i, begin - 1);
    }
    if (end > begin) {
      fetch(0, begin);
      __builtin_amdgcn_sched_barrier(0);  // (in this order: the loop counts on it)
      fetch(1, min(begin + 1, end - 1));
    }
    if (with_left) {
#pragma unroll
      for (int i = 0; i < SA::N; ++i) la[i] = SA::trimmed(la[i], i, left, tid);
#pragma unroll
      for (int i = 0; i < SB::N; ++i) lb[i] = SB::trimmed(lb[i], i, left, tid);
      put(lds[0], la, lb, true);
    } else {
      put(lds[0], la, lb, false);
    }
    __syncthreads();
    multiply(lds[0]);
    auto step = [&](int d, int s) {
      char* buf = lds[d ^ 1];
      if constexpr (ODD) __builtin_amdgcn_sched_barrier(0);  // (or both steps' chunks are put together here, behind all loads)
      put(buf, ra[d], rb[d], false);
      fetch(d, min(s + 2, end - 1));  // (without a branch, so that a step's loads can be waited for alone)
      __syncthreads();                // one barrier a step: the buffer written next was read before it
      multiply(buf);
    };
    // Two steps a turn and no way out between them: from there the compiler sees one back to the loop's head on which the loads wanted there are the latest,
    // and waits for all of them there.  f16 900 x 1000 x 4001 29.2 -> 24.4 us, 1000 x 777 x 1531 14.2 -> 12.8; f32 497 x 391 x 2100 whole 45.3 -> 43.6.
    int s = begin;
    for (; s + 2 <= end; s += 2) step(0, s), step(1, s + 1);
    if (s < end) step(0, s);
  }

  // element e of lane l of block (i, j): row l % 32, column 8 (e / 4) + 4 (l / 32) + e % 4
  typedef typename Result<T, SPLIT>::type R;
  R* __restrict__ C = (SPLIT ? reinterpret_cast<R*>(ws + slab * slab_elems) : static_cast<R*>(p.c)) + (size_t)batch * p.c_bs;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int row = m0 + wm + 32 * i + (lane & 31);
    if (row >= p.M) continue;
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int col = n0 + wn + 32 * j + 8 * g + 4 * (lane >> 5);
        R* q = C + (size_t)row * p.N + col;
        if (col + 4 <= p.N) {
          store4(q, f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]});
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (col + e < p.N) q[e] = (R)acc[i][j][4 * g + e];
        }
      }
  }
}

// 32 x 32 tiles, for products of so few larger ones that most CUs would have none.  A wave has a block of its own parts of K, LDS of its own and no barriers
// in its loop; the four waves' sums meet in LDS.  Part i (of 4 nsplit) has the steps per * i .. per * (i + 1) - 1, of which there may be none; K is more than one step.
// What bounds it: launch and first bytes, then a wave's chain of steps (0.6 us, in 16 bits 8 KB of a CU's share of the caches).  f32 625 x 319 x 353 on 64 x 64 tiles 10.3 us, 6.3 so;
// what it takes, and more figures: gemm_ragged_plan.
template <typename T, bool A_KC, bool B_KC, bool SPLIT, bool ODD>
__global__ void __launch_bounds__(256) gemm_ragged32(MMArgs p, int batches, int tiles_m, int tiles_n, int nsplit, int per, float* __restrict__ ws, size_t slab_elems) {
  typedef Side<T, 32, A_KC, 64, ODD && A_KC> SA;
  typedef Side<T, 32, B_KC, 64, ODD && B_KC> SB;
  constexpr int KE = SA::KE, BUF = SA::BYTES + SB::BYTES;
  static_assert(BUF >= 4 * 1024);  // a wave's sums go where its operands were
  __shared__ __attribute__((aligned(16))) char lds[4][BUF];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tpb = tiles_m * tiles_n, tiles = batches * tpb * (SPLIT ? nsplit : 1), run = (tiles + 7) >> 3;
  int bid = (int)(blockIdx.x & 7) * run + (int)(blockIdx.x >> 3);
  if (bid >= tiles) return;
  const int slab = SPLIT ? bid / (batches * tpb) : 0;
  if (SPLIT) bid -= slab * batches * tpb;
  const int batch = bid / tpb, in_batch = bid - batch * tpb, tm = in_batch / tiles_n, tn = in_batch - tm * tiles_n, m0 = tm * 32, n0 = tn * 32;
  const int full = (p.K - 1) / KE, left = p.K - full * KE;
  const int from = (slab * 4 + wave) * per, to = min(from + per, full + 1);
  const bool with_left = to == full + 1;
  f32x16 acc;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[e] = 0.f;
  char* buf = lds[wave];
  if (from < to) {
    SA a;
    SB b;
    a.place(static_cast<const T*>(p.a) + (size_t)batch * p.a_bs, m0, p.M, p.a_rs, p.a_cs, lane);
    b.place(static_cast<const T*>(p.b) + (size_t)batch * p.b_bs, n0, p.N, p.b_cs, p.b_rs, lane);
    // behind the first one, K's remainder or the part's first
    const int begin = with_left ? from : from + 1, end = with_left ? full : to;
    u32x4 ra[2][SA::N], rb[2][SB::N], la[SA::N], lb[SB::N];
    auto fetch = [&](int d, int s) {
#pragma unroll
      for (int i = 0; i < SA::N; ++i) ra[d][i] = a.load(i, s);
#pragma unroll
      for (int i = 0; i < SB::N; ++i) rb[d][i] = b.load(i, s);
    };
    // (a wave's LDS operations complete in order; the fences keep the compiler from moving lanes' reads over other lanes' writes)
    auto turn = [&](const u32x4* va, const u32x4* vb, bool whole, auto&& next) {  // whole: chunks as they are
#pragma unroll
      for (int i = 0; i < SA::N; ++i) *reinterpret_cast<u32x4*>(buf + a.lds_at[i]) = whole ? va[i] : a.chunk(va[i], i, lane);
#pragma unroll
      for (int i = 0; i < SB::N; ++i) *reinterpret_cast<u32x4*>(buf + SA::BYTES + b.lds_at[i]) = whole ? vb[i] : b.chunk(vb[i], i, lane);
      next();
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      u32x4 fa[4], fb[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) fa[c] = SA::frag(buf, 0, c, lane), fb[c] = SB::frag(buf + SA::BYTES, 0, c, lane);
#pragma unroll
      for (int c = 0; c < 4; ++c) mma(T(), fb[c], fa[c], acc);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    };
    a.begin_at(from, lane);
    b.begin_at(from, lane);
    if (with_left) {
#pragma unroll
      for (int i = 0; i < SA::N; ++i) la[i] = a.load_end(i, full, left, m0, p.M, lane);
#pragma unroll
      for (int i = 0; i < SB::N; ++i) lb[i] = b.load_end(i, full, left, n0, p.N, lane);
    } else {
#pragma unroll
      for (int i = 0; i < SA::N; ++i) la[i] = a.load(i, from);
#pragma unroll
      for (int i = 0; i < SB::N; ++i) lb[i] = b.load(i, from);
    }
    if (end > begin) {
      fetch(0, begin);
      __builtin_amdgcn_sched_barrier(0);  // (in this order: the loop counts on it)
      fetch(1, min(begin + 1, end - 1));
    }
    if (with_left) {
#pragma unroll
      for (int i = 0; i < SA::N; ++i) la[i] = SA::trimmed(la[i], i, left, lane);
#pragma unroll
      for (int i = 0; i < SB::N; ++i) lb[i] = SB::trimmed(lb[i], i, left, lane);
      turn(la, lb, true, [] {});
    } else {
      turn(la, lb, false, [] {});
    }
    auto step = [&](int d, int s) {
      if constexpr (ODD) __builtin_amdgcn_sched_barrier(0);
      turn(ra[d], rb[d], false, [&] { fetch(d, min(s + 2, end - 1)); });
    };
    int s = begin;
    for (; s + 2 <= end; s += 2) step(0, s), step(1, s + 1);  // (no way out between the two: as in gemm_ragged)
    if (s < end) step(0, s);
  }
  // quad g of lane l: row l % 32, columns 8 g + 4 (l / 32) and the next three.  Wave w finishes quad w, summed over the waves in the order of K.
#pragma unroll
  for (int g = 0; g < 4; ++g) *reinterpret_cast<f32x4*>(buf + (g * 64 + lane) * 16) = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  __syncthreads();
  f32x4 v = *reinterpret_cast<const f32x4*>(lds[0] + (wave * 64 + lane) * 16);
#pragma unroll
  for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(lds[w] + (wave * 64 + lane) * 16);
  const int row = m0 + (lane & 31), col = n0 + 8 * wave + 4 * (lane >> 5);
  if (row >= p.M) return;
  typedef typename Result<T, SPLIT>::type R;
  R* __restrict__ q = (SPLIT ? reinterpret_cast<R*>(ws + slab * slab_elems) : static_cast<R*>(p.c)) + (size_t)batch * p.c_bs + (size_t)row * p.N + col;
  if (col + 4 <= p.N) {
    store4(q, v);
  } else {
#pragma unroll
    for (int e = 0; e < 3; ++e)
      if (col + e < p.N) q[e] = (R)v[e];
  }
}

// c = the slabs' sum, in their order
template <typename T>
__global__ void __launch_bounds__(256) gemm_ragged_fold(const float* __restrict__ ws, T* __restrict__ c, size_t elems, size_t slab_elems, int nsplit) {
  const size_t at = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (at >= elems) return;
  f32x4 s = *reinterpret_cast<const f32x4*>(ws + at);
  for (int k = 1; k < nsplit; ++k) s += *reinterpret_cast<const f32x4*>(ws + k * slab_elems + at);
  if (at + 4 <= elems) {
    store4(c + at, s);
  } else {
#pragma unroll
    for (int e = 0; e < 3; ++e)
      if (at + e < elems) c[at + e] = (T)s[e];
  }
}

// Whether an operand's contiguous lines, `rows` of them, may start in the middle of a 4-byte word.
bool odd_rows(const void* base, long long rows, long long pitch, size_t batch, long long batch_stride) {
  return (reinterpret_cast<uintptr_t>(base) & 2) || (rows > 1 && (pitch & 1)) || (batch > 1 && (batch_stride & 1));
}
// ODD where both operands start anywhere and the address unit is what a step waits for; with one of them aligned putting chunks together takes as long as it saves.  us before /
// so: f16 1000 x 776 x 2057 [n, k]-major 15.3 / 13.3, 12 of 17 x 1728 x 3185 47.3 / 35.5, bf16 2692 x 1660 x 3123 (128 x 128) 74.0 / 64.7, [k, n]-major 1000 x 777 x 1531 12.6 / 11.9;
// x 776 x 2057, the lhs alone, 12.1 / 12.9 from L2, 13.3 / 13.2 past it.
bool by_words(const MMArgs& p, size_t batch) {
  const bool ak = p.a_cs == 1, bk = p.b_rs == 1;
  return (ak || bk) && odd_rows(p.a, ak ? p.M : p.K, ak ? p.a_rs : p.a_cs, batch, p.a_bs) && odd_rows(p.b, bk ? p.N : p.K, bk ? p.b_cs : p.b_rs, batch, p.b_bs);
}
// BT 32: gemm_ragged32
template <typename T, int BT, Form FORM, bool ODD = false>
hipError_t launch(hipStream_t stream, const MMArgs& p, size_t batch, int nsplit, float* ws) {
  const bool ak = p.a_cs == 1, bk = p.b_rs == 1;
  if constexpr (sizeof(T) == 2 && FORM != ONE && !ODD)
    if (by_words(p, batch))
      return launch<T, BT, FORM, true>(stream, p, batch, nsplit, ws);
  const int tiles_m = (p.M + BT - 1) / BT, tiles_n = (p.N + BT - 1) / BT, ke = 128 / (int)sizeof(T), steps = (p.K + ke - 1) / ke;
  const int parts = BT == 32 ? 4 * nsplit : nsplit, per = (steps + parts - 1) / parts;
  const unsigned grid = (unsigned)((batch * tiles_m * tiles_n * nsplit + 7) / 8 * 8);
  const size_t elems = batch * p.M * p.N, slab = (elems + 3) / 4 * 4;
  auto go = [&](auto a_kc, auto b_kc) {
    constexpr bool odd = ODD && (a_kc() || b_kc());
    if constexpr (BT == 32) gemm_ragged32<T, a_kc(), b_kc(), FORM == SPLIT_K, odd><<<grid, 256, 0, stream>>>(p, (int)batch, tiles_m, tiles_n, nsplit, per, ws, slab);
    else gemm_ragged<T, BT, a_kc(), b_kc(), FORM, odd><<<grid, 256, 0, stream>>>(p, (int)batch, tiles_m, tiles_n, nsplit, per, ws, slab);
  };
  if (ak && bk) go(std::true_type(), std::true_type());
  else if (ak) go(std::true_type(), std::false_type());
  else if (bk) go(std::false_type(), std::true_type());
  else go(std::false_type(), std::false_type());
  if (FORM == SPLIT_K) gemm_ragged_fold<T><<<(unsigned)((elems + 1023) / 1024), 256, 0, stream>>>(ws, static_cast<T*>(p.c), elems, slab, nsplit);
  return hipGetLastError();
}
template <typename T>
hipError_t launch_plan(hipStream_t stream, const MMArgs& p, size_t batch, const RaggedPlan& pl, float* ws) {
  if (pl.tile == 32) return pl.nsplit > 1 ? launch<T, 32, SPLIT_K>(stream, p, batch, pl.nsplit, ws) : launch<T, 32, WHOLE>(stream, p, batch, 1, nullptr);
  if (pl.nsplit > 1) return launch<T, 64, SPLIT_K>(stream, p, batch, pl.nsplit, ws);
  if (p.K <= 128 / (int)sizeof(T)) return pl.tile == 128 ? launch<T, 128, ONE>(stream, p, batch, 1, nullptr) : launch<T, 64, ONE>(stream, p, batch, 1, nullptr);
  return pl.tile == 128 ? launch<T, 128, WHOLE>(stream, p, batch, 1, nullptr) : launch<T, 64, WHOLE>(stream, p, batch, 1, nullptr);
}

}  // namespace

static bool supported(const MMArgs& p, size_t batch) {
  // an operand that is contiguous along its other dimension: eight elements or more from one k to the next, so that a chunk over the end of a
  // row stays inside the rows behind it
  const bool a = p.a_cs == 1 || (p.a_rs == 1 && p.a_cs >= 8 && p.M >= 8), b = p.b_rs == 1 || (p.b_cs == 1 && p.b_rs >= 8 && p.N >= 8);
  return a && b && p.M > 0 && p.N > 0 && p.K > 0 && p.a_rs >= 0 && p.b_cs >= 0 && batch <= 65535 && batch * ((p.M + 63) / 64) * ((p.N + 63) / 64) < (1u << 24);
}

// Where each tile is the faster one, measured (us, by element / 64 x 64 / 128 x 128); the large one from 256 of them on, one round of the chip, where no
// more than a quarter of them is padding (100 f16 products of 9 x 700 x 1001, half of it padding: 261 / 42 / 52):
//   f32 up to K = 16, one step of the kernel by element, is its store: 3001 x 3003 x 16 13.8 / 15.4 / 20.6, 2001^2 x 8 8.0 / 9.0 / 10.1; at K = 17 17.7 /
//   15.4 / 20.8.  The f32 matrix pipe is busy on small tiles already (2001^2 x 129 28.4 / 17.1 / 19.9, 7 x 512 x 1219 x 333 70 / 36 / 52, 3501^2 x 1001 205 small, 263
//   large), but for long sums in three rounds or more whose last is nearly full: 3999^2 x 2000 1014 / 520 / 510, 4095^3 1048 small, 1028 large.
//   16 bits: the large tile's prologue wants more than one step to pay for it, or a last round that is nearly full: 2001^2 x 8 8.3 / 7.7 / 8.3, x 33 10.0 / 9.0 / 8.5, x 127
//   18.1 / 14.3 / 11.9, x 1001 141 / 31.2 / 23.5, 3187 x 2088 x 64 16.3 small, 14.5 large, 7 x 512 x 1219 x 63 19.6 / 13.1 / 15.4, x 129 37.8 / 13.1 / 15.0, x 1001 283 /
//   37.5 / 35.0.
//   16 bits, fewer than 256 large ones: 64 x 64 tiles that share a CU wait for its loads, so four of them and a long sum (1216 x 3200 x 1652 44.3 small, 27.2 large,
//   1489 x 2130 x 932 24.7 / 19.2, 1215 x 2795 x 593 22.6 / 17.0; 2893 x 1238 x 202 10.5 / 10.3) or three and a longer one (1613 x 1568 x 3947 71.5 / 58.3, 3038 x 886 x 1694 27.4 /
//   24.8; 2415 x 1244 x 861 18.3 / 19.2) are better off as one; two are not (2020 x 1018 x 2436 24.7 / 30.7).
static int tile_of(int dtype, const MMArgs& p, size_t big, size_t small) {
  if (3 * big > small) return 64;
  if (dtype == UGHIP_F32) return big >= 768 && (big + 64) % 256 <= 64 && p.K >= 1024 ? 128 : 64;
  if (big < 256) return (small > 768 && p.K > 256) || (small > 600 && p.K >= 1536) ? 128 : 64;
  return p.K > 64 || (p.K > 8 && big * 5 >= (big + 255) / 256 * 256 * 4) ? 128 : 64;
}

// Fewer than 256 small tiles: 64 x 64 or, where that leaves most CUs without one, 32 x 32 with K over the workgroup's waves; and with a long sum slabs of K in the
// workspace and a launch that adds them (2.5 us and 0.1 a slab, the slabs' way to memory and back, and 8.8 us at the least: a program's thread takes that for the two).
//   64 x 64: a step takes 0.25 us and up to 0.16 more as the chip fills (f32: 0.56 and 0.06), 0.75 (1.1) beside another tile on its CU
//   32 x 32: a quarter of the steps at 0.6 us (f32: 0.66, as many times as a CU has tiles); 16 bits wait for their 8 KB a step as well, 0.12 us and as much again when the chip is full
// Measured, us 64 whole / 64 split / 32 whole / 32 split, the best split each: f32 300^3 9.0 / 8.7 / 6.3 / -, 625 x 319 x 353 10.3 / 9.7 / 6.3 / -, 15 of 19 x 18 x 640 14.8 / 9.1 /
// 6.7 / 9.0, 700 x 700 x 500 13.0 / 12.5 / 10.2 / 14.9, 777 x 500 x 1500 30.6 / 20.8 / 19.2 / 22.8, 39 x 801 x 3001 56 / 12.9 / 18.2 / 11.5, 38 x 20 x 1920 37 / 11.0 / 12.3 / 9.1,
// 1000 x 777 x 399 11.7 / 16.1 / 14.0 / -; f16 23 x 148 x 1355 8.4 / 8.9 / 6.2 / 8.9, 200 x 200 x 1000 7.2 / 8.6 / 6.0 / 8.8, 497 x 391 x 2100 13.4 / 10.6 / 10.0 / 14.4, 150 x 1000 x
// 4001 21.7 / 11.7 / 15.6 / 15.1, 39 x 801 x 3001 15.1 / 9.0 / 10.8 / 9.0, 777 x 500 x 1500 10.2 / 10.4 / 11.1 / 16.7.  At most 32 MB of slabs, the least that the block of
// partial tiles holds.
static double few_tiles_us(int dtype, int tile, int steps, size_t tiles, int ns, size_t slab_bytes) {
  const bool f32 = dtype == UGHIP_F32;
  const double share = (double)(tiles * ns) / 256;
  const int per = (steps + ns - 1) / ns, part = (steps + 4 * ns - 1) / (4 * ns), on_cu = (int)((tiles * ns + 255) / 256);
  double us = f32 ? 3.2 : 3.0;
  if (tile == 32) us += 0.3 * on_cu + (f32 ? 0.66 * part * on_cu : std::max(0.6 * part, (0.12 + 0.12 * share) * per));
  else us += per * (share > 1 ? (f32 ? 1.1 : 0.75) : f32 ? 0.56 + 0.06 * share : 0.25 + 0.16 * share);
  return ns == 1 ? us : std::max(8.8, us + 2.5 + 0.1 * ns + (double)(ns + 1) * slab_bytes / 5e6);
}

bool gemm_ragged_words(int dtype, const MMArgs& p, size_t batch, const RaggedPlan& plan) { return plan.tile && dtype != UGHIP_F32 && p.K > 64 && by_words(p, batch); }

bool gemm_ragged_takes(int dtype, const MMArgs& p, size_t batch) { return supported(p, batch) && !(dtype == UGHIP_F32 && p.K <= 16); }

RaggedPlan gemm_ragged_plan(int dtype, const MMArgs& p, size_t batch) {
  RaggedPlan pl;
  if (!gemm_ragged_takes(dtype, p, batch)) return pl;
  auto tiles = [&](int t) { return batch * ((p.M + t - 1) / t) * ((p.N + t - 1) / t); };
  const size_t small = tiles(64), slab_bytes = (batch * p.M * p.N + 3) / 4 * 16;
  pl.tile = tile_of(dtype, p, tiles(128), small);
  if (pl.tile == 128 || small >= 256) return pl;
  const int ke = dtype == UGHIP_F32 ? 32 : 64, steps = (p.K + ke - 1) / ke;
  if (steps == 1) return pl;  // (nothing to share)
  double best = 0.95 * few_tiles_us(dtype, 64, steps, small, 1, slab_bytes);
  for (int tile : {32, 64}) {
    const size_t n = tiles(tile);
    for (int ns = 1; ns <= 32 && ns * (tile == 32 ? 8 : 2) <= std::max(steps, 8) && (ns == 1 || (n * ns <= 512 && ns * slab_bytes <= RaggedPlan::MAX_WS)); ++ns) {
      const int per = (steps + ns - 1) / ns;
      if (tile == 64 && (ns == 1 || (steps + per - 1) / per != ns)) continue;  // (a slab would have no steps)
      const double us = few_tiles_us(dtype, tile, steps, n, ns, slab_bytes);
      if (us < best) best = us, pl.tile = tile, pl.nsplit = ns;
    }
  }
  if (pl.nsplit > 1) pl.ws_bytes = pl.nsplit * slab_bytes;
  return pl;
}

hipError_t gemm_ragged_launch(hipStream_t stream, int dtype, const MMArgs& p, size_t batch, const RaggedPlan& pl, float* ws) {
  if (!supported(p, batch) || (pl.tile != 32 && pl.tile != 64 && pl.tile != 128) || pl.nsplit < 1 || (pl.nsplit > 1 && (pl.tile == 128 || !ws))) return hipErrorInvalidValue;
  if ((pl.tile == 32 || pl.nsplit > 1) && p.K <= (dtype == UGHIP_F32 ? 32 : 64)) return hipErrorInvalidValue;
  if (dtype == UGHIP_F32) return launch_plan<float>(stream, p, batch, pl, ws);
  return dtype == UGHIP_F16 ? launch_plan<_Float16>(stream, p, batch, pl, ws) : launch_plan<__bf16>(stream, p, batch, pl, ws);
}

}  // namespace ughip
