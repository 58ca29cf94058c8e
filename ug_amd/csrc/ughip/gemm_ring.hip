// 16-bit MFMA GEMM for products that leave the chip idle or waiting on gemm_dma4's tiles: C = A x B, f32 accumulate, K tile 64.
//
//   Eight waves, 4 x 2, each BM / 4 x BN / 2 of the result in 16 x 16 accumulators (v_mfma_f32_16x16x32): a wave's waits are filled by the other
//   one of its SIMD.  The k order of every sum is that of gemm_dma4 and gemm_tiled, so the results are theirs bit for bit.
//   32 x 32, four waves and eight stages, for rows only: a CU has some 55 KB on its way whatever it is asked for, so where 64 x 64 tiles are few it is their bytes per CU that count (us on
//   64 x 64 and so, weights from memory: 54 rows of 2048 x 2048 / 4096 / 5632 11.3 / 19.6 / 26.8 -> 6.7 / 10.6 / 14.1, 509 rows of 256 x 2048 8.9 -> 6.4, 228 of 2048 x 2048 11.3 -> 9.8).
//   192 x 192 for rows only: 700 rows against 11264 x 2048 are 236 of them, one round (52 us with 256 x 256, 54 with 256 x 128, 34 so).
//   A ring of four stages (three for 256 x 128, 192 x 192 and 192 columns of 128 rows, two for 256 x 192, eight for 32 x 32): the loads of a K tile go out (global_load_lds_dwordx4, as in gemm_dma4) when the tile
//   that many in front of it has been read, so all but one of them are on their way while one is multiplied.  One barrier per K tile.
//
// What bounds it: the operands' way to a CU.  2048^2 x 5632 on 128 x 128 tiles, one to a CU, takes 42 us, 0.44 per K tile of 32 KB, with the operands in
// the memory-side cache (matrix pipes busy 61 % of the time) and 54 us, 0.57, with both from HBM (42 %); gemm_dma4's two stages 58 and 75.  From HBM
// it takes as long without its MFMAs, and a loop of nothing but the loads takes 0.33 / 0.52 us: a CU gets some 100 / 60 bytes per ns however many it has
// on their way (deeper rings, loads that bypass the cache and a wave that touches the lines for L2 ahead of the others made nothing faster).
// So tiles are as large as leaves every CU one, by the model in gemm_dma.hip.
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "gemm_dma.h"
#include "internal.h"
#include "layers.h"
#include "ughip.h"

namespace ughip {
namespace {

constexpr int waves(int bm) { return bm == 32 ? 4 : 8; }  // two to a row of them
constexpr int stages(int bm, int bn) { return bm == 32 ? 8 : bm == 256 && bn == 192 ? 2 : bm >= 192 || bm * bn > 128 * 128 ? 3 : 4; }
constexpr int lds_bytes(int bm, int bn, bool planes = false) { return (stages(bm, bn) * bm + (planes ? 2 : stages(bm, bn)) * bn) * BK * 2; }  // planes: two tiles of the rhs

// One tile: rows [m0, m_end) (BM of them at most) and the columns of column tile tn, of one batch or group.
// Template parameters and DmaRows as in gemm_dma4; ROWS 3: rows that leave as gelu(y) times an element of their token's row of a table.
template <typename T, int BM, int BN, bool B_KN, bool F32OUT, int BDIV, int ROWS>
__device__ __forceinline__ void ring_tile(const MMArgs& p, int batch, int group, int m0, int m_end, int tn, const float* __restrict__ residual, const DmaRows& rw) {
  static_assert(ROWS == 0 || (BDIV == 1 && !B_KN && !F32OUT), "rows: one plane against an [n, k]-major rhs");
  static_assert(BDIV == 1 || !B_KN, "planes of the lhs: against an [n, k]-major rhs only");
  static_assert(!B_KN || BN >= 128, "the swizzle of an n-contiguous tile wants eight 32-byte pieces per row");
  extern __shared__ u32x4 lds[];
  constexpr int S = stages(BM, BN);
  constexpr int W = waves(BM), WR = W / 2;  // waves, and rows of them
  constexpr int NI = BM / (16 * WR), NJ = BN / 32, NM = NI * NJ;  // 16-row and 16-column fragments and MFMAs of a wave and step of 32 k
  constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2, STAGE_BYTES = A_BYTES + B_BYTES;
  constexpr int NDA = BM / (8 * W), NDB = BN / (8 * W), ND = NDA + NDB;   // loads per wave and K tile
  constexpr int R = NI + NJ;                                      // fragment reads per step
  // SHARED: the three planes of a lhs tile meet one rhs tile, which is loaded once for them, into one of two places of its own behind the ring.
  constexpr bool SHARED = BDIV == 3;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const int n0 = tn * BN;
  const long long lda = p.a_rs, ldb = B_KN ? p.b_rs : p.b_cs;
  const char* Ab = reinterpret_cast<const char*>(static_cast<const T*>(p.a) + (size_t)batch * p.a_bs + (ROWS ? 0 : (size_t)m0 * lda));
  const char* Bb = reinterpret_cast<const char*>(static_cast<const T*>(p.b) + (size_t)batch * p.b_bs + (ROWS ? (size_t)group * rw.w_group : 0) +
                                                 (ROWS == 2 ? 0 : B_KN ? (size_t)n0 : (size_t)n0 * ldb));
  const int KT = p.K / BK;
  const int wm = (wave >> 1) * (BM / WR), wn = (wave & 1) * (BN / 2);
  const unsigned lds_addr = (unsigned)(size_t)(__attribute__((address_space(3))) char*)lds;
  // per-lane byte offsets of this wave's loads; rows past the end fetch the last row again (their results are not stored)
  unsigned voff[ND];
  const int m_last = m_end - 1 - m0, n_left = p.N - n0;
#pragma unroll
  for (int i = 0; i < NDA; ++i) {
    const int row = (i * W + wave) * 8 + (lane >> 3), cp = lane & 7;
    int src = min(row, m_last);
    if constexpr (ROWS != 0) {
      src += m0;
      if (rw.row_index) src = max(0, min(rw.row_index[src], rw.x_rows - 1));
    }
    voff[i] = (unsigned)(src * lda * 2 + ((cp ^ ((row >> 1) & 7)) << 4));
  }
#pragma unroll
  for (int i = 0; i < NDB; ++i) {
    const int g = i * W + wave;
    if (!B_KN) {
      const int row = g * 8 + (lane >> 3), cp = lane & 7;
      int src = min(row, n_left - 1);
      if constexpr (ROWS == 2) {  // a wave's half of the tile: BN / 4 gate columns, then the same columns of up
        const int q = row % (BN / 2);
        src = min(tn * (BN / 2) + row / (BN / 2) * (BN / 4) + q % (BN / 4), rw.n_out - 1) + (q >= BN / 4 ? rw.n_out : 0);
      }
      voff[NDA + i] = (unsigned)(src * ldb * 2 + ((cp ^ ((row >> 1) & 7)) << 4));
    } else {
      constexpr int CPR = BN / 8;  // 16-byte chunks per row of k
      const int k = g * (64 / CPR) + lane / CPR, cpos = lane % CPR;
      const int src = (((cpos >> 1) ^ kn_h(k)) << 1) | (cpos & 1);
      voff[NDA + i] = (unsigned)(k * ldb * 2 + (min(src, n_left / 8 - 1) << 4));  // N % 8 == 0: whole 16-byte chunks
    }
  }
  const long long a_step = BK * 2, b_step = B_KN ? (long long)BK * ldb * 2 : BK * 2;
  auto dma = [&](int tile, int idx) {  // idx: compile-time after unrolling
    const unsigned st = lds_addr + (unsigned)tile % S * (SHARED ? A_BYTES : STAGE_BYTES);
    if (idx < NDA) dma16(Ab + lhs_k_tile<BDIV>(tile) * a_step, voff[idx], st + (idx * W + wave) * 1024);
    else dma16(Bb + rhs_k_tile<BDIV>(tile) * b_step, voff[idx], (SHARED ? lds_addr + S * A_BYTES + (tile / 3 & 1) * B_BYTES : st + A_BYTES) + ((idx - NDA) * W + wave) * 1024);
  };

  floatx4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  u32x4 fa[2][NI], fb[2][NJ];
  auto read_frag = [&](int tile, int step, int idx, int set) {
    const int stage = (unsigned)tile % S;
    if (idx < NI) {
      fa[set][idx] = lds[stage * ((SHARED ? A_BYTES : STAGE_BYTES) / 16) + kc_idx(wm + idx * 16 + (lane & 15), 4 * step + (lane >> 4))];
    } else if (!B_KN) {
      fb[set][idx - NI] = lds[(SHARED ? S * A_BYTES + (tile / 3 & 1) * B_BYTES : stage * STAGE_BYTES + A_BYTES) / 16 + kc_idx(wn + (idx - NI) * 16 + (lane & 15), 4 * step + (lane >> 4))];
    } else {
      typedef __attribute__((address_space(3))) s16x4 lds_v4;  // transposing reads: as in gemm_dma4
      const int g = lane >> 4, li = lane & 15, q = li & 3, e = li >> 2;
      const char __attribute__((address_space(3)))* Bs = (const char __attribute__((address_space(3)))*)lds + stage * STAGE_BYTES + A_BYTES;
      const int n = wn + (idx - NI) * 16 + 4 * q, k0 = step * 32 + 8 * g + e;
      const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(Bs + kn_byte<BN>(k0, n))));
      const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(Bs + kn_byte<BN>(k0 + 4, n))));
      fb[set][idx - NI] = u32x4{lo.x, lo.y, hi.x, hi.y};
    }
  };

  // MFMAs of one step on register set X, the first RS of the next step's reads (tile rt, step rs: into the other set) and LD loads (LA of the lhs of tile dt, the rest of the rhs of tile bt)
  // dealt over them
  auto step = [&](auto set, auto reads, int rt, int rs, auto lhs, int dt, auto rhs, int bt) {
    constexpr int X = decltype(set)::value, RS = decltype(reads)::value, LA = decltype(lhs)::value, LD = LA + decltype(rhs)::value;
#pragma unroll
    for (int g = 0; g < NM; ++g) {
#pragma unroll
      for (int r = 0; r < RS; ++r)
        if (r * NM / RS == g) read_frag(rt, rs, r, X ^ 1);
#pragma unroll
      for (int d = 0; d < LD; ++d)
        if (d * NM / LD == g) {
          if (d < LA) dma(dt, d);
          else dma(bt, NDA + d - LA);
        }
      acc[g / NJ][g % NJ] = mma16(T(), fb[X][g % NJ], fa[X][g / NJ], acc[g / NJ][g % NJ]);  // operands swapped: a lane gets 4 columns of a row
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using CS = std::integral_constant<int, S>;
  // Everybody has read the stage of tile kt, and tile kt + 1 has landed, behind which `behind` loads may still be on their way.
  auto turn = [&](auto behind) {
    if constexpr (decltype(behind)::value >= 0) wait_vmcnt<decltype(behind)::value>();
    wait_lgkmcnt0();
    __builtin_amdgcn_s_barrier();
  };
  // A K tile: the first step's fragments are in set 0, the turn comes between the steps, behind it the tile's stage takes the loads of the tile
  // S further on.  A: how many tiles follow kt (S stands for that many or more).
  auto body = [&](int kt, auto ahead) {
    constexpr int A = decltype(ahead)::value, MORE = A == S, BEHIND = ((A < S ? A : S - 1) - 1) * ND;
    step(C0(), std::integral_constant<int, R>(), kt, 1, C0(), 0, C0(), 0);
    turn(std::integral_constant<int, (A > 0 ? BEHIND : -1)>());
    step(C1(), std::integral_constant<int, (A > 0 ? R : 0)>(), kt + 1, 0, std::integral_constant<int, (MORE ? NDA : 0)>(), kt + S, std::integral_constant<int, (MORE ? NDB : 0)>(), kt + S);
  };
  // The same with a shared rhs tile, kt being plane P of it: its fragments of step 1 are read in plane 0's first step, the next one's of step 0 in plane 2's second, where the registers have had
  // their last use.  Behind plane 0's turn its place is free: the rhs tile two further on goes there (B: there is one), six K tiles ahead of its use.  llama's output projection of 1900 rows (128 x 128 tiles): 51.5 -> 46.9 us.
  auto body_shared = [&](int kt, auto plane, auto ahead, auto more_rhs) {
    constexpr int P = decltype(plane)::value, A = decltype(ahead)::value, B = decltype(more_rhs)::value, MORE = A == S;
    static_assert(!SHARED || S == 3 || S == 4, "which loads lie between tile kt + 1's and the turn");
    // (the lhs tiles kt + 2 .. kt + S - 1 and the rhs tile asked for behind the latest turn of a plane 0, with plane 0 itself only where that one still comes behind lhs tile kt + 1)
    constexpr int BEHIND = A < S ? (A - 1) * NDA : (S - 2) * NDA + (B && (P != 0 || S == 4) ? NDB : 0);
    step(C0(), std::integral_constant<int, NI + (P == 0 ? NJ : 0)>(), kt, 1, C0(), 0, C0(), 0);
    turn(std::integral_constant<int, (A > 0 ? BEHIND : -1)>());
    step(C1(), std::integral_constant<int, (A > 0 ? NI + (P == 2 ? NJ : 0) : 0)>(), kt + 1, 0, std::integral_constant<int, (MORE ? NDA : 0)>(), kt + S, std::integral_constant<int, (B && P == 0 ? NDB : 0)>(), kt + 6);
  };
  if constexpr (SHARED) {  // six K tiles at least (the host checks)
#pragma unroll
    for (int d = 0; d < ND; ++d) dma(0, d);
#pragma unroll
    for (int t = 1; t < S; ++t)
#pragma unroll
      for (int d = 0; d < NDA; ++d) dma(t, d);
#pragma unroll
    for (int d = NDA; d < ND; ++d) dma(3, d);
    wait_vmcnt<(S - 1) * NDA + NDB>();
  } else {
#pragma unroll
    for (int t = 0; t < S; ++t)
      if (t < KT) {
#pragma unroll
        for (int d = 0; d < ND; ++d) dma(t, d);
      }
    if (KT >= S) wait_vmcnt<(S - 1) * ND>();
    else wait_vmcnt<0>();
  }
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int r = 0; r < R; ++r) read_frag(0, 0, r, 0);
  if constexpr (SHARED) {
    using C2 = std::integral_constant<int, 2>;
    int kt = 0;
    for (; kt < KT - 6; kt += 3) body_shared(kt, C0(), CS(), C1()), body_shared(kt + 1, C1(), CS(), C1()), body_shared(kt + 2, C2(), CS(), C1());
    using A3 = std::integral_constant<int, 3>;  // S or three
    body_shared(KT - 6, C0(), CS(), C0()), body_shared(KT - 5, C1(), CS(), C0()), body_shared(KT - 4, C2(), A3(), C0());
    body_shared(KT - 3, C0(), C2(), C0()), body_shared(KT - 2, C1(), C1(), C0()), body_shared(KT - 1, C2(), C0(), C0());
  } else {
    for (int kt = 0; kt < KT - S; ++kt) body(kt, CS());
    auto left = [&](auto ahead) {
      if constexpr (decltype(ahead)::value < S)
        if (KT > decltype(ahead)::value) body(KT - 1 - decltype(ahead)::value, ahead);
    };
    left(std::integral_constant<int, 7>());
    left(std::integral_constant<int, 6>());
    left(std::integral_constant<int, 5>());
    left(std::integral_constant<int, 4>());
    left(std::integral_constant<int, 3>());
    left(std::integral_constant<int, 2>());
    left(C1());
    body(KT - 1, C0());
  }

  // Register e of lane l of block (i, j): row wm + 16 i + l % 16, column wn + 16 j + 4 (l / 16) + e.
  static_assert(S * A_BYTES + (SHARED ? 2 : S) * B_BYTES >= W * (NI > 1 ? 2 : 1) * 16 * (BN / 2 * 4 + 16), "what rows and f32 sums leave by: pieces of 16 rows of a wave's columns");
  if constexpr (ROWS != 0) {
    rows_out<T, ROWS>(acc, rw, m0, m_last, wm, ROWS == 2 ? tn * (BN / 2) + (wave & 1) * (BN / 4) : n0 + wn, wave, lds);
    return;
  }
  if constexpr (F32OUT) {
    const size_t at = (size_t)batch * p.c_bs + (size_t)m0 * p.N + n0;
    sums_out(acc, static_cast<float*>(p.c) + at, residual ? residual + at : nullptr, p.N, m_last, n_left, wm, wn, wave, lds);
    return;
  }
  // 16-bit result through LDS, out in 16-byte pieces of whole rows past the cache.
  constexpr int PITCH = BN * 2 + 8;
  char __attribute__((address_space(3)))* Cs = (char __attribute__((address_space(3)))*)lds;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      typedef T tx4 __attribute__((ext_vector_type(4)));
      tx4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (T)acc[i][j][e];
      const int row = wm + i * 16 + (lane & 15), col = wn + j * 16 + (lane >> 4) * 4;
      *(u32x2 __attribute__((address_space(3)))*)(Cs + row * PITCH + col * 2) = __builtin_bit_cast(u32x2, v);
    }
  __syncthreads();
  constexpr int CPR = BN / 8, RPP = 64 * W / CPR;
  T* __restrict__ C = static_cast<T*>(p.c) + (size_t)batch * p.c_bs + (size_t)m0 * p.N + n0;
  const int c = tid % CPR, r0 = tid / CPR;
#pragma unroll
  for (int pass = 0; pass < BM / RPP; ++pass) {
    const int row = pass * RPP + r0;
    const u32x2 lo = *(const u32x2 __attribute__((address_space(3)))*)(Cs + row * PITCH + c * 16);
    const u32x2 hi = *(const u32x2 __attribute__((address_space(3)))*)(Cs + row * PITCH + c * 16 + 8);
    if (row <= m_last && c * 8 < n_left) __builtin_nontemporal_store(u32x4{lo.x, lo.y, hi.x, hi.y}, reinterpret_cast<u32x4*>(C + (size_t)row * p.N + c * 8));
  }
}

// The tiles of a launch, dealt to its workgroups.
template <typename T, int BM, int BN, bool B_KN, bool F32OUT, int BDIV, int ROWS>
__global__ void __launch_bounds__(64 * waves(BM)) gemm_ring(MMArgs p, int batches, int tiles_m, int tiles_n, const float* __restrict__ residual, DmaRows rw) {
  const int lane = threadIdx.x & 63;
  // XCD-aware order of the tiles: as in gemm_dma4 (the grid is 8 more at least, the runs are of equal length)
  int tiles = batches * tiles_m * tiles_n;
  GroupTiles<BM> by_group{rw.group_end, rw.groups, p.M, lane};
  if (ROWS != 0 && rw.groups) {
    tiles_m = by_group.count();
    tiles = tiles_m * tiles_n;
  }
  const int per = (tiles + 7) >> 3;
  if ((int)blockIdx.x >= 8 * per) return;
  const int bid = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (bid >= tiles) return;
  const int tpb = tiles_m * tiles_n;
  const int batch = bid / tpb;
  const int t_in = bid - batch * tpb;
  int tm, tn;
  if ((tiles_m & 3) == 0) {
    const int sr = t_in / (4 * tiles_n), rem = t_in - sr * 4 * tiles_n;
    tm = sr * 4 + (rem & 3);
    tn = rem >> 2;
  } else {
    tm = t_in / tiles_n;
    tn = t_in - tm * tiles_n;
  }
  int m0 = tm * BM, m_end = p.M, group = 0;
  if (ROWS != 0 && rw.groups && !by_group.find(tm, group, m0, m_end)) return;  // the same for the whole workgroup
  ring_tile<T, BM, BN, B_KN, F32OUT, BDIV, ROWS>(p, batch, group, m0, m_end, tn, residual, rw);
}

// Rows by group (bf16), each group's rows dealt evenly over as few tiles of at most 256 rows as hold them and every tile as high as its rows want, in steps of
// 64.  What bounds such a product are its operands' bytes on their way to the CUs, in rounds of 256 workgroups: tiles of one height load and multiply
// rows that nobody asked for, and a few groups above that height are a second round of nearly empty tiles.  16 groups, us on the best of the tiles of one height and so: n 2 x 1408,
// k 2048, 768 rows 50.6 -> 47.1 (192 columns); n 2048, k 1408, 768 / 1024 / 1280 / 1600 rows 28.4 / 30.3 / 31.6 / 34.5 -> 25.1 / 26.3 / 28.1 / 30.4 (128 columns), 3200 / 4096 / 8192
// rows 54.5 / 55 / 88 -> 47 / 48 / 83 (192 columns).
template <int BN, int ROWS>
__global__ void __launch_bounds__(512) gemm_ring_groups(MMArgs p, int tiles_n, DmaRows rw) {
  GroupTiles<256, true> by_group{rw.group_end, rw.groups, p.M, (int)threadIdx.x & 63};
  const int tiles_m = by_group.count(), tiles = tiles_m * tiles_n, per = (tiles + 7) >> 3;
  if ((int)blockIdx.x >= 8 * per) return;
  const int bid = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (bid >= tiles) return;
  const int tm = bid / tiles_n, tn = bid - tm * tiles_n;
  int m0, m_end, group;
  if (!by_group.find(tm, group, m0, m_end)) return;
  const int rows = m_end - m0;
  if (rows <= 64) ring_tile<__bf16, 64, BN, false, false, 1, ROWS>(p, 0, group, m0, m_end, tn, nullptr, rw);
  else if (rows <= 128) ring_tile<__bf16, 128, BN, false, false, 1, ROWS>(p, 0, group, m0, m_end, tn, nullptr, rw);
  else if (rows <= 192) ring_tile<__bf16, 192, BN, false, false, 1, ROWS>(p, 0, group, m0, m_end, tn, nullptr, rw);
  else ring_tile<__bf16, 256, BN, false, false, 1, ROWS>(p, 0, group, m0, m_end, tn, nullptr, rw);
}

template <typename K>
hipError_t allow_lds(K kernel, int bytes, std::atomic<unsigned long long>& configured) {  // configured: one bit per device, the attribute is per device
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  const unsigned long long bit = dev < 64 ? 1ull << dev : 0;
  if (bit && (configured.load(std::memory_order_relaxed) & bit)) return hipSuccess;
  if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes)) return e;
  configured.fetch_or(bit, std::memory_order_relaxed);
  return hipSuccess;
}

template <typename T, int BM, int BN, bool B_KN, bool F32OUT, int BDIV, int ROWS>
hipError_t launch(hipStream_t stream, const MMArgs& p, size_t batch, const float* residual, const DmaRows& rw) {
  constexpr int LDS_BYTES = lds_bytes(BM, BN, BDIV == 3);  // the result's rows fit as well
  static_assert(LDS_BYTES >= BM * (BN * 2 + 8));
  static std::atomic<unsigned long long> configured{0};
  auto kernel = gemm_ring<T, BM, BN, B_KN, F32OUT, BDIV, ROWS>;
  if (hipError_t e = allow_lds(kernel, LDS_BYTES, configured)) return e;
  const int tiles_m = (p.M + BM - 1) / BM + rw.groups, tiles_n = (p.N + BN - 1) / BN;
  const size_t total = (batch * (size_t)tiles_m * tiles_n + 7) / 8 * 8 + (rw.groups ? 8 : 0);
  kernel<<<dim3((unsigned)total), dim3(64 * waves(BM)), LDS_BYTES, stream>>>(p, (int)batch, tiles_m, tiles_n, residual, rw);
  return hipGetLastError();
}

template <int BN, int ROWS>
hipError_t launch_groups(hipStream_t stream, const MMArgs& p, const DmaRows& rw) {
  constexpr int A = lds_bytes(64, BN), B = lds_bytes(128, BN), C = lds_bytes(192, BN), D = lds_bytes(256, BN);
  constexpr int AB = A > B ? A : B, CD = C > D ? C : D, LDS_BYTES = AB > CD ? AB : CD;
  static std::atomic<unsigned long long> configured{0};
  auto kernel = gemm_ring_groups<BN, ROWS>;
  if (hipError_t e = allow_lds(kernel, LDS_BYTES, configured)) return e;
  const int tiles_m = (p.M + 255) / 256 + rw.groups, tiles_n = (p.N + BN - 1) / BN;
  kernel<<<dim3((unsigned)(((size_t)tiles_m * tiles_n + 7) / 8 * 8 + 8)), dim3(512), LDS_BYTES, stream>>>(p, tiles_n, rw);
  return hipGetLastError();
}

template <typename T, bool F32OUT, int BDIV, int ROWS>
hipError_t launch_nt(hipStream_t stream, const MMArgs& p, size_t batch, int tile, const float* residual, const DmaRows& rw) {
  if constexpr (BDIV == 1) {
    if (tile == 129) return launch<T, 256, 128, false, F32OUT, BDIV, ROWS>(stream, p, batch, residual, rw);
  }
  if constexpr (ROWS == 1 || ROWS == 2) {
    if (tile == 193) return launch_groups<192, ROWS>(stream, p, rw);
    if (tile == 130) return launch_groups<128, ROWS>(stream, p, rw);
    if (tile == 97) return launch<T, 192, 192, false, F32OUT, BDIV, ROWS>(stream, p, batch, residual, rw);
  }
  if constexpr (ROWS == 1 || ROWS == 3) {
    if (tile == 16) return launch<T, 32, 32, false, F32OUT, BDIV, ROWS>(stream, p, batch, residual, rw);
  }
  if (tile == 65) return launch<T, 128, 128, false, F32OUT, BDIV, ROWS>(stream, p, batch, residual, rw);
  if (tile == 48) return launch<T, 64, 128, false, F32OUT, BDIV, ROWS>(stream, p, batch, residual, rw);
  return tile == 32 ? launch<T, 64, 64, false, F32OUT, BDIV, ROWS>(stream, p, batch, residual, rw) : hipErrorInvalidValue;
}
template <typename T>
hipError_t launch_plain(hipStream_t stream, const MMArgs& p, size_t batch, int tile, const float* residual, const DmaRows& rw) {
  if (!(p.b_cs == 1 && p.b_rs != 1)) return launch_nt<T, false, 1, 0>(stream, p, batch, tile, residual, rw);
  if (tile == 129) return launch<T, 256, 128, true, false, 1, 0>(stream, p, batch, residual, rw);
  if (tile == 65) return launch<T, 128, 128, true, false, 1, 0>(stream, p, batch, residual, rw);
  return tile == 48 ? launch<T, 64, 128, true, false, 1, 0>(stream, p, batch, residual, rw) : hipErrorInvalidValue;
}

}  // namespace

hipError_t gemm_ring_launch(hipStream_t stream, int dtype, DmaForm form, const MMArgs& p, size_t batch, int tile, const float* residual, const DmaRows& rw) {
  switch (form) {
    case DmaForm::ROWS: return launch_nt<__bf16, false, 1, 1>(stream, p, batch, tile, residual, rw);
    case DmaForm::ROWS_LOOKUP: return launch_nt<__bf16, false, 1, 3>(stream, p, batch, tile, residual, rw);
    case DmaForm::ROWS_GLU: return launch_nt<__bf16, false, 1, 2>(stream, p, batch, tile, residual, rw);
    case DmaForm::PLANES3: return launch_nt<__bf16, true, 3, 0>(stream, p, batch, tile, residual, rw);
    case DmaForm::PLAIN: break;
  }
  return dtype == UGHIP_F16 ? launch_plain<_Float16>(stream, p, batch, tile, residual, rw) : launch_plain<__bf16>(stream, p, batch, tile, residual, rw);
}

}  // namespace ughip
