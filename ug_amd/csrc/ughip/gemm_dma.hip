// 16-bit MFMA GEMM for gfx950 with one wave per SIMD: C[b] = A[b] x B[b], f32 accumulate, bf16 or f16.
//
//   block tile BM x BN (256 x 256, 256 x 192, 256 x 128 or 128 x 128), K tile 64, 4 waves laid out 2 x 2, each owning BM/2 x BN/2 of the result
//   (any M, N a multiple of 8: a last tile hangs over the end, reads the last row again and stores what exists):
//   (BM / 32) x (BN / 32) accumulators of 16 x 16 (v_mfma_f32_16x16x32: 4 registers each) live in the accumulation
//   registers -- all 256 of them for the largest tile, which a lone wave per SIMD can have -- and leave the
//   architectural registers to two sets of operand fragments; a K tile is two steps of 32: 16 (12, 8) fragment reads
//   feed 64 (32, 16) MFMAs, so the 128 x 128 tile is bound by its LDS reads like the register-staged kernel and is
//   there for products whose larger tiles would leave CUs idle.  The 16 x 16 x 32 shape moves a fifth less through the
//   register file per flop than 32 x 32 x 16 (half the accumulator traffic, twice the operand traffic); under this
//   kernel the chip is held back by power, and the same schedule on the larger shape ran 5-6 % slower.
//   global -> LDS with global_load_lds_dwordx4 (no staging registers), two 64 KiB stages.  The address unit of a CU
//   needs 16 cycles per such instruction and a K tile takes 64 of them, half the tile's time: they are dealt one by one
//   in front of MFMAs over as much of the tile as the stage they fill allows (see the two schedules in the kernel)
//   rhs [n, k]-major: operand fragments are 128-bit LDS reads of k-contiguous rows (XOR-swizzled chunks, conflict free);
//   rhs [k, n]-major: the tile stays [k][n] in LDS (32-byte pieces XOR-swizzled by k so that the reads meet no bank twice)
//   and ds_read_b64_tr_b16 hands every lane 4 consecutive k of its own column: no transposing pass through registers
//   the MFMA operands are swapped (B fragment first): a lane then holds 4 consecutive columns of one result row, the
//   epilogue packs them and goes through LDS so that the result leaves in 16-byte pieces of whole rows
//
// What bounds it: power first, then the address unit.  With U(-1, 1) operands the chip runs this kernel at 1.4-1.8 GHz
// of its 2.4 GHz by box (CU busy cycles against the kernel's duration), and the matrix pipes are busy 80 % of those
// cycles at 8192^3 (89 % with the DMAs taken out, 92 % with the fragment reads taken out as well: the loads cost MFMA
// issue slots, not waiting time -- warming L2 ahead of them or four stages of 32 k instead of two of 64 made it slower).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <type_traits>

#include "bf16_split.h"
#include "gemm_dma.h"
#include "internal.h"
#include "rows_prices.h"
#include "ughip.h"

namespace ughip {
namespace {

// The same in two halves with an MFMA between them as the wait state that the write of M0 needs.  The first half names M0
// as clobbered; nothing can tell the compiler that the second half reads it, so nothing it emits between the two may
// write M0.  This kernel has no instruction that would (no LDS instruction of gfx950 needs M0); the build is held to that
// by a test that reads the compiler's assembly of this file (every global_load_lds is preceded by our own write of M0
// with exactly one MFMA and no other mention of M0 between), and the tests that hold the results bit for bit against the
// register-staged kernel's would show a load gone astray.
__device__ __forceinline__ void dma16_m0(unsigned lds_byte_addr, unsigned stage_offset) {
  asm volatile("s_add_u32 m0, %0, %1" : : "s"(lds_byte_addr), "s"(stage_offset) : "memory", "scc", "m0");
}
__device__ __forceinline__ void dma16_go(const void* base, unsigned voff) { asm volatile("global_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(base) : "memory"); }

// z / (1 + exp(-z)) with no more error than expf and a division give it, in three quarters of their instructions (an epilogue has nothing to hide
// them behind): t = -z log2(e) rounded and what is left of -z beside t ln 2, s; 2^t (1 + s), rounded, and what that leaves; a quotient from the reciprocal, corrected by its remainder once.
// All at a quarter of their size, so that no reciprocal of a finite 1 + exp(-z) is subnormal (z from -88.7 to -87.3).  The limits stand for what the remainders are where t or the quotient is infinite:
// they change no finite one.  Emulated with every step rounded (exp2 and reciprocal to nearest): 1.92 units of the last place at most and 4.03e-8 rms over N(0, 1), as expf and a division do; a
// sum of rounded terms times a reciprocal after a step of Newton's, 13 instructions for 17, 3.27 and 4.93e-8.
__device__ __forceinline__ float silu_32(float z) {
  constexpr float L2E = 1.44269502162933349609375f, LN2_HI = 0.693147182464599609375f, LN2_LO = -1.90465429995776e-9f, MOST = 3.402823466e38f;
  const float t = -z * L2E, zs = 0.25f * z;
  const float s = __builtin_amdgcn_fmed3f(__builtin_fmaf(-t, LN2_LO, __builtin_fmaf(-t, LN2_HI, -z)), -1e-3f, 1e-3f);
  const float p = 0.25f * __builtin_amdgcn_exp2f(t), e = __builtin_fmaf(p, s, p), e_left = __builtin_fmaf(p, s, p - e);
  const float d = 0.25f + e, q = __builtin_amdgcn_rcpf(d), y = zs * q;
  const float left = __builtin_fmaf(-e_left, y, __builtin_fmaf(-d, y, zs));
  return __builtin_fmaf(__builtin_amdgcn_fmed3f(left, -MOST, MOST), q, y);
}

// Lane l feeds row / column l % 16, k = 8 (l / 16) .. + 7 of a step of 32.  TWO: the schedule with two barriers per K tile.
// F32OUT: the result leaves as f32 (+ residual when given) instead of as T, through LDS either way.
// BDIV > 1 ([n, k]-major rhs): K tile t of the lhs meets K tile t / BDIV of the rhs -- an lhs that holds BDIV planes of every
// 64 columns side by side (a row split into bf16 terms) against one matrix, whose tile is loaded once for the three planes of one of the lhs (SHARED, below).
// BDIV == 6 (either rhs layout): both operands hold three planes (hi, mid, lo: planes 0, 1, 2) of every 64 elements of k side
// by side, and K tile t of the loop is term t % 6 of k tile t / 6 of an f32 product taken as six bf16 ones -- (hi, lo),
// (lo, hi), (mid, mid), (hi, mid), (mid, hi), (hi, hi), the small ones first; (mid, lo), (lo, mid) and (lo, lo) stay below
// 2^-24 of the product and are left out.
// ROWS (1, or 2 with SwiGLU): the lhs rows, the matrix and the result are those of DmaRows.  ROWS 4: planes of rows against gate rows then up rows,
// silu(gate) * up out (DmaRows: dst, n_out, dst_bf16 for the three planes of rows of n_out elements, else f32).
template <typename T, int BM, int BN, bool B_KN, bool TWO, bool F32OUT = false, int BDIV = 1, int ROWS = 0>
__global__ void __launch_bounds__(256) gemm_dma4(MMArgs p, int tiles_m, int tiles_n, const float* __restrict__ residual, DmaRows rw) {
  static_assert(ROWS == 0 || ROWS == 4 || (BDIV == 1 && !B_KN && !F32OUT), "rows: one plane against an [n, k]-major rhs");
  static_assert(ROWS != 4 || (BDIV == 3 && BN == 192 && F32OUT), "gated planes: 96 columns of three planes are what LDS takes on the way out");
  constexpr bool GATED = ROWS == 2 || ROWS == 4, BY_ROW = ROWS == 1 || ROWS == 2;
  static_assert(BDIV != 3 || TWO, "shared rhs tiles are scheduled with two barriers");
  static_assert(BDIV == 1 || BDIV == 6 || !B_KN, "planes of the lhs alone: against an [n, k]-major rhs only");
  static_assert(BN != 192 || (!B_KN && (F32OUT || BY_ROW)), "192 columns: neither the swizzle of an n-contiguous tile nor the way out of whole tiles through LDS divides them");
  extern __shared__ u32x4 lds[];
  constexpr int NI = BM / 32, NJ = BN / 32;            // 16-row and 16-column fragments per wave
  constexpr int NM = NI * NJ;                          // MFMAs per k32 step
  constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2, STAGE_BYTES = A_BYTES + B_BYTES;
  constexpr int NDA = BM / 32, NDB = BN / 32, ND = NDA + NDB;  // DMA instructions per wave and K tile
  // SHARED: the three planes of a lhs tile meet one rhs tile, which is loaded once for them, into a place of its own behind the lhs stages, and whose fragments stay in registers.
  constexpr bool SHARED = BDIV == 3;
  constexpr int A_STAGE = SHARED ? A_BYTES : STAGE_BYTES, B_AT = SHARED ? 2 * A_BYTES : A_BYTES, B_STAGE = SHARED ? 0 : STAGE_BYTES;
  constexpr int R = NI + NJ;                           // fragment reads per step
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // Block ids go round-robin over the 8 XCDs: id -> (id % 8) * (grid / 8) + id / 8 hands every XCD a contiguous run of
  // tiles, and tiles are numbered in super-rows of 4 tile rows, column by column inside, so that such a run is a 4-row
  // block: its workgroups share few A and B panels in their XCD's L2.
  int bid = blockIdx.x;
  GroupTiles<BM> by_group{rw.group_end, rw.groups, p.M, lane};
  if constexpr (BY_ROW) {
    if (rw.groups) {
      // how many tile rows there are is known here only: the workgroups past them leave before the runs are dealt
      const int rows = by_group.count();
      const int tiles = rows * tiles_n, per = (tiles + 7) >> 3;
      if (bid >= 8 * per) return;
      bid = (bid & 7) * per + (bid >> 3);
      if (bid >= tiles) return;
      tiles_m = rows;
    } else if ((gridDim.x & 7) == 0) {
      bid = (bid & 7) * (int)(gridDim.x >> 3) + (bid >> 3);
    }
  } else if ((gridDim.x & 7) == 0) bid = (bid & 7) * (int)(gridDim.x >> 3) + (bid >> 3);
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
  const int n0 = tn * BN;
  if (BY_ROW && rw.groups && !by_group.find(tm, group, m0, m_end)) return;  // the same for the whole workgroup
  const long long lda = p.a_rs, ldb = B_KN ? p.b_rs : p.b_cs;
  const char* Ab = reinterpret_cast<const char*>(static_cast<const T*>(p.a) + (size_t)batch * p.a_bs + (BY_ROW ? 0 : (size_t)m0 * lda));
  const char* Bb = reinterpret_cast<const char*>(static_cast<const T*>(p.b) + (size_t)batch * p.b_bs + (BY_ROW ? (size_t)group * rw.w_group : 0) +
                                                 (GATED ? 0 : B_KN ? (size_t)n0 : (size_t)n0 * ldb));
  const int KT = p.K / BK;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const unsigned lds_addr = (unsigned)(size_t)(__attribute__((address_space(3))) char*)lds;
  // per-lane byte offsets of this wave's DMA instructions (the same for every K tile; the scalar base moves)
  unsigned voff[ND];
  // a last tile may hang over the end of M or N: rows past the end fetch the last row again (their results are not
  // stored), so every address stays inside the operands
  const int m_last = m_end - 1 - m0, n_left = p.N - n0;
#pragma unroll
  for (int i = 0; i < NDA; ++i) {
    const int row = (i * 4 + wave) * 8 + (lane >> 3), cp = lane & 7;
    int src = min(row, m_last);
    if constexpr (BY_ROW) {
      src += m0;
      if (rw.row_index) src = max(0, min(rw.row_index[src], rw.x_rows - 1));
    }
    voff[i] = (unsigned)(src * lda * 2 + ((cp ^ ((row >> 1) & 7)) << 4));
  }
#pragma unroll
  for (int i = 0; i < NDB; ++i) {
    const int g = i * 4 + wave;
    if (!B_KN) {
      const int row = g * 8 + (lane >> 3), cp = lane & 7;
      int src = min(row, n_left - 1);
      if constexpr (GATED) {  // a wave's half of the tile: BN / 4 gate columns, then the same columns of up
        const int q = row % (BN / 2);
        src = min(tn * (BN / 2) + row / (BN / 2) * (BN / 4) + q % (BN / 4), rw.n_out - 1) + (q >= BN / 4 ? rw.n_out : 0);
      }
      voff[NDA + i] = (unsigned)(src * ldb * 2 + ((cp ^ ((row >> 1) & 7)) << 4));
    } else {
      // one instruction fills 1 KB = 512 / BN rows of k; the lane at LDS position (k, 16-byte chunk cpos) fetches the
      // chunk that the swizzle of the row's 32-byte pieces maps there
      constexpr int CPR = BN / 8;  // 16-byte chunks per row
      const int k = g * (64 / CPR) + lane / CPR, cpos = lane % CPR;
      const int src = (((cpos >> 1) ^ kn_h(k)) << 1) | (cpos & 1);
      voff[NDA + i] = (unsigned)(k * ldb * 2 + (min(src, n_left / 8 - 1) << 4));  // N % 8 == 0: whole 16-byte chunks
    }
  }
  const long long a_step = BK * 2, b_step = B_KN ? (long long)BK * ldb * 2 : BK * 2;
  auto dma = [&](int tile, int idx) {  // idx: compile-time after unrolling
    if (idx < NDA) dma16(Ab + lhs_k_tile<BDIV>(tile) * a_step, voff[idx], lds_addr + (tile & 1) * A_STAGE + (idx * 4 + wave) * 1024);
    else dma16(Bb + rhs_k_tile<BDIV>(tile) * b_step, voff[idx], lds_addr + (tile & 1) * B_STAGE + B_AT + ((idx - NDA) * 4 + wave) * 1024);
  };
  auto dma_m0 = [&](int tile, int idx) {
    const unsigned in_stage = lds_addr + (idx < NDA ? (idx * 4 + wave) * 1024 : B_AT + ((idx - NDA) * 4 + wave) * 1024);  // loop invariant
    dma16_m0(in_stage, (tile & 1) * (idx < NDA ? A_STAGE : B_STAGE));
    // the MFMA that follows in the source has to follow in the code: without this the compiler may hoist it above the
    // write of M0, and the load would then come right behind that write, without the wait state it needs
    __builtin_amdgcn_sched_barrier(0);
  };
  auto dma_go = [&](int tile, int idx) {
    if (idx < NDA) dma16_go(Ab + lhs_k_tile<BDIV>(tile) * a_step, voff[idx]);
    else dma16_go(Bb + rhs_k_tile<BDIV>(tile) * b_step, voff[idx]);
  };

  floatx4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  u32x4 fa[2][NI], fb[2][NJ];
  auto read_frag = [&](int stage, int s, int idx, int set) {
    if (idx < NI) {
      fa[set][idx] = lds[stage * (A_STAGE / 16) + kc_idx(wm + idx * 16 + (lane & 15), 4 * s + (lane >> 4))];
    } else if (!B_KN) {
      fb[set][idx - NI] = lds[stage * (B_STAGE / 16) + B_AT / 16 + kc_idx(wn + (idx - NI) * 16 + (lane & 15), 4 * s + (lane >> 4))];
    } else {
      // lane q + 4 e of a 16-lane group names row k0 + e, columns 4 q .. 4 q + 3 of the fragment's 16: lane i receives
      // k0 .. k0 + 3 of column i; group g takes k = 8 g .. 8 g + 7 of the step in two such reads
      typedef __attribute__((address_space(3))) s16x4 lds_v4;
      const int g = lane >> 4, li = lane & 15, q = li & 3, e = li >> 2;
      const char __attribute__((address_space(3)))* Bs = (const char __attribute__((address_space(3)))*)lds + stage * STAGE_BYTES + A_BYTES;
      const int n = wn + (idx - NI) * 16 + 4 * q, k0 = s * 32 + 8 * g + e;
      const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(Bs + kn_byte<BN>(k0, n))));
      const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4*)(Bs + kn_byte<BN>(k0 + 4, n))));
      fb[set][idx - NI] = u32x4{lo.x, lo.y, hi.x, hi.y};
    }
  };

  // prologue: tiles 0 and 1 requested, tile 0 landed (tile 1 is waited for at the first barrier that publishes it)
#pragma unroll
  for (int i = 0; i < ND; ++i) dma(0, i);
  constexpr int ND1 = SHARED ? NDA : ND;  // (tile 1 meets tile 0's rhs)
#pragma unroll
  for (int i = 0; i < ND1; ++i) dma(1, i);
  wait_vmcnt<ND1>();
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < R; ++i) read_frag(0, 0, i, 0);

  // One barrier per K tile.  Step 0 carries the fragment reads of step 1; step 1 starts behind the barrier that frees
  // this tile's stage and carries the reads of the next tile's step 0 (RN) and all the DMAs of tile kt + 2 (D), which
  // then have a whole step's time to land.  (The memory instructions are pinned one by one in front of MFMAs: a wave
  // alone on its SIMD has nobody to hide a burst of loads behind.)
  auto tile_one = [&](int kt, auto d, auto rn) {
    constexpr bool D = decltype(d)::value, RN = decltype(rn)::value;
    const int cur = kt & 1, nxt = cur ^ 1;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int fc = s, fn = s ^ 1;
      if (s == 1) {
        wait_vmcnt<0>();
        wait_lgkmcnt0();
        __builtin_amdgcn_s_barrier();
      }
      const int n_reads = (s == 0 || RN) ? R : 0, n_dmas = (s == 1 && D) ? ND : 0;
      const int n_ops = n_reads + n_dmas;
#pragma unroll
      for (int g = 0; g < NM; ++g) {
        // the memory instructions in front of MFMA g: those t with t * NM / n_ops == g
        constexpr int PER = (R + ND + NM - 1) / NM;
        static_assert(PER == 1, "at most one memory instruction per MFMA: M0 is written one MFMA ahead of its DMA");
        const int t_lo = (g * n_ops + NM - 1) / NM, t_hi = ((g + 1) * n_ops + NM - 1) / NM;
#pragma unroll
        for (int u = 0; u < PER; ++u) {
          const int t = t_lo + u;
          if (t < t_hi) {
            // reads and DMAs of a step are dealt in proportion: op t is DMA number t * n_dmas / n_ops when that number moves
            const int di = t * n_dmas / n_ops, di_next = (t + 1) * n_dmas / n_ops;
            const bool is_dma = di_next > di;
            const int ri = t - di;
            if (is_dma) dma_m0(kt + 2, di);  // M0 in front of this MFMA, the load behind it: the MFMA is the wait state M0 needs
            else read_frag(s == 0 ? cur : nxt, s == 0 ? 1 : 0, ri, fn);
          }
        }
        const int i = g / NJ, j = g % NJ;
        acc[i][j] = mma16(T(), fb[fc][j], fa[fc][i], acc[i][j]);  // operands swapped: rows of the block are columns of C
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < PER; ++u) {
          const int t = t_lo + u;
          if (t < t_hi) {
            const int di = t * n_dmas / n_ops, di_next = (t + 1) * n_dmas / n_ops;
            if (di_next > di) dma_go(kt + 2, di);
          }
        }
      }
    }
  };
  // Two barriers per K tile, so that the DMAs need not all come in one step (64 x 16 cycles of the address unit
  // against the 1024 cycles of a step's MFMAs): 2-3 % faster with an [n, k]-major rhs.  Step 0 reads the fragments of
  // step 1 in front of its first R MFMAs; barrier A, in front of MFMA BAR, then says that nobody reads this tile's
  // stage any more, and the DMAs of tile kt + 2 go out from there to the end of step 1, evenly (EARLY of them in
  // step 0).  Barrier B, at the head of step 1, says that tile kt + 1 has landed (its last DMA went out a whole step
  // ago; the EARLY ones behind it may still be on their way).
  auto tile_two = [&](int kt, auto d, auto rn) {
    constexpr bool D = decltype(d)::value, RN = decltype(rn)::value;
    constexpr int BAR = (R + 4 > NM * 3 / 8 ? R + 4 : NM * 3 / 8) < NM - 1 ? (R + 4 > NM * 3 / 8 ? R + 4 : NM * 3 / 8) : NM - 1;
    constexpr int EARLY = ND * (NM - BAR) / (2 * NM - BAR);
    static_assert(R + ND - EARLY <= NM, "at most one memory instruction per MFMA: M0 is written one MFMA ahead of its DMA");
    const int cur = kt & 1, nxt = cur ^ 1;
#pragma unroll
    for (int g = 0; g < NM; ++g) {
      if (g < R) read_frag(cur, 1, g, 1);
      if (g == BAR) {
        wait_lgkmcnt0();
        __builtin_amdgcn_s_barrier();
      }
      if (D && g > BAR && EARLY > 0) {
        // DMA e goes out in front of the MFMA after this one; M0 is written in front of this one
        const int e = (g - BAR - 1) * EARLY / (NM - BAR - 1), e_next = (g - BAR) * EARLY / (NM - BAR - 1);
        if (e_next > e && e < EARLY) dma_m0(kt + 2, e);
      }
      const int i = g / NJ, j = g % NJ;
      acc[i][j] = mma16(T(), fb[0][j], fa[0][i], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
      if (D && g > BAR && EARLY > 0) {
        const int e = (g - BAR - 1) * EARLY / (NM - BAR - 1), e_next = (g - BAR) * EARLY / (NM - BAR - 1);
        if (e_next > e && e < EARLY) dma_go(kt + 2, e);
      }
    }
    if (RN) {
      if (D) wait_vmcnt<EARLY>();
      else wait_vmcnt<0>();
      __builtin_amdgcn_s_barrier();
    }
    const int n_reads = RN ? R : 0, n_dmas = D ? ND - EARLY : 0;
    const int n_ops = n_reads + n_dmas;
#pragma unroll
    for (int g = 0; g < NM; ++g) {
      constexpr int PER = (R + ND + NM - 1) / NM;
      const int t_lo = (g * n_ops + NM - 1) / NM, t_hi = ((g + 1) * n_ops + NM - 1) / NM;
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int t = t_lo + u;
        if (t < t_hi) {
          const int di = t * n_dmas / n_ops, di_next = (t + 1) * n_dmas / n_ops;
          if (di_next > di) dma_m0(kt + 2, EARLY + di);
          else read_frag(nxt, 0, t - di, 0);
        }
      }
      const int i = g / NJ, j = g % NJ;
      acc[i][j] = mma16(T(), fb[1][j], fa[1][i], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < PER; ++u) {
        const int t = t_lo + u;
        if (t < t_hi) {
          const int di = t * n_dmas / n_ops, di_next = (t + 1) * n_dmas / n_ops;
          if (di_next > di) dma_go(kt + 2, EARLY + di);
        }
      }
    }
  };
  // SHARED, with those two barriers: tile kt is plane P of its rhs tile.  The rhs fragments of step 1 are read with plane 0's first step and those of step 0 with plane 2's second one, where
  // the registers of the rhs tile before have had their last use; from plane 0's barrier A on nobody reads that tile in LDS any more, and the next one's loads go out behind it, a half each with
  // planes 0 and 1 (b).  Of loads and fragment reads it has three tenths less than tile by tile (10 loads a tile for 14, 20
  // reads for 28 on 256 x 192), and the chip, held back by power, its clock: llama's gate and up of 1900 rows 228 -> 215 us, down 106 -> 99, q | k | v 63.7 -> 61.  The order of the sums is the same.
  auto tile_shared = [&](int kt, auto plane, auto d, auto rn, auto b) {
    constexpr int P = decltype(plane)::value;
    constexpr bool D = decltype(d)::value, RN = decltype(rn)::value;
    constexpr int R0 = NI + (P == 0 ? NJ : 0), R1 = RN ? NI + (P == 2 ? NJ : 0) : 0;
    constexpr int NB0 = NDB / 2, B_FIRST = P == 1 ? NB0 : 0, NB = !decltype(b)::value || P == 2 ? 0 : P == 0 ? NB0 : NDB - NB0;
    constexpr int NA = D ? NDA : 0, N = NA + NB;
    constexpr int LOW = R0 + 4 > NM * 3 / 8 ? R0 + 4 : NM * 3 / 8, BAR = LOW < NM - 1 ? LOW : NM - 1;
    constexpr int EARLY = N * (NM - BAR) / (2 * NM - BAR), LATE = N - EARLY, OPS = R1 + LATE;
    static_assert(R0 <= NM && OPS <= NM && EARLY <= NM - BAR - 1, "at most one memory instruction per MFMA: M0 is written one MFMA ahead of its DMA");
    const int cur = kt & 1, nxt = cur ^ 1;
    // load e of this tile: the lhs of tile kt + 2 first, then its share of the next rhs tile
    auto m0_of = [&](int e) { e < NA ? dma_m0(kt + 2, e) : dma_m0(kt + 3 - P, NDA + B_FIRST + e - NA); };
    auto go_of = [&](int e) { e < NA ? dma_go(kt + 2, e) : dma_go(kt + 3 - P, NDA + B_FIRST + e - NA); };
#pragma unroll
    for (int g = 0; g < NM; ++g) {
      if (g < R0) read_frag(cur, 1, g, 1);
      if (g == BAR) {
        wait_lgkmcnt0();
        __builtin_amdgcn_s_barrier();
      }
      const int e = EARLY > 0 && g > BAR ? (g - BAR - 1) * EARLY / (NM - BAR - 1) : 0, e_next = EARLY > 0 && g > BAR ? (g - BAR) * EARLY / (NM - BAR - 1) : 0;
      const bool load = e_next > e && e < EARLY;
      if (load) m0_of(e);
      acc[g / NJ][g % NJ] = mma16(T(), fb[0][g % NJ], fa[0][g / NJ], acc[g / NJ][g % NJ]);
      __builtin_amdgcn_sched_barrier(0);
      if (load) go_of(e);
    }
    if (RN) {
      wait_vmcnt<EARLY>();
      __builtin_amdgcn_s_barrier();
    }
#pragma unroll
    for (int g = 0; g < NM; ++g) {
      const int t = (g * OPS + NM - 1) / NM, t_hi = ((g + 1) * OPS + NM - 1) / NM;
      const int di = OPS ? t * LATE / OPS : 0, di_next = OPS ? (t + 1) * LATE / OPS : 0;
      const bool load = t < t_hi && di_next > di;
      if (load) m0_of(EARLY + di);
      else if (t < t_hi) read_frag(nxt, 0, t - di, 0);
      acc[g / NJ][g % NJ] = mma16(T(), fb[1][g % NJ], fa[1][g / NJ], acc[g / NJ][g % NJ]);
      __builtin_amdgcn_sched_barrier(0);
      if (load) go_of(EARLY + di);
    }
  };
  auto tile = [&](int kt, auto d, auto rn) {
    if constexpr (TWO) tile_two(kt, d, rn);
    else tile_one(kt, d, rn);
  };
  using Y = std::true_type;
  using N_ = std::false_type;
  if constexpr (SHARED) {
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    using P2 = std::integral_constant<int, 2>;
    for (int kt = 0; kt < KT - 3; kt += 3) {
      tile_shared(kt, P0(), Y(), Y(), Y());
      tile_shared(kt + 1, P1(), Y(), Y(), Y());
      tile_shared(kt + 2, P2(), Y(), Y(), Y());
    }
    tile_shared(KT - 3, P0(), Y(), Y(), N_());
    tile_shared(KT - 2, P1(), N_(), Y(), N_());
    tile_shared(KT - 1, P2(), N_(), N_(), N_());
  } else {
    for (int kt = 0; kt < KT - 2; ++kt) tile(kt, Y(), Y());
    tile(KT - 2, N_(), Y());
    tile(KT - 1, N_(), N_());
  }

  // Register e of lane l of block (i, j): row wm + 16 i + l % 16, column wn + 16 j + 4 (l / 16) + e.
  if constexpr (ROWS == 4) {
    // As the fold of slabs has it: silu(gate) * up of the f32 sums, rounded to f32, then its three terms.  In registers it saves the f32 sums' way to memory and back and the
    // launch that folds them: gate and up of 1900 rows, n 2 x 5632, k 2048, 218 us and a fold of 24 -> 228.  The ten are the vector instructions of two rounds of tiles, which a
    // lone wave per SIMD has nothing to hide behind (19 with expf, a division and a store's place worked out for every piece).
    constexpr int NC = NJ / 2, COLS = BN / 2;
    auto gated = [&](int i, int j, int e) {
      float y = silu_32(acc[i][j][e]) * acc[i][j + NC][e];
      asm("" : "+v"(y));  // the terms of the f32 value, as if it had been stored
      return y;
    };
    if (!rw.dst_bf16) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NC; ++j) {
          const int row = wm + i * 16 + (lane & 15), col = tn * COLS + (wave & 1) * (COLS / 2) + j * 16 + (lane >> 4) * 4;
          if (row <= m_last && col < rw.n_out)
            *reinterpret_cast<floatx4*>(static_cast<float*>(rw.dst) + (size_t)(m0 + row) * rw.n_out + col) = floatx4{gated(i, j, 0), gated(i, j, 1), gated(i, j, 2), gated(i, j, 3)};
        }
      return;
    }
    // rows of [hi | mid | lo], 96 columns each, through LDS: 16 rows of a wave's writes start in 16 different groups of four banks
    constexpr int PITCH = 3 * COLS * 2 + 16, CHUNKS = COLS / 8;
    char __attribute__((address_space(3)))* Cs = (char __attribute__((address_space(3)))*)lds;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        u32x2 hi, mid, lo;
        unsigned h, m, l;
        split3_pair(gated(i, j, 0), gated(i, j, 1), h, m, l);
        hi.x = h, mid.x = m, lo.x = l;
        split3_pair(gated(i, j, 2), gated(i, j, 3), h, m, l);
        hi.y = h, mid.y = m, lo.y = l;
        char __attribute__((address_space(3)))* at = Cs + (wm + i * 16 + (lane & 15)) * PITCH + ((wave & 1) * (COLS / 2) + j * 16 + (lane >> 4) * 4) * 2;
        *(u32x2 __attribute__((address_space(3)))*)at = hi;
        *(u32x2 __attribute__((address_space(3)))*)(at + COLS * 2) = mid;
        *(u32x2 __attribute__((address_space(3)))*)(at + COLS * 4) = lo;
      }
    __syncthreads();
    // three quarters of the threads, so that a pass is 16 whole rows of a plane and a thread's place in the row stays
    const int c = tid % CHUNKS, r0 = tid / CHUNKS, col = tn * COLS + c * 8;
    if (r0 >= 16 || col >= rw.n_out) return;  // n_out % 64 == 0: whole chunks
    uint16_t* __restrict__ X3 = static_cast<uint16_t*>(rw.dst) + (size_t)(m0 + r0) * 3 * rw.n_out + col / 64 * 192 + col % 64;
    const char __attribute__((address_space(3)))* from = Cs + r0 * PITCH + c * 16;
#pragma unroll
    for (int pass = 0; pass < BM / 16; ++pass) {
      if (pass * 16 + r0 > m_last) break;
#pragma unroll
      for (int plane = 0; plane < 3; ++plane)
        *reinterpret_cast<u32x4*>(X3 + plane * 64) = *(const u32x4 __attribute__((address_space(3)))*)(from + pass * 16 * PITCH + plane * COLS * 2);
      X3 += (size_t)48 * rw.n_out;
    }
    return;
  }
  static_assert(2 * A_BYTES + (SHARED ? 1 : 2) * B_BYTES >= 4 * (NI > 1 ? 2 : 1) * 16 * (BN / 2 * 4 + 16), "what rows and f32 sums leave by: pieces of 16 rows of a wave's columns");
  if constexpr (BY_ROW) {
    rows_out<T, ROWS>(acc, rw, m0, m_last, wm, ROWS == 2 ? tn * (BN / 2) + (wave & 1) * (BN / 4) : n0 + wn, wave, lds);
    return;
  }
  if constexpr (F32OUT) {
    const size_t at = (size_t)batch * p.c_bs + (size_t)m0 * p.N + n0;
    sums_out(acc, static_cast<float*>(p.c) + at, residual ? residual + at : nullptr, p.N, m_last, n_left, wm, wn, wave, lds);
    return;
  }
  // Epilogue through LDS.
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
  constexpr int CPR = BN / 8, RPP = 256 / CPR;
  T* __restrict__ C = static_cast<T*>(p.c) + (size_t)batch * p.c_bs + (size_t)m0 * p.N + n0;
  const int c = tid % CPR, r0 = tid / CPR;
#pragma unroll 4
  for (int pass = 0; pass < BM / RPP; ++pass) {
    const int row = pass * RPP + r0;
    const u32x2 lo = *(const u32x2 __attribute__((address_space(3)))*)(Cs + row * PITCH + c * 16);
    const u32x2 hi = *(const u32x2 __attribute__((address_space(3)))*)(Cs + row * PITCH + c * 16 + 8);
    // past the cache: nobody in this launch reads the result, and 256 CUs that store their tiles at the same moment are
    // through sooner when L2 does not hold the lines for the write-back at the kernel's end (8 x 1024^3: 18.7 -> 17.5 us)
    if (row <= m_last && c * 8 < n_left) __builtin_nontemporal_store(u32x4{lo.x, lo.y, hi.x, hi.y}, reinterpret_cast<u32x4*>(C + (size_t)row * p.N + c * 8));
  }
}

template <typename T, int BM, int BN, bool B_KN, bool F32OUT = false, int BDIV = 1, int ROWS = 0>
hipError_t launch(hipStream_t stream, const MMArgs& p, size_t batch, const float* residual = nullptr, const DmaRows& rw = DmaRows()) {
  constexpr int STAGES = (BDIV == 3 ? 2 * BM + BN : 2 * (BM + BN)) * BK * 2, EPI = ROWS == 4 ? BM * (3 * BN + 16) : F32OUT || ROWS ? 0 : BM * (BN * 2 + 8);
  constexpr int LDS_BYTES = STAGES > EPI ? STAGES : EPI;
  static std::atomic<unsigned long long> configured{0};  // one bit per device: the attribute is per device
  // the schedule with two barriers, except where it does not fit the registers (the transposing reads of the
  // largest tile need pairs of temporaries: 256 registers and spills)
  constexpr bool TWO = !(B_KN && BM == 256 && BN == 256);
  auto kernel = gemm_dma4<T, BM, BN, B_KN, TWO, F32OUT, BDIV, ROWS>;
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  const unsigned long long bit = dev < 64 ? 1ull << dev : 0;
  if (!bit || !(configured.load(std::memory_order_relaxed) & bit)) {
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES)) return e;
    configured.fetch_or(bit, std::memory_order_relaxed);
  }
  const int tiles_m = (p.M + BM - 1) / BM + rw.groups, tiles_n = (p.N + BN - 1) / BN;
  // (8 more for groups: the kernel deals the tiles that exist in 8 equal runs)
  const size_t total = batch * (size_t)tiles_m * tiles_n + (rw.groups ? 8 : 0);
  kernel<<<dim3((unsigned)total), dim3(256), LDS_BYTES, stream>>>(p, tiles_m, tiles_n, residual, rw);
  return hipGetLastError();
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

namespace {
// tile codes of the entry points below: 256 = 256 x 256, 192 = 256 x 192 (three planes and rows), 128 = 256 x 128, 64 = 128 x 128; on gemm_ring 129 = 256 x 128, 65 = 128 x 128, 48 = 64 x 128,
// 32 = 64 x 64 ([n, k]-major rhs only), 97 = 192 x 192 (rows only), 16 = 32 x 32 (rows only, not gated), 193 / 130 = 256 x 192 / 256 x 128 and lower ones of that width (rows by group only)
bool tile_dims(int tile, int* bm, int* bn) {
  if (tile == 256) *bm = 256, *bn = 256;
  else if (tile == 192 || tile == 193) *bm = 256, *bn = 192;
  else if (tile == 128 || tile == 129 || tile == 130) *bm = 256, *bn = 128;
  else if (tile == 97) *bm = 192, *bn = 192;
  else if (tile == 64 || tile == 65) *bm = 128, *bn = 128;
  else if (tile == 48) *bm = 64, *bn = 128;
  else if (tile == 32) *bm = 64, *bn = 64;
  else if (tile == 16) *bm = 32, *bn = 32;
  else return false;
  return true;
}
}  // namespace

static size_t tile_count(const MMArgs& p, size_t batch, int tile) {  // 0: no such tile
  int bm, bn;
  return tile_dims(tile, &bm, &bn) ? batch * (size_t)((p.M + bm - 1) / bm) * (size_t)((p.N + bn - 1) / bn) : 0;
}
static bool by_height(int tile) { return tile == 193 || tile == 130; }  // rows by group: tiles of up to that height
static bool ring_tile(int tile) { return tile == 129 || by_height(tile) || tile == 97 || tile == 65 || tile == 48 || tile == 32 || tile == 16; }
static int least_k(int tile) { return ring_tile(tile) ? BK : 4 * BK; }
static const char* waves_name(int tile) { return tile == 16 ? "256t,ring" : ring_tile(tile) ? "512t,ring" : "256t"; }  // in the names of these kernels
// (tuning aid) the tile code that GEMM_SHAPE names, 0: none of these kernels'
int gemm_dma_forced_tile(long long shape) {
  switch (shape) {
    case 3: return 256;
    case 4: return 128;
    case 5: return 64;
    case 9: return 32;
    case 10: return 129;
    case 11: return 97;
    case 12: return 65;
    case 13: return 48;
    case 14: return 192;
    case 15: return 193;
    case 16: return 130;
    case 17: return 16;
  }
  return 0;
}

bool gemm_dma_supported(int dtype, const MMArgs& p, size_t batch, int tile) {
  if (dtype != UGHIP_BF16 && dtype != UGHIP_F16) return false;
  int bm, bn;
  if (!tile_dims(tile, &bm, &bn)) return false;
  if (p.M <= 0 || p.N <= 0 || p.N % 8 || p.K % BK || p.K < least_k(tile) || batch == 0) return false;
  if (p.a_cs != 1 || p.a_rs % 8 || (batch > 1 && (p.a_bs % 8 || p.b_bs % 8 || p.c_bs % 8))) return false;
  const bool nn = p.b_cs == 1 && p.b_rs != 1, nt = p.b_rs == 1 && p.b_cs != 1;
  if (nn == nt || (nn && tile == 32) || tile == 97 || tile == 16 || by_height(tile) || (tile == 192 && p.b_k_div != 3)) return false;
  const long long ldb = nn ? p.b_rs : p.b_cs;
  if (ldb % 8) return false;
  // per-lane offsets are 32-bit: the furthest row of a tile has to stay below 4 GiB from the tile's first byte
  if ((unsigned long long)p.a_rs * 2 * bm >= (1ull << 32) || (unsigned long long)ldb * 2 * (nn ? BK : bn) >= (1ull << 32)) return false;
  if (!aligned16(p.a) || !aligned16(p.b) || !aligned16(p.c)) return false;
  return batch * (size_t)((p.M + bm - 1) / bm) * (size_t)((p.N + bn - 1) / bn) < (1u << 24);
}

// What `tiles` tiles of the ring kernel take: a fixed part and, per round of 256 tiles, the K tiles.  The time of a K tile is mostly that of its
// bytes on their way to a CU, some 100 bytes per ns from the memory-side cache and 60 from HBM however many are asked for at once (operands from
// HBM: the kernel takes as long without its MFMAs), so it goes by where the operands come from.  MEMORY is a matrix nobody has read lately,
// as the weights of a model's next layer are; CACHE what a product finds whose operands were written or read just before.  Fitted to (m x n x k, us): 2048^2 x 5632 from memory 51 (128 x 128) / 67 (256 x 128), 1024 x 2048 x
// 5632 from memory 38 (64 x 128), 509 x 2048 x 5632 from memory 26 (64 x 64), 2048 x 11264 x 2048 from memory 89 (256 x 128), 700 x
// 11264 x 2048 from memory 34 and 1500 x 11264 x 2048 68 (192 x 192); 2048^3 19.2 (128 x 128),
// 1024 x 2048 x 4096 21.1 (64 x 128), 256 x 4096^2 14.7 (64 x 64), 584 x 360 x 6656 20.9 and 9 x 64 x 4416 13.2 (64 x 64).
enum class Operands { MEMORY, CACHE };
static double ring_cost_us(size_t tiles, int kt, int tile, Operands from) {
  const bool memory = from == Operands::MEMORY;
  // 32 x 32, two workgroups to a CU: 54 rows of 2048 x 5632 14.1, 228 of 2048 x 2048 9.8, 228 of 3072 x 768 7.6
  if (tile == 16) return 2.3 + kt * (0.135 + (tiles > 256 ? 0.09 * std::min(1.0, (tiles - 256.0) / 256) : 0) + (tiles > 512 ? 0.2 * (tiles - 512.0) / 256 : 0));
  const double t0 = tile == 129 ? 0.64 : tile == 97 ? 0.62 : tile == 65 ? (memory ? 0.54 : 0.30) : tile == 48 ? (memory ? 0.40 : 0.21) : memory ? 0.255 : 0.14;
  const double t1 = tile == 129 ? 0.22 : tile == 97 ? 0.30 : memory ? 0 : tile == 65 ? 0.17 : tile == 48 ? 0.07 : 0.045;
  double us = tile == 129 || tile == 97 ? 5.0 : tile == 65 ? 4.0 : 3.3;
  for (size_t left = tiles; left > 0; left -= left < 256 ? left : 256) us += kt * (t0 + t1 * (left < 256 ? (double)left : 256.0) / 256.0);
  return us;
}

// Which tile this kernel should take the problem with (a tile code), or 0 when the register-staged kernel is expected to
// be faster.  Both are priced.  This kernel: a fixed cost (launch and first tile, 4 us, and the result's way out at the
// rate of a stream) plus, per round of up to 256 workgroups, the K tiles at a time that grows with the share of the chip
// that is busy -- the chip is power-bound under this kernel, a half-empty round runs at a higher clock: 0.9 + 0.6 x busy
// us per K tile for 256 x 256, 0.62 + 0.2 x busy for 256 x 128, fitted to 4096^3 (108 us), 8 x 1024^3 (20), 3072 x 4096^2
// (92 / 112), 5120^2 x 1024 (54 / 65), 2048 x 2560 x 2048 (40 / 29), 2816^3 (58 / 44), 1280 x 8192 x 2048 (46), 2048^2 x 5632
// (97 / 72).  The other kernel: the model that chooses its own tiles.  Against "256 x 256 tiles when they number 200 or
// more, else 256 x 128 under the same rule" this moves products with 130-250 tiles or a short last round to this kernel
// (3072 x 4096^2: 131 -> 91 us, 5120^2 x 1024: 77 -> 54, 1280 x 8192 x 2048: 64 -> 47, 2048 x 2560 x 2048: 35 -> 29,
// 2304^3: 39 -> 35) and leaves those with about 128 tiles where they were (2048^2 x 5632: 56 us against 72).  The
// 128 x 128 tile (two workgroups per CU) takes what neither fits: 2304^3 35 -> 31 us, 2048 x 2560 x 2048 29 -> 27.
// UGHIP_GEMM_SHAPE=3 / 4 / 5 forces 256 x 256 / 256 x 128 / 128 x 128 where the kernel applies, 10 / 12 / 13 / 9 the ring's 256 x 128 / 128 x 128 / 64 x 128 / 64 x 64, 0..2, 6 and 7 keep both out (tuning aid).
double gemm_dma_cost_us(const MMArgs& p, size_t batch, int tile) {
  const size_t tiles = tile_count(p, batch, tile);
  if (!tiles) return 1e30;
  const int kt = p.K / BK;
  const bool nn = p.b_cs == 1 && p.b_rs != 1;
  if (ring_tile(tile))
    return ring_cost_us(tiles, kt, tile, Operands::CACHE) * (nn ? 1.1 : 1.0) + (double)batch * p.M * p.N * 2 / 6.4e6;
  double us = 4.0 + (double)batch * p.M * p.N * 2 / 6.4e6;
  // (the figures below were fitted to the kernel on 32 x 32 x 16 MFMAs; on 16 x 16 x 32 and with the loads spread behind two
  // barriers every K tile takes 8 % less: 4096^3 97 us, 8 x 1024^3 18.8, 1024 x 4096^2 41 on 128 x 128 tiles)
  const double layout = (nn ? 1.08 : 1.0) * 0.92;
  if (tile == 64) {
    // two workgroups share a CU: a round is 512 tiles at 0.88 us per K tile; up to 256 tiles run one per CU at
    // 0.47 + 0.16 x busy, the next 256 fill the second slots (2048^3 24.7 us, 2304^3 31.3, 2816^3 45.5, 5120^2 x 1024 61)
    us += kt * 0.88 * (double)(tiles / 512) * layout;
    const size_t left = tiles % 512;
    if (left > 256) us += kt * (0.63 + 0.25 * (double)(left - 256) / 256.0) * layout;
    else if (left) us += kt * (0.47 + 0.16 * (double)left / 256.0) * layout;
    return us;
  }
  const double t0 = tile == 256 ? 0.9 : 0.62, t1 = tile == 256 ? 0.6 : 0.2;
  for (size_t left = tiles; left > 0; left -= left < 256 ? left : 256) {
    const double busy = (left < 256 ? (double)left : 256.0) / 256.0;
    us += kt * (t0 + t1 * busy) * layout;
  }
  return us;
}

int gemm_dma_pick(int dtype, const MMArgs& p, size_t batch) {
  if (long long s; tune_get(TUNE_GEMM_SHAPE, &s)) {
    const int forced = gemm_dma_forced_tile(s);
    return forced && gemm_dma_supported(dtype, p, batch, forced) ? forced : 0;
  }
  int best = 0;
  double best_us = 0;
  // The ring where 128 x 128 tiles would leave CUs without one (us by box, best of gemm_dma4 and gemm_tiled -> ring: 1024^3 [k, n]-major
  // 11.4 -> 7.9, 2048 x 1024^2 10.8 -> 8.2, 1024 x 2048 x 4096 28.7 -> 21.1 and 37.3 -> 24.5, 1536^3 16.2 -> 13.1, 96^2 x 4096 [k, n]-major 33 -> 15.4).
  // Past one round 2304^3 takes 29.2 in place of the ring's 33.4.  Three kinds of product keep their plans, which callers hold them to, though the
  // ring is the faster one for most of them (us there / ring): exactly one round of tiles (2048^3 23.5 / 20.0, 2048^2 x 5632 54.5 / 42.8, 4 x 1024^3 13.1 / 9.9);
  // [n, k]-major, up to 64 tiles, K up to 1024 (1024^3 10.3 / 6.3, 512^3 6.5 / 5.6, 64^2 x 1024 8.7 / 5.6, 64^2 x 128 6.2 / 5.6); up to 128 rows
  // whose K gemm_tiled splits (64 x 2048^2 10.8 / 7.7, 128 x 256 x 2048 9.8 / 7.8; 64 x 256 x 4096 11.5 / 12.5, 64 x 2048 x 4096 12.6 / 13.5).
  const size_t tiles = batch * (size_t)((p.M + 127) / 128) * (size_t)((p.N + 127) / 128);
  const bool few = tiles < 256 && !(p.b_rs == 1 && tiles <= 64 && p.K <= 1024) && !(p.M <= 128 && gemm_tiled_workspace_bytes(dtype, p, batch) != 0);
  for (int tile : {256, 128, 64, 65, 48, 32}) {
    if ((ring_tile(tile) && !few) || !gemm_dma_supported(dtype, p, batch, tile)) continue;
    const double us = gemm_dma_cost_us(p, batch, tile);
    if (!best || us < best_us * 0.97) best = tile, best_us = us;  // the larger tile on a near tie: fewer operand bytes
  }
  if (!best) return 0;
  if (ring_tile(best)) {
    // What gemm_tiled is priced at: 0-20 % below what [k, n]-major products take, up to a quarter above what those take whose K it splits (5 x 220 x 352
    // x 7488 18.8 us there, 23.0 here).  Operands that the memory-side cache cannot hold come from memory: 7 x 2512 x 64 x 5952, 215 MB, 51 us there, 64
    // here; 4 x 3760 x 64 x 8000, one round of tiles, 55 and 50.
    const double tiled = gemm_tiled_cost_us(dtype, p, batch);
    const bool memory = 2.0 * batch * p.K * ((double)p.M + p.N) > 192e6;
    if (memory) best_us = ring_cost_us(tile_count(p, batch, best), p.K / BK, best, Operands::MEMORY);
    return tiled < 0 || best_us < tiled * (!memory && gemm_tiled_workspace_bytes(dtype, p, batch) ? 0.945 : 1.0) ? best : 0;
  }
  // the 128 x 128 tile runs at the register-staged kernel's pace (both are bound by their LDS reads): it has to be
  // clearly cheaper to take the product from it
  const double other = gemm_tiled_cost_us(dtype, p, batch);
  return other < 0 || best_us < other * (best == 64 ? 0.95 : 1.0) ? best : 0;
}

void gemm_dma_name(int dtype, const MMArgs& p, int tile, char* out, size_t out_len) {
  int bm = 0, bn = 0;
  tile_dims(tile, &bm, &bn);
  const bool nn = p.b_cs == 1 && p.b_rs != 1;
  snprintf(out, out_len, "gemm_dma4<%s,%s,%dx%d,%s>", dtype == UGHIP_F16 ? "f16" : "bf16", nn ? "NN" : "NT", bm, bn, waves_name(tile));
}

hipError_t gemm_dma_launch(hipStream_t stream, int dtype, const MMArgs& p, size_t batch, int tile) {
  if (!gemm_dma_supported(dtype, p, batch, tile)) return hipErrorInvalidValue;
  int bm = 0, bn = 0;
  tile_dims(tile, &bm, &bn);
  const bool nn = p.b_cs == 1 && p.b_rs != 1;
  {
    char name[96];
    gemm_dma_name(dtype, p, tile, name, sizeof name);
    note_kernel("%s", name);
  }
  if (ring_tile(tile)) return gemm_ring_launch(stream, dtype, DmaForm::PLAIN, p, batch, tile, nullptr, DmaRows());
#define UGHIP_DMA_CASE(T)                                                                                                  \
  if (tile == 256) return nn ? launch<T, 256, 256, true>(stream, p, batch) : launch<T, 256, 256, false>(stream, p, batch); \
  if (tile == 128) return nn ? launch<T, 256, 128, true>(stream, p, batch) : launch<T, 256, 128, false>(stream, p, batch); \
  return nn ? launch<T, 128, 128, true>(stream, p, batch) : launch<T, 128, 128, false>(stream, p, batch);
  if (dtype == UGHIP_F16) {
    UGHIP_DMA_CASE(_Float16)
  }
  UGHIP_DMA_CASE(__bf16)
#undef UGHIP_DMA_CASE
}

// bf16 planes of f32 rows (three per 64 columns: p.K = 3 k, p.b_k_div = 3) against an [n, k]-major bf16 matrix, f32 result
// [M, N] (+ residual [M, N] when given), or nsplit slabs of it: the splits of K run as the kernel's batches, with the
// batch strides of the operands standing for a split's offset in K (a whole number of groups of three planes).
bool gemm_dma_planes3_split_ok(const MMArgs& p, int nsplit) {
  if (nsplit < 1 || p.K % (BK * nsplit)) return false;
  const int kts = p.K / BK / nsplit;
  return kts % 3 == 0 && kts >= 4;
}

// What three planes against a matrix take on `tile` in `nsplit` parts of K, the result's way out with it (gated: 256 x 192 writes gated planes) but not a fold of slabs; < 0: not to be taken.
// A fixed part (without the gap between two launches) and, per round of tiles, their K tiles (planes counted) at a time that grows with the share of the chip that is busy: with every workgroup that a CU holds (`per_cu`) a
// new step and a slope.  Fitted to 107 products of 384 .. 4096 rows (3400 timed calls, each tile and 1, 2, 4, 8 parts): the choices by it are 1.1 % from the fastest in the mean; by the prices of one plane, with
// 256 x 192 compared at a second price, they were 3.3 %.  us then -> now: 600 x 2 of 2816 x 1024 40.6 -> 33.0, 900 x 4096 x 4096 101 -> 85, 1650 x 1024 x 2816 45.2 -> 40.0, 450 x 2560 x 2048 32.6 -> 29.1, 509 x 2048 x 5632
// 47.9 -> 45.3; llama's products of 1024 rows and more keep their tiles or gain up to a tenth.
// The ring past one round: where a CU holds several workgroups their ends spread, and a little more than a round takes a quarter longer, not twice as long (1900 x 2560 x 2048, 600 tiles of 64 x 128: 65 us, 70 in two parts on 256 x 192).
// That holds up to a round and a half: of 379 products of k 128 .. 960 that are priced so, the 301 within it take 0.95 to 1.8 times as long on the tiles priced next (1.12 in the mean; 640 x 7600 x 640 27.3 us, 29.1 on 128 x 128; 964 x
// 4928 x 256 16.8 and 18.1; 1650 x 2472 x 512 23.1 and 34.6 on the register-staged kernel), those of more rounds 0.88 to 1.15 times (3107 x 5608 x 896 101.8 us, 89.8 on 128 x 128), and a long K loses there as well
// (1849 x 4616 x 5312 275 us, 244 on 256 x 192).  `ends`: below 24 K tiles the large tiles' way in and out is not hidden by the K loop (k 128, us above the price without it: 256 x 256 9, 256 x 192 7, 256 x 128 6, 128 x 128 5.5, the ring's 4).
double gemm_dma_planes3_cost_us(const MMArgs& p, int tile, int nsplit, bool gated) {
  static const struct Price {
    int tile, per_cu, ends;
    double fixed, step[3], slope[3];
  } prices[] = {
      {256, 1, 10, 3.3, {1.036}, {0.225}},
      {192, 1, 6, 3.2, {1.075}, {0}},
      {128, 1, 4, 3.4, {0.716}, {0.044}},
      {64, 2, 3, 2.95, {0.440, 0.144}, {0.142, 0.110}},
      {65, 1, 0, 4.1, {0.231}, {0.186}},
      {48, 2, 0, 4.25, {0.205, 0.152}, {0.015, 0.111}},
      {32, 3, 0, 3.95, {0.091, 0.065, 0.109}, {0.099, 0.027, 0.050}},
  };
  const size_t tiles = tile_count(p, (size_t)nsplit, tile);
  for (const Price& c : prices) {
    if (c.tile != tile) continue;
    const size_t round = 256 * (size_t)c.per_cu;
    const double kt = (double)(p.K / BK / nsplit);
    double us = c.fixed + (double)p.M * p.N * 4 / 6.4e6 * (gated ? 0.25 : nsplit), rounds = (double)(tiles / round);
    us += 0.021 * c.ends * std::max(0.0, 24 - kt);
    size_t last = tiles % round;
    if (ring_tile(tile) && tiles > round) {
      if (c.per_cu == 1 || nsplit > 1 || 2 * tiles > 3 * round) return -1.0;
      rounds = std::max(1.25, (double)tiles / round), last = 0;
    }
    for (int j = 0; j < c.per_cu; ++j) {
      const double left = std::min(256.0, std::max(0.0, (double)last - 256.0 * j));
      us += kt * (rounds * (c.step[j] + c.slope[j]) + (left > 0 ? c.step[j] + c.slope[j] * left / 256 : 0.0));
    }
    return us;
  }
  return -1.0;
}

void gemm_dma_planes3_name(int tile, int nsplit, const char* tail, char* out, size_t out_len) {
  int bm = 0, bn = 0;
  tile_dims(tile, &bm, &bn);
  char split[24] = "";
  if (nsplit > 1) snprintf(split, sizeof split, ",splitK=%d", nsplit);
  snprintf(out, out_len, "gemm_dma4<bf16,NT,%dx%d,%s,3 planes%s,f32 out%s>", bm, bn, waves_name(tile), split, tail ? tail : "");
}

// (the up rows of a tile lie n_out rows behind its gate rows, and both are reached from the matrix's first row with 32-bit offsets)
bool gemm_dma_planes3_gates(const MMArgs& p, int tile, int nsplit) {
  return tile == 192 && nsplit == 1 && p.N % 16 == 0 && (unsigned long long)p.b_cs * 2 * p.N < (1ull << 32);
}

hipError_t gemm_dma_launch_planes3(hipStream_t stream, const MMArgs& p, int tile, int nsplit, const float* residual, const char* note_tail, bool gated, uint16_t* gated_planes) {
  if (p.b_k_div != 3 || !(p.b_rs == 1 && p.b_cs != 1) || !gemm_dma_planes3_split_ok(p, nsplit) || (nsplit > 1 && residual) || (gated && !gemm_dma_planes3_gates(p, tile, nsplit)))
    return hipErrorInvalidValue;
  MMArgs q = p;
  if (nsplit > 1) {
    q.K = p.K / nsplit;
    q.a_bs = q.K, q.b_bs = q.K / 3, q.c_bs = (long long)p.M * p.N;
  }
  if (!gemm_dma_supported(UGHIP_BF16, q, (size_t)nsplit, tile)) return hipErrorInvalidValue;
  if (residual && !aligned16(residual)) return hipErrorInvalidValue;
  char name[160];
  gemm_dma_planes3_name(tile, nsplit, note_tail, name, sizeof name);
  note_kernel("%s", name);
  if (ring_tile(tile)) return gemm_ring_launch(stream, UGHIP_BF16, DmaForm::PLANES3, q, (size_t)nsplit, tile, residual, DmaRows());
  if (tile == 256) return launch<__bf16, 256, 256, false, true, 3>(stream, q, (size_t)nsplit, residual);
  if (tile == 192 && gated) {
    DmaRows rw;
    rw.dst = gated_planes ? static_cast<void*>(gated_planes) : p.c, rw.n_out = p.N / 2, rw.dst_bf16 = gated_planes != nullptr;
    if (gated_planes && (rw.n_out % 64 || !aligned16(gated_planes))) return hipErrorInvalidValue;
    return launch<__bf16, 256, 192, false, true, 3, 4>(stream, q, 1, nullptr, rw);
  }
  if (tile == 192) return launch<__bf16, 256, 192, false, true, 3>(stream, q, (size_t)nsplit, residual);
  if (tile == 128) return launch<__bf16, 256, 128, false, true, 3>(stream, q, (size_t)nsplit, residual);
  return launch<__bf16, 128, 128, false, true, 3>(stream, q, (size_t)nsplit, residual);
}


bool gemm_dma_rows_supported(const MMArgs& p, const DmaRows& r, RowsAct act, int tile) {
  int bm, bn;
  if (!tile_dims(tile, &bm, &bn) || (tile != 256 && tile != 192 && !ring_tile(tile)) || ((tile == 256 || tile == 192 || tile == 97) && act == RowsAct::LOOKUP) || (by_height(tile) && (!r.groups || act == RowsAct::LOOKUP)))
    return false;
  if (tile == 16 && act == RowsAct::GLU) return false;
  if (p.M <= 0 || p.N <= 0 || p.N % 8 || p.K % BK || p.K < least_k(tile) || p.a_cs != 1 || p.a_rs % 8 || p.b_rs != 1 || p.b_cs % 8) return false;
  if (r.n_out <= 0 || r.n_out % 4 || p.N != (act == RowsAct::GLU ? 2 * r.n_out : r.n_out) || r.dst_stride % 4 || r.w_group % 8) return false;
  // per-lane offsets are 32-bit: rows of x anywhere, matrix rows of a tile (of the whole matrix with SwiGLU)
  const unsigned long long x_rows = r.row_index ? r.x_rows : p.M;
  if (x_rows * p.a_rs * 2 >= (1ull << 31) || (unsigned long long)p.b_cs * 2 * (act == RowsAct::GLU ? p.N : bn) >= (1ull << 31)) return false;
  if (!aligned16(p.a) || !aligned16(p.b) || !aligned16(r.dst) || (r.bias && !aligned16(r.bias))) return false;
  return ((size_t)(p.M + bm - 1) / bm + r.groups) * (size_t)((p.N + bn - 1) / bn) < (1u << 24);
}

// What rows by group take, spread as SHARES says (taken as even, groups of 127 rows went to 192 x 192 tiles, of which one in eight is then two: 85 us where 59 are possible): a fixed part and, for every round of
// 256 tiles, their K tiles, at a time that grows with the share of the chip that is busy; of a last round that is not full `tail` of the rest counts.  Tiles by height (193, 130): a K tile by the height in
// 64s; one round lasts for its highest tiles mostly, several go by the mean and leave `last` of one of the highest behind.  Whether tiles near 256 are one round or two is seen by the router's rows alone: in between.
// Fitted to 2000 products on each of the eight tiles (2 to 128 groups of 4 to 2048 rows, 18 matrices from 512 x 512 to 8192 x 4096, shares of the rows that differ by 20, 40 and 60 %, up to six draws of them): the choice is
// 1.2 % from the fastest in the mean, 0.4 % for 16 groups of the decoders' matrices.  Prices fitted to those 16 groups alone, with every column of a matrix from memory once per tile, were 4.6 % and 2.8 % from it, and a tenth or
// more slower than the best of the tiles of one height for 92 of the products, 14 so: 8 groups of 2048 rows, n 8192, k 4096 1295 us on 256 x 192 by height, 886 on 256 x 256; 32 of 800 rows 2200 and 1574; 8 of 200, n 2 x 4096, k 1024 54.7 and 37.8.
struct GroupedRows {
  double tiles[4] = {}, heights[4] = {};  // tile rows of 64, 128, 192 and 256 rows; those of up to 256 by their height in 64s
  GroupedRows(int m, int groups) {
    for (double share : SHARES) {
      const int rows = share_rows(m, groups, share), n = (rows + 255) / 256;
      tiles[0] += (rows + 63) / 64, tiles[1] += (rows + 127) / 128, tiles[2] += (rows + 191) / 192, tiles[3] += n;
      heights[std::min(4, (((rows + n - 1) / n + 15) / 16 * 16 + 63) / 64) - 1] += n;
    }
    for (double* counts : {tiles, heights})
      for (int i = 0; i < 4; ++i) counts[i] *= groups / 16.0;
  }
};
static double grouped_cost_us(const MMArgs& p, const GroupedRows& rows, int tile) {
  static const struct {
    int tile;
    double fixed, first, busy, tail;
  } prices[] = {{256, 6.25, 1.214, 0.612, 0.78}, {129, 3.93, 1.055, 0.151, 0.4}, {97, 3.0, 1.013, 0.228, 0.645}, {65, 2.02, 0.429, 0.508, 0.78}, {48, 2.48, 0.339, 0.304, 1.0}, {32, 3.04, 0.047, 0.332, 0.285}};
  static const struct {
    double fixed, height[4], last;
  } by_heights[] = {{2.63, {0.656, 0.839, 1.157, 1.612}, 0.70}, {2.99, {0.456, 0.636, 0.917, 1.087}, 0.61}};
  constexpr double NEAR = 0.055;
  int bm, bn;
  tile_dims(tile, &bm, &bn);
  const double columns = (p.N + bn - 1) / bn, kt = p.K / BK, tiles = rows.tiles[bm / 64 - 1] * columns, rounds = tiles / 256;
  const double two = std::min(1.0, std::max(0.0, (rounds - (1 - NEAR)) / (2 * NEAR)));  // of one round and more
  if (by_height(tile)) {
    const auto& high = by_heights[tile == 193 ? 0 : 1];
    double sum = 0, highest = 0;
    for (int h = 0; h < 4; ++h)
      if (rows.heights[h] > 0) sum += rows.heights[h] * columns * high.height[h], highest = high.height[h];
    const double one = 0.89 * highest + 0.11 * sum / tiles, more = std::max(sum / 256 + high.last * highest, rounds < 1 + NEAR ? one : 0.0);
    return high.fixed + kt * (one + (more - one) * two);
  }
  for (const auto& c : prices)
    if (c.tile == tile) {
      const double past = std::max(rounds, 1.001), more = past + c.tail * (std::ceil(past - 1e-9) - past);
      return c.fixed + kt * (c.first + c.busy * std::min(1.0, rounds)) * (1 + (more - 1) * two);
    }
  return 1e30;
}

int gemm_dma_rows_pick(const MMArgs& p, const DmaRows& r, RowsAct act) {
  if (long long s; tune_get(TUNE_GEMM_SHAPE, &s)) {  // tuning aid, as for gemm_dma_pick
    const int tile = gemm_dma_forced_tile(s), forced = tile == 128 ? 129 : tile == 64 ? 65 : tile;  // (256 x 128 and 128 x 128 tiles of rows are the ring's)
    return forced && gemm_dma_rows_supported(p, r, act, forced) ? forced : 0;
  }
  // A model's products: the matrix comes from memory.  256 x 256 and 256 x 192 tiles of gemm_dma4 and the ring's, by what they are expected to take
  // (2048 positions: down 74 -> 51 us, gate and up 105 -> 89, output 26 -> 18, attention's input 37 -> 29; 509 positions: state-space output
  // 53 -> 19, input 43 -> 32, dense gate and up 40 -> 30; 700 positions' gate and up 52 -> 34; 33 rows of 11264 x 2048 31 -> 13).  256 x 192 where they are nearly whole rounds: 256 x 256 / 256 x 192 / the best of
  // the ring, us: 2048 x 2 of 5632 x 2048 98 / 86 / 91, 2048 x 2 of 2816 x 1024 29.5 / 26.9 / 34.4, 1544 x 2 of 3072 x 4160 90 / 78 / 100, 3305 x 6336 x 3328 134 / 125 / 132, 877 x 9984 x 2304 51 / 44 / 59; 2048 x 6592 x
  // 2048, 208 tiles and 280, 48 / 71 / 59.  46 products of 300 to 4096 rows: what is taken by these prices is the fastest but for 4 % at most (3706 x 2 of 1152 x 512, 1.5 us, as before).
  int best = 0;
  double best_us = 0;
  if (r.groups > 1) {
    const GroupedRows rows(p.M, r.groups);
    for (int tile : {256, 129, 65, 48, 32, 97, 193, 130}) {
      if (!gemm_dma_rows_supported(p, r, act, tile)) continue;
      const double us = grouped_cost_us(p, rows, tile);
      if (!best || us < best_us) best = tile, best_us = us;
    }
    return best;
  }
  for (int tile : {256, 192, 129, 65, 48, 32, 16, 97}) {
    if (!gemm_dma_rows_supported(p, r, act, tile)) continue;
    if (tile == 16 && p.K < 8 * BK) continue;  // shorter than its ring it gains nothing (54 rows of 2048 x 256 4.0 us on either)
    int bm, bn;
    tile_dims(tile, &bm, &bn);
    const size_t tiles = (size_t)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn);
    const int kt = p.K / BK;
    double us = 6.0;
    if (!ring_tile(tile))
      for (size_t left = tiles; left > 0; left -= left < 256 ? left : 256) us += kt * ((tile == 256 ? 1.23 : 0.8) + (tile == 256 ? 0.33 : 0.47) * (left < 256 ? (double)left : 256.0) / 256.0);
    else us = ring_cost_us(tiles, kt, tile, Operands::MEMORY);
    // the larger tile on a near tie; 192 x 192 last, where it clearly saves a round
    if (!best || us < best_us * (tile == 97 ? 0.9 : 0.97)) best = tile, best_us = us;
  }
  return best;
}

hipError_t gemm_dma_launch_rows(hipStream_t stream, const MMArgs& p, const DmaRows& r, RowsAct act, int tile) {
  if (!gemm_dma_rows_supported(p, r, act, tile)) return hipErrorInvalidValue;
  int bm = 0, bn = 0;
  tile_dims(tile, &bm, &bn);
  note_kernel("gemm_dma4<bf16,NT,%dx%d,%s,rows%s%s>", bm, bn, waves_name(tile), act == RowsAct::GLU ? ",swiglu" : act == RowsAct::LOOKUP ? ",lookup" : "", r.groups ? ",grouped" : "");
  if (ring_tile(tile)) return gemm_ring_launch(stream, UGHIP_BF16, act == RowsAct::GLU ? DmaForm::ROWS_GLU : act == RowsAct::LOOKUP ? DmaForm::ROWS_LOOKUP : DmaForm::ROWS, p, 1, tile, nullptr, r);
  if (tile == 192) return act == RowsAct::GLU ? launch<__bf16, 256, 192, false, false, 1, 2>(stream, p, 1, nullptr, r) : launch<__bf16, 256, 192, false, false, 1, 1>(stream, p, 1, nullptr, r);
  return act == RowsAct::GLU ? launch<__bf16, 256, 256, false, false, 1, 2>(stream, p, 1, nullptr, r) : launch<__bf16, 256, 256, false, false, 1, 1>(stream, p, 1, nullptr, r);
}

// Both operands as three bf16 planes per 64 elements of k (p.K = 6 k, rows of 3 k elements), f32 result: see BDIV == 6.
bool gemm_dma_planes6_supported(const MMArgs& p, size_t batch, int tile) { return p.K % (6 * BK) == 0 && gemm_dma_supported(UGHIP_BF16, p, batch, tile); }

void gemm_dma_planes6_name(const MMArgs& p, int tile, char* out, size_t out_len) {
  int bm = 0, bn = 0;
  tile_dims(tile, &bm, &bn);
  const bool nn = p.b_cs == 1 && p.b_rs != 1;
  snprintf(out, out_len, "gemm_dma4<bf16,%s,%dx%d,256t,6 terms of 3 x 3 planes,f32 out>", nn ? "NN" : "NT", bm, bn);
}

hipError_t gemm_dma_launch_planes6(hipStream_t stream, const MMArgs& p, size_t batch, int tile) {
  if (!gemm_dma_planes6_supported(p, batch, tile)) return hipErrorInvalidValue;
  char name[112];
  gemm_dma_planes6_name(p, tile, name, sizeof name);
  note_kernel("%s", name);
  const bool nn = p.b_cs == 1 && p.b_rs != 1;
  if (tile == 256) return nn ? launch<__bf16, 256, 256, true, true, 6>(stream, p, batch) : launch<__bf16, 256, 256, false, true, 6>(stream, p, batch);
  if (tile == 128) return nn ? launch<__bf16, 256, 128, true, true, 6>(stream, p, batch) : launch<__bf16, 256, 128, false, true, 6>(stream, p, batch);
  return nn ? launch<__bf16, 128, 128, true, true, 6>(stream, p, batch) : launch<__bf16, 128, 128, false, true, 6>(stream, p, batch);
}

}  // namespace ughip
