// Products of one row with their neighbours folded in (ughip_product_row): a decode step of the layers in ughip_layers.h.
//
// row_wide_kernel: the whole workgroup on every matrix row, the input row -- residual add with the norm of the sublayer in front, gate,
// norm -- made in registers in every workgroup while the matrix is on its way.  It costs a workgroup a few cache reads and spares the
// launches that would make it; the first one stores the new residual.  PLAIN: the row is x as it is (or, routed, times the experts' weights).
// row_step_kernel: rows of any length and alignment.  A workgroup of four waves takes 4 R columns, R per wave: runs of 512 elements of the
// matrix rows (eight elements per lane and run), four to a batch, batch b + NB asked for where batch b was; the input row in LDS.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "layers.h"
#include "route.h"

using namespace ughip;

namespace {

struct RowArgs {
  const float* x;
  const float* y;
  const float* y_norm;
  const float* gate;
  const float* norm;
  float* x_out;  // null: not kept
  float* dst;
  const void* w;
  const float* bias;
  const void* table;
  const int* ids;
  size_t table_stride, table_col, w_group;
  const float* extra;  // joins x too
  GluForm glu;
  float eps, inv_k;
  int n, k, cols, norm_groups, table_rows, segs;
  bool table_bf16, gate_after;
  const float* logits;
  RouteArgs route;
  int* route_ids;
  float* route_weights;
};

constexpr int RUN = 512, PRE = 4;

template <typename WT>
struct Eight;
template <>
struct Eight<uint16_t> {
  u32x4_t v;
  __device__ void clear() { v = u32x4_t{0, 0, 0, 0}; }
  __device__ void load(const uint16_t* p) { v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p)); }
  __device__ void load_some(const uint16_t* p, int left) {
    uint32_t e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = i < left ? p[i] : 0;
    v = u32x4_t{e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16};
  }
  __device__ float dot(const f32x4_t& a, const f32x4_t& b, float s) const {
    s += __uint_as_float(v.x << 16) * a.x;
    s += __uint_as_float(v.x & 0xffff0000u) * a.y;
    s += __uint_as_float(v.y << 16) * a.z;
    s += __uint_as_float(v.y & 0xffff0000u) * a.w;
    s += __uint_as_float(v.z << 16) * b.x;
    s += __uint_as_float(v.z & 0xffff0000u) * b.y;
    s += __uint_as_float(v.w << 16) * b.z;
    s += __uint_as_float(v.w & 0xffff0000u) * b.w;
    return s;
  }
};
template <>
struct Eight<float> {
  f32x4_t u, v;
  __device__ void clear() { u = v = f32x4_t{0.f, 0.f, 0.f, 0.f}; }
  __device__ void load(const float* p) {
    u = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(p));
    v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(p) + 1);
  }
  __device__ void load_some(const float* p, int left) {
    float e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = i < left ? p[i] : 0.f;
    u = f32x4_t{e[0], e[1], e[2], e[3]}, v = f32x4_t{e[4], e[5], e[6], e[7]};
  }
  __device__ float dot(const f32x4_t& a, const f32x4_t& b, float s) const {
    s += u.x * a.x;
    s += u.y * a.y;
    s += u.z * a.z;
    s += u.w * a.w;
    s += v.x * b.x;
    s += v.y * b.y;
    s += v.z * b.z;
    s += v.w * b.w;
    return s;
  }
};

// What becomes of column `col`'s sum (with NM 2: the gate's and the up row's).
template <int NM>
__device__ __forceinline__ float finished(const RowArgs& a, int col, const float (&sums)[NM]) {
  float v = sums[0];
  if (a.bias) v += a.bias[col];
  if constexpr (NM == 2) {
    float u = sums[1];
    if (a.bias) u += a.bias[a.n + col];
    return glu_f(v, u, a.glu);
  }
  if (a.table) {
    const int id = a.ids[0];
    float t = __uint_as_float(0x7fc00000u);
    if (id >= 0 && id < a.table_rows) {
      const size_t at = (size_t)id * a.table_stride + a.table_col + col;
      t = a.table_bf16 ? bf16_to_f32(static_cast<const uint16_t*>(a.table)[at]) : static_cast<const float*>(a.table)[at];
    }
    v = gelu_tanh_f(v) * t;
  }
  return v;
}

// R columns of NM matrices per wave; VEC: rows are 16-byte aligned and a multiple of 8 long.  ROUTE as in ughip_row_step: with 2 a
// column's row is the chosen experts' rows one after the other, each from a batch of its own on.
template <typename WT, int R, int NM, int ROUTE, bool VEC, int NB>
__global__ void __launch_bounds__(256) row_step_kernel(RowArgs a) {
  extern __shared__ __attribute__((aligned(16))) float in[];  // the row (segments `padded` apart), then ROUTE 1: logits and work space
  __shared__ float red[4][4];
  __shared__ int s_ids[64];
  __shared__ float s_wts[64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int padded = (a.k + RUN - 1) / RUN * RUN, bps = (padded / RUN + PRE - 1) / PRE, batches = (ROUTE == 2 ? a.segs : 1) * bps;
  const int col0 = (blockIdx.x * 4 + wave) * R;
  if constexpr (ROUTE == 1) {  // which experts' matrices: before anything of them can be asked for
    float* lg = in + padded;
    for (int e = threadIdx.x; e < a.route.experts; e += 256) lg[e] = a.logits[e];
    __syncthreads();
    if (wave == 0) {
      float* work = lg + a.route.experts;
      int* ids = reinterpret_cast<int*>(work + route_lds_floats(a.route.experts, a.route.groups));
      float* wts = reinterpret_cast<float*>(ids + a.route.top);
      route_choose(lg, a.route, work, ids, wts);
      if (lane < a.route.top) s_ids[lane] = ids[lane];
      if (blockIdx.x == 0 && lane < a.route.top) a.route_ids[lane] = ids[lane], a.route_weights[lane] = wts[lane];
    }
    __syncthreads();
  }
  if constexpr (ROUTE == 2) {
    if (threadIdx.x < (unsigned)a.segs) {
      const int e = a.route_ids[threadIdx.x];
      s_ids[threadIdx.x] = e >= 0 && e < a.route.experts ? e : 0;
      s_wts[threadIdx.x] = a.route_weights[threadIdx.x];
    }
    __syncthreads();
  }
  // a column's matrix row; ROUTE 1: column j n + c is column c of the j-th chosen expert
  const WT* rows[NM][R];
  bool live[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int col = col0 + r;
    live[r] = col < a.cols;
    size_t at = (size_t)(live[r] ? col : 0) * a.k;
    if (ROUTE == 1) {
      const int j = live[r] ? col / a.n : 0;
      at = (size_t)s_ids[j] * a.w_group + (size_t)((live[r] ? col : 0) - j * a.n) * a.k;
    }
    rows[0][r] = static_cast<const WT*>(a.w) + at;
    if (NM == 2) rows[NM - 1][r] = static_cast<const WT*>(a.w) + at + (size_t)a.n * a.k;  // gate rows, then up rows
  }
  Eight<WT> held[NB][NM][R][PRE];
  int fj = 0, fc = 0;  // the next batch to ask for: segment and batch inside it
  auto fetch = [&](Eight<WT>(&to)[NM][R][PRE]) {
    if (ROUTE == 2 ? fj >= a.segs : fc >= bps) return;  // the same for the whole workgroup
    const size_t seg = ROUTE == 2 ? (size_t)s_ids[fj] * a.w_group : 0;
#pragma unroll
    for (int c = 0; c < PRE; ++c) {
      const int kk = (fc * PRE + c) * RUN + lane * 8;
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < NM; ++m) {
          Eight<WT>& e = to[m][r][c];
          // every lane loads (past the row's end: its first elements, which meet zeros): with branches around loads the compiler
          // waits for all of them at once
          if constexpr (VEC) e.load(rows[m][r] + seg + (kk < a.k ? kk : 0));
          else e.load_some(rows[m][r] + seg + kk, live[r] ? a.k - kk : 0);
        }
    }
    if (ROUTE == 2 && fc + 1 == bps) ++fj, fc = 0;
    else ++fc;
  };
#pragma unroll
  for (int b = 0; b < NB; ++b) fetch(held[b]);
  __builtin_amdgcn_sched_barrier(0);

  // the input row
  float ss = 0.f;
  if constexpr (ROUTE == 2) {
    for (int j = 0; j < a.segs; ++j) {
      const float w = s_wts[j];
      for (int i = threadIdx.x; i < padded; i += 256) in[j * padded + i] = i < a.k ? a.x[j * a.k + i] * w : 0.f;
    }
  } else {
    for (int i = threadIdx.x; i < padded; i += 256) {
      float v = 0.f;
      if (i < a.k) {
        v = a.y ? a.y[i] : a.x[i];
        if (a.gate && !a.gate_after) v *= silu_f(a.gate[i]);
      }
      in[i] = v;  // read back by the same thread until the last barrier
      ss += v * v;
    }
    if (a.y) {
      ss = block_sum<4>(ss, red[0]);
      const float inv = 1.f / sqrtf(ss / (float)a.k + a.eps);
      ss = 0.f;
      for (int i = threadIdx.x; i < a.k; i += 256) {
        const float v = a.x[i] + in[i] * inv * a.y_norm[i] + (a.extra ? a.extra[i] : 0.f);
        in[i] = v;
        ss += v * v;
        if (a.x_out && blockIdx.x == 0) a.x_out[i] = v;
      }
    }
    if (a.norm && a.norm_groups == 1) {
      ss = block_sum<4>(ss, red[1]);
      const float inv = 1.f / sqrtf(ss / (float)a.k + a.eps);
      for (int i = threadIdx.x; i < a.k; i += 256) in[i] *= inv * a.norm[i];
    } else if (a.norm) {
      const int part = a.k / a.norm_groups;
      __syncthreads();  // a part is summed by one wave
      for (int g = wave; g < a.norm_groups; g += 4) {
        float s = 0.f;
        for (int i = lane; i < part; i += 64) s += in[g * part + i] * in[g * part + i];
        s = wave_sum(s);
        const float inv = 1.f / sqrtf(s / (float)part + a.eps);
        for (int i = lane; i < part; i += 64) in[g * part + i] *= inv * a.norm[g * part + i];
      }
    }
    if (a.gate && a.gate_after) {
      __syncthreads();
      for (int i = threadIdx.x; i < a.k; i += 256) in[i] *= sigmoid_f(a.gate[i]);
    }
  }
  __syncthreads();

  float acc[NM][R];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int r = 0; r < R; ++r) acc[m][r] = 0.f;
  int dj = 0, dc = 0;  // the batch to multiply
  auto multiply = [&](const Eight<WT>(&from)[NM][R][PRE]) {
    const float* row = in + dj * padded + dc * PRE * RUN + lane * 8;
    const int left = padded / RUN - dc * PRE;
#pragma unroll
    for (int c = 0; c < PRE; ++c) {
      if (c < left) {
        const f32x4_t xa = *reinterpret_cast<const f32x4_t*>(row + c * RUN), xb = *reinterpret_cast<const f32x4_t*>(row + c * RUN + 4);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int m = 0; m < NM; ++m) acc[m][r] = from[m][r][c].dot(xa, xb, acc[m][r]);
      }
    }
    if (ROUTE == 2 && dc + 1 == bps) ++dj, dc = 0;
    else ++dc;
  };
  for (int b0 = 0; b0 < batches; b0 += NB) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (b0 + b < batches) {
        multiply(held[b]);
        if (b0 + b + NB < batches) fetch(held[b]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
#pragma unroll
    for (int m = 0; m < NM; ++m) acc[m][r] = wave_sum(acc[m][r]);
    if (lane != 0 || !live[r]) continue;
    const int col = col0 + r;
    float u[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) u[m] = acc[m][r];
    a.dst[col] = finished<NM>(a, col, u);
  }
}

// The sum over the NW waves of a workgroup, NW up to 16 and known when it runs; `red` holds 16 floats of which those past NW are zero.
__device__ __forceinline__ float any_block_sum(float v, float* red) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return row_sum16(red[threadIdx.x & 15]);
}

// The same product with the whole workgroup on every matrix row: thread t holds elements 8 t .. 8 t + 7 of the input row in registers (of
// ROUTE 2: of the chosen experts' rows one after the other), as many waves as that takes, and the workgroup walks B batches of R columns, two
// batches on their way.
template <typename WT, int NM, int R, int B, int ROUTE, bool PLAIN>
__global__ void __launch_bounds__(1024) row_wide_kernel(RowArgs a) {
  extern __shared__ __attribute__((aligned(16))) float route_work[];  // ROUTE 1: logits and work space
  __shared__ float red[3][16];
  __shared__ float part[NM * B * R][17];
  __shared__ int s_ids[64];
  __shared__ float s_wts[64];
  constexpr int NB = B < 2 ? B : 2;
  const int total = (ROUTE == 2 ? a.segs : 1) * a.k, waves = (total + 511) >> 9;  // (blockDim is a trip to memory)
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), e0 = t * 8;
  const bool ok = e0 < total;
  const int at0 = ok ? e0 : 0;  // (a lane past the end reads the row's first elements and multiplies them with zeros)
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t v[2], y[2], yn[2], nm[2], ex[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    v[i] = *reinterpret_cast<const f32x4_t*>(a.x + at0 + 4 * i);
    if constexpr (!PLAIN) {
      if (a.y || a.gate) y[i] = *reinterpret_cast<const f32x4_t*>((a.y ? a.y : a.gate) + at0 + 4 * i);
      if (a.y) yn[i] = *reinterpret_cast<const f32x4_t*>(a.y_norm + at0 + 4 * i);
      if (a.norm) nm[i] = *reinterpret_cast<const f32x4_t*>(a.norm + at0 + 4 * i);
      if (a.extra) ex[i] = *reinterpret_cast<const f32x4_t*>(a.extra + at0 + 4 * i);
    }
  }
  if constexpr (!PLAIN)
    if (t < 48) red[t >> 4][t & 15] = 0.f;
  if constexpr (ROUTE == 1) {  // which experts' matrices: before anything of them can be asked for
    float* lg = route_work;
    for (int e = t; e < a.route.experts; e += 64 * waves) lg[e] = a.logits[e];
    __syncthreads();
    if (wave == 0) {
      float* work = lg + a.route.experts;
      int* ids = reinterpret_cast<int*>(work + route_lds_floats(a.route.experts, a.route.groups));
      float* wts = reinterpret_cast<float*>(ids + a.route.top);
      route_choose(lg, a.route, work, ids, wts);
      if (lane < a.route.top) s_ids[lane] = ids[lane];
      if (blockIdx.x == 0 && lane < a.route.top) a.route_ids[lane] = ids[lane], a.route_weights[lane] = wts[lane];
    }
    __syncthreads();
  }
  int seg = 0;
  if constexpr (ROUTE == 2) {
    if (t < a.segs) {
      const int e = a.route_ids[t];
      s_ids[t] = e >= 0 && e < a.route.experts ? e : 0;
      s_wts[t] = a.route_weights[t];
    }
    __syncthreads();
    seg = (int)(((float)at0 + 0.5f) * a.inv_k);  // never within a rounding of a whole number
  }
  const int col0 = blockIdx.x * (B * R);
  const WT* mine = static_cast<const WT*>(a.w) + (ROUTE == 2 ? (size_t)s_ids[seg] * a.w_group + (size_t)(at0 - seg * a.k) : (size_t)at0);
  Eight<WT> held[NB][NM][R];
  auto fetch = [&](int b, Eight<WT>(&to)[NM][R]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int col = min(col0 + b * R + r, a.cols - 1);
      size_t at = (size_t)col * a.k;
      if (ROUTE == 1) {
        const int j = col / a.n;
        at = (size_t)__builtin_amdgcn_readfirstlane(s_ids[j]) * a.w_group + (size_t)(col - j * a.n) * a.k;
      }
#pragma unroll
      for (int m = 0; m < NM; ++m) to[m][r].load(mine + at + (m ? (size_t)a.n * a.k : 0));
    }
  };
#pragma unroll
  for (int b = 0; b < NB; ++b) fetch(b, held[b]);
  __builtin_amdgcn_sched_barrier(0);

  // the input row
  if (!ok) v[0] = v[1] = zero;
  if constexpr (ROUTE == 2) {
    const float w = s_wts[seg];
    v[0] *= w, v[1] *= w;
  }
  if constexpr (!PLAIN) {
    auto square = [](const f32x4_t& p, const f32x4_t& q) { return p.x * p.x + p.y * p.y + p.z * p.z + p.w * p.w + (q.x * q.x + q.y * q.y + q.z * q.z + q.w * q.w); };
    __syncthreads();  // (`red` is clear)
    if (a.y) {
      const float ss = any_block_sum(ok ? square(y[0], y[1]) : 0.f, red[0]), inv = 1.f / sqrtf(ss / (float)a.k + a.eps);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        v[i] = v[i] + y[i] * inv * yn[i];
        if (a.extra) v[i] += ex[i];
        if (a.x_out && blockIdx.x == 0 && ok) *reinterpret_cast<f32x4_t*>(a.x_out + e0 + 4 * i) = v[i];
      }
    } else if (a.gate && !a.gate_after) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] *= silu_f(y[i][e]);
    }
    if (!ok) v[0] = v[1] = zero;
    const int part = a.norm ? a.k / a.norm_groups : 0;
    if (part == 4) {
#pragma unroll
      for (int i = 0; i < 2; ++i) v[i] = v[i] * (1.f / sqrtf((v[i].x * v[i].x + v[i].y * v[i].y + v[i].z * v[i].z + v[i].w * v[i].w) / 4.f + a.eps)) * nm[i];
      if (!ok) v[0] = v[1] = zero;
    } else if (part) {
      float ss = square(v[0], v[1]);
      if (a.norm_groups == 1) {
        ss = any_block_sum(ss, red[1]);
      } else if (part < 256) {  // 1, 2, 4, 8 or 16 lanes (the host checks)
        for (int d = part >> 4; d; d >>= 1) ss += __shfl_xor(ss, d, 64);
      } else {  // whole waves, or whole halves of them (the host checks)
        const int shift = part & 256 ? 5 : 6, mine = t >> shift, run = part >> (shift + 3), first = mine / run * run;
        if (shift == 6) ss = wave_sum(ss);
        else ss = row_sum16(ss), ss += __shfl_xor(ss, 16, 64);
        float* sums = &red[1][0];  // 32 of them
        if ((t & ((1 << shift) - 1)) == 0) sums[mine] = ss;
        __syncthreads();
        ss = 0.f;
        for (int i = 0; i < run; ++i) ss += sums[first + i];
      }
      const float inv = 1.f / sqrtf(ss / (float)part + a.eps);
#pragma unroll
      for (int i = 0; i < 2; ++i) v[i] = v[i] * inv * nm[i];
      if (!ok) v[0] = v[1] = zero;
    }
    if (a.gate && a.gate_after) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] *= sigmoid_f(y[i][e]);
      if (!ok) v[0] = v[1] = zero;
    }
  }
#pragma unroll
  for (int b = 0; b < B; ++b) {
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float s = wave_sum(held[b % NB][m][r].dot(v[0], v[1], 0.f));
        if (lane == 0) part[(m * B + b) * R + r][wave] = s;
      }
    if (b + NB < B) fetch(b + NB, held[b % NB]);
  }
  __syncthreads();
  const int col = col0 + t;
  if (t >= B * R || col >= a.cols) return;
  float u[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    u[m] = 0.f;
    for (int w = 0; w < waves; ++w) u[m] += part[m * B * R + t][w];
  }
  a.dst[col] = finished<NM>(a, col, u);
}

template <typename WT, int R, int NM, int ROUTE, bool VEC>
hipError_t launch_one(hipStream_t st, const RowArgs& a, size_t lds) {
  const unsigned grid = (unsigned)((a.cols + 4 * R - 1) / (4 * R));
  auto kernel = row_step_kernel<WT, R, NM, ROUTE, VEC, VEC ? 2 : 1>;
  if (lds > 60 * 1024)
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); e != hipSuccess) return e;
  kernel<<<grid, 256, lds, st>>>(a);
  return hipGetLastError();
}

template <typename WT, int R, int NM, int ROUTE>
hipError_t launch_vec(hipStream_t st, const RowArgs& a, size_t lds, bool vec) {
  return vec ? launch_one<WT, R, NM, ROUTE, true>(st, a, lds) : launch_one<WT, R, NM, ROUTE, false>(st, a, lds);
}

template <typename WT, int NM, int ROUTE>
hipError_t launch_rows(hipStream_t st, const RowArgs& a, size_t lds, bool vec) {
  // enough workgroups for the chip first, then more columns for each of them to share the input row
  const int r = a.cols >= 8192 && NM == 1 ? 4 : a.cols >= 2048 ? 2 : 1;
  if constexpr (NM == 1)
    if (r == 4) return launch_vec<WT, 4, NM, ROUTE>(st, a, lds, vec);
  return r >= 2 ? launch_vec<WT, 2, NM, ROUTE>(st, a, lds, vec) : launch_vec<WT, 1, NM, ROUTE>(st, a, lds, vec);
}

template <typename WT>
hipError_t launch_any(hipStream_t st, const RowArgs& a, int route, bool up, size_t lds, bool vec) {
  if (route == 1) return up ? launch_rows<WT, 2, 1>(st, a, lds, vec) : hipErrorInvalidValue;
  if (route == 2) return launch_rows<WT, 1, 2>(st, a, lds, vec);
  return up ? launch_rows<WT, 2, 0>(st, a, lds, vec) : launch_rows<WT, 1, 0>(st, a, lds, vec);
}

constexpr int WIDE_MAX = 8192;  // elements of the input row: eight to a thread

// Columns per workgroup: the more, the fewer times the input row is read and made, but every CU wants a workgroup and some six waves to keep
// enough of the matrix on its way (and past 16 matrix rows the last ones wait).  Weights from memory, us by columns per workgroup 1 / 2 / 4 / 8 / 16, bf16, then f32:
//   1024 of 1024 4.5 / 4.1 / 4.2 / 5.0 / 5.9, 4.7 / 4.0 / 4.3 / 5.0 / 5.8; 3336 of 1024 6.7 / 5.8 / 4.9 / 5.1 / 6.0, 7.8 / 7.0 / 6.1 / 5.6 / 6.2; gated 2816 of 1024 7.2 / 6.7 / 5.8 / 6.3,
//   9.2 / 7.7 / 7.9 / 8.0; 1024 of 2816 7.9 / 6.5 / 5.1 / 5.6 / 6.6, 8.5 / 7.2 / 6.1 / 7.1 / 10.0; 6416 of 2048 18.5 / 12.7 / 10.2 / 8.5 / 7.6, 24.2 / 18.1 / 14.8 / 14.1 / 13.6; gated 5632 of 2048
//   20.4 / 15.5 / 12.9 / 11.3, 29.1 / 22.9 / 21.1 / 19.5; 2048 of 5632 23.0 / 14.2 / 10.5 / 8.7 / 9.5, 26.6 / 18.8 / 15.5 / 12.2 / 17.2; 8192 of 512 7.0 / 5.9 / 5.0 / 5.2 / 5.9, 7.8 / 7.0 / 6.2 / 5.9 / 6.2;
//   32000 of 1024 31.5 / 20.8 / 15.9 / 14.4 / 13.7, 43.4 / 37.4 / 31.2 / 27.0 / 25.0 (in a reply, whose weights are partly cached, - / - / 16.6 / 14.7 / 14.0, - / - / 31.5 / 27.7 / 26.1);
//   32000 of 2048 78 / 49 / 34 / 27 / 24, 111 / 77 / 59 / 52 / 49.
int wide_columns(int cols, int threads, int matrices, int cus) {
  int most = 16 / matrices;
  while (most > 1 && ((cols + most - 1) / most < cus || (cols + most - 1) / most * (threads / 64) < cus * 11 / 2)) most /= 2;
  return most;
}

template <typename WT, int NM, int ROUTE, bool PLAIN>
hipError_t launch_wide(ughip_device* dev, const RowArgs& a, size_t lds) {
  const int total = (ROUTE == 2 ? a.segs : 1) * a.k, threads = (total / 8 + 63) / 64 * 64;
  auto go = [&](auto kernel, int columns) {
    kernel<<<(unsigned)((a.cols + columns - 1) / columns), threads, lds, dev->stream>>>(a);
    return hipGetLastError();
  };
  switch (wide_columns(a.cols, threads, NM, dev->num_cus)) {
    case 1: return go(row_wide_kernel<WT, NM, 1, 1, ROUTE, PLAIN>, 1);
    case 2: return go(row_wide_kernel<WT, NM, 2, 1, ROUTE, PLAIN>, 2);
    case 4: return go(row_wide_kernel<WT, NM, 2, 2, ROUTE, PLAIN>, 4);
    case 8: return go(row_wide_kernel<WT, NM, 2, 4, ROUTE, PLAIN>, 8);
    default:
      if constexpr (NM == 1) return go(row_wide_kernel<WT, NM, 4, 4, ROUTE, PLAIN>, 16);
      return hipErrorInvalidValue;
  }
}

constexpr size_t ROW_MAX = 16000;

}  // namespace

extern "C" int ughip_product_row(ughip_device* dev, const ughip_row_step* p) {
  const char* what = "product_row";
  if (!dev || !p || !p->w || !p->x || !p->dst) return set_error(UGHIP_ERR_INVALID, "%s: null argument", what);
  if (p->act < UGHIP_ACT_NONE || p->act > UGHIP_ACT_GLU || p->route < 0 || p->route > 2) return set_error(UGHIP_ERR_INVALID, "%s: act %d, route %d", what, p->act, p->route);
  if (p->n == 0) return UGHIP_OK;
  const size_t segs = p->route == 2 ? p->top : 1, total = segs * p->k;
  if (p->k == 0 || p->k > ROW_MAX || segs == 0 || segs > 64 || segs * ((p->k + RUN - 1) / RUN * RUN) > 32 * RUN) return set_error(UGHIP_ERR_UNSUPPORTED, "%s: %zu rows of %zu elements, up to %zu in all (in runs of %d) are supported", what, segs, p->k, (size_t)32 * RUN, RUN);
  if (p->n > 0x7fffffffull / 128) return set_error(UGHIP_ERR_INVALID, "%s: shape too large", what);
  if (p->w->dtype != UGHIP_F32 && p->w->dtype != UGHIP_BF16) return set_error(UGHIP_ERR_UNSUPPORTED, "%s: matrices are F32 or BF16", what);
  const bool glu = p->act == UGHIP_ACT_SWIGLU || p->act == UGHIP_ACT_GLU;  // gate and up rows
  const size_t mats = p->route ? p->experts : 1, w_rows = glu ? 2 * p->n : p->n;
  if (p->route) {
    if (int rc = route_check(p->experts, p->groups, p->keep, p->top, what)) return rc;
    if (p->top > 64) return set_error(UGHIP_ERR_UNSUPPORTED, "%s: up to 64 experts per row", what);
    if (p->bias || (p->route == 1 && !glu) || (p->route == 2 && p->act != UGHIP_ACT_NONE) || p->y || p->norm || p->gate)
      return set_error(UGHIP_ERR_UNSUPPORTED, "%s: routed products are SwiGLU (1) or plain (2), on x as it is", what);
    if (int rc = check_buf(dev, p->route_ids, p->top, UGHIP_I32, "product_row ids")) return rc;
    if (int rc = check_buf(dev, p->route_weights, p->top, UGHIP_F32, "product_row weights")) return rc;
  }
  auto row = [&](const ughip_slice* s, size_t off, size_t n, int dtype) { return check_view(dev, ughip_view{const_cast<ughip_slice*>(s), off, n}, 1, n, dtype, what); };
  if (int rc = row(p->x, p->x_offset, total, UGHIP_F32)) return rc;
  if (p->y) {
    if (int rc = row(p->y, p->y_offset, p->k, UGHIP_F32)) return rc;
    if (int rc = row(p->y_norm, 0, p->k, UGHIP_F32)) return rc;
  }
  if (p->extra) {
    if (!p->y) return set_error(UGHIP_ERR_INVALID, "%s: extra rows come with y", what);
    if (int rc = row(p->extra, p->extra_offset, p->k, UGHIP_F32)) return rc;
  }
  if (p->gate_after && !p->gate) return set_error(UGHIP_ERR_INVALID, "%s: gate_after without a gate", what);
  if (p->gate)
    if (int rc = row(p->gate, p->gate_offset, p->k, UGHIP_F32)) return rc;
  if (p->gate && p->y) return set_error(UGHIP_ERR_UNSUPPORTED, "%s: a gate or a residual, not both", what);
  const size_t norm_groups = p->norm_groups ? p->norm_groups : 1;
  if (p->norm) {
    if (p->k % norm_groups) return set_error(UGHIP_ERR_INVALID, "%s: %zu elements in %zu groups", what, p->k, norm_groups);
    if (int rc = row(p->norm, 0, p->k, UGHIP_F32)) return rc;
  }
  if (int rc = row(p->w, 0, mats * w_rows * p->k, -1)) return rc;
  if (p->bias)
    if (int rc = row(p->bias, 0, w_rows, UGHIP_F32)) return rc;
  const size_t cols = p->route == 1 ? p->top * p->n : p->n;
  if (int rc = row(p->dst, p->dst_offset, cols, UGHIP_F32)) return rc;
  if (p->keep_x) {
    if (!p->y) return set_error(UGHIP_ERR_INVALID, "%s: nothing joins x", what);
    if (int rc = row(p->dst, p->x_out, p->k, UGHIP_F32)) return rc;
  }
  if (p->dst == p->x || p->dst == p->y || p->dst == p->gate || (p->extra && p->dst == p->extra)) return set_error(UGHIP_ERR_INVALID, "%s: dst aliases an input", what);
  if (p->act == UGHIP_ACT_GELU_MUL) {
    if (!p->table || (p->table->dtype != UGHIP_F32 && p->table->dtype != UGHIP_BF16)) return set_error(UGHIP_ERR_INVALID, "%s: a gate's table is F32 or BF16", what);
    if (int rc = row(p->table, 0, p->table_rows * p->table_stride, -1)) return rc;
    if (p->table_col > p->table_stride || p->n > p->table_stride - p->table_col) return set_error(UGHIP_ERR_BOUNDS, "%s: table columns %zu + %zu of %zu", what, p->table_col, p->n, p->table_stride);
    if (int rc = row(p->ids, 0, 1, UGHIP_I32)) return rc;
  }
  if (p->route == 1) {
    if (int rc = row(p->logits, p->logits_offset, p->experts, UGHIP_F32)) return rc;
    if (p->correction)
      if (int rc = row(p->correction, 0, p->experts, UGHIP_F32)) return rc;
  }
  if (int rc = device_activate(dev)) return rc;
  RowArgs a{};
  a.x = buf_ptr<float>(p->x) + p->x_offset;
  if (p->y) a.y = buf_ptr<float>(p->y) + p->y_offset, a.y_norm = buf_ptr<float>(p->y_norm);
  if (p->gate) a.gate = buf_ptr<float>(p->gate) + p->gate_offset, a.gate_after = p->gate_after != 0;
  if (p->extra) a.extra = buf_ptr<float>(p->extra) + p->extra_offset;
  a.glu = glu_form(p->act, p->act_alpha, p->act_shift, p->act_limit);
  a.norm = buf_ptr<float>(p->norm), a.norm_groups = (int)norm_groups;
  float* d = static_cast<float*>(p->dst->ptr);
  a.x_out = p->keep_x ? d + p->x_out : nullptr;
  a.dst = d + p->dst_offset;
  a.w = p->w->ptr;
  a.bias = buf_ptr<float>(p->bias);
  if (p->act == UGHIP_ACT_GELU_MUL) {
    a.table = p->table->ptr, a.table_bf16 = p->table->dtype == UGHIP_BF16, a.table_rows = (int)p->table_rows;
    a.table_stride = p->table_stride, a.table_col = p->table_col, a.ids = buf_ptr<int>(p->ids);
  }
  a.w_group = w_rows * p->k, a.eps = p->eps, a.inv_k = 1.f / (float)p->k, a.n = (int)p->n, a.k = (int)p->k, a.cols = (int)cols, a.segs = (int)segs;
  size_t lds = segs * ((p->k + RUN - 1) / RUN * RUN) * sizeof(float);
  if (p->route) {
    a.route = RouteArgs{buf_ptr<float>(p->correction), (int)p->experts, (int)p->groups, (int)p->keep, (int)p->top};
    a.route_ids = static_cast<int*>(p->route_ids->ptr), a.route_weights = static_cast<float*>(p->route_weights->ptr);
    if (p->route == 1) {
      a.logits = buf_ptr<float>(p->logits) + p->logits_offset;
      lds += (p->experts + (size_t)route_lds_floats(a.route.experts, a.route.groups) + 2 * p->top) * sizeof(float);
    }
  }
  const bool vec = p->k % 8 == 0 && (reinterpret_cast<uintptr_t>(a.w) & 15) == 0;
  auto a16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const size_t part = p->k / norm_groups;
  // pieces of eight elements, a thread each, and normed parts of whole halves of waves, of a power of two of lanes or of half a lane's
  const bool parts_fit = !p->norm || norm_groups == 1 || part % 256 == 0 || (part >= 4 && part < 256 && (part & (part - 1)) == 0);
  if (vec && total <= (size_t)WIDE_MAX && parts_fit && a16(a.x) && a16(a.y) && a16(a.gate) && a16(a.x_out) && a16(a.extra)) {
    const size_t work = p->route == 1 ? (p->experts + (size_t)route_lds_floats(a.route.experts, a.route.groups) + 2 * p->top) * sizeof(float) : 0;
    const bool plain = !a.y && !a.gate && !a.norm;
    auto go = [&](auto type) {
      using WT = decltype(type);
      if (p->route == 1) return launch_wide<WT, 2, 1, true>(dev, a, work);
      if (p->route == 2) return launch_wide<WT, 1, 2, true>(dev, a, 0);
      if (glu) return plain ? launch_wide<WT, 2, 0, true>(dev, a, 0) : launch_wide<WT, 2, 0, false>(dev, a, 0);
      return plain ? launch_wide<WT, 1, 0, true>(dev, a, 0) : launch_wide<WT, 1, 0, false>(dev, a, 0);
    };
    UGHIP_HIPCHK(p->w->dtype == UGHIP_BF16 ? go(uint16_t()) : go(float()));
    return UGHIP_OK;
  }
  UGHIP_HIPCHK(p->w->dtype == UGHIP_BF16 ? launch_any<uint16_t>(dev->stream, a, p->route, glu, lds, vec) : launch_any<float>(dev->stream, a, p->route, glu, lds, vec));
  return UGHIP_OK;
}
