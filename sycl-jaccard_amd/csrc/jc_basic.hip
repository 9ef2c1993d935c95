// Streaming kernels of the vertex-centric pipeline and the EC row expansion.
//
//   k_fill             FillKernel            jaccard.cpp:150-182
//   k_rowsum_*         Jaccard_RowSumKernel  jaccard.cpp:235-313 (+ parallel_prefix_sum :53-137)
//   k_vertex_weights   weighted-VC preamble  main.cpp:211-275 (W(k) = sum of row k's edge weights)
//   k_jw_*             Jaccard_JwKernel      jaccard.cpp:607-653
//   k_ec_scan          Jaccard_ec_scan       jaccard.cpp:654-700
//   k_count_above      the "non zero pairs" count  jaccard.cpp:811-819
//
// Row sums are one wave per row: the row is read with coalesced 256-byte loads
// and reduced with an xor butterfly (double-double, exact for fp32 addends of
// moderate dynamic range) instead of the reference's LDS-emulated 32-lane
// shuffle scan with two barriers per step.
#include <algorithm>
#include <numeric>

#include "jc_device.hpp"
#include "jc_internal.hpp"
#include "jc_profile.hpp"

namespace jc {

namespace {

struct DD2 {
  double hi, lo;
};

__device__ __forceinline__ DD2 add_dd(DD2 a, DD2 b) {
  const double s = a.hi + b.hi;
  const double bb = s - a.hi;
  const double e = (a.hi - (s - bb)) + (b.hi - bb);
  double t = a.lo + b.lo;
  t += e;
  const double hi = s + t;
  return DD2{hi, t - (hi - s)};
}

__device__ __forceinline__ DD2 add_d(DD2 a, double v) {
  const double s = a.hi + v;
  const double bb = s - a.hi;
  const double e = (a.hi - (s - bb)) + (v - bb);
  const double t = a.lo + e;
  const double hi = s + t;
  return DD2{hi, t - (hi - s)};
}

int grid_for(int64_t items, int per_block, int cap_per_cu) {
  const int64_t g = (items + per_block - 1) / per_block;
  return (int)std::max<int64_t>(1, std::min<int64_t>(g, (int64_t)device_cu_count() * cap_per_cu));
}

// Grid for kernels that stride over rows with one wave per row: an odd
// workgroup count, so rows at ids with many trailing zero bits (the hubs of
// RMAT-like graphs) do not all land on the same few waves.
int grid_rows(int64_t rows, int waves_per_block, int cap_per_cu) {
  return grid_for(rows, waves_per_block, cap_per_cu) | 1;
}

}  // namespace

template <typename T>
__global__ void k_fill(T* __restrict__ x, int64_t n, T v, const int* skip) {
  if (skip && *skip) return;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    x[i] = v;
}

hipError_t launch_fill_f32(float* x, int64_t n, float v, hipStream_t s) {
  ProfScope ps_("fill", s);
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill<float>, dim3(grid_for(n, 256 * 4, 32)), dim3(256), 0, s, x, n, v,
                     (const int*)nullptr);
  return hipGetLastError();
}
hipError_t launch_fill_u32(uint32_t* x, int64_t n, uint32_t v, hipStream_t s, const int* skip) {
  ProfScope ps_("fill", s);
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill<uint32_t>, dim3(grid_for(n, 256 * 4, 32)), dim3(256), 0, s, x, n, v, skip);
  return hipGetLastError();
}
hipError_t launch_fill_u64(uint64_t* x, int64_t n, uint64_t v, hipStream_t s, const int* skip) {
  ProfScope ps_("fill", s);
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill<uint64_t>, dim3(grid_for(n, 256 * 4, 32)), dim3(256), 0, s, x, n, v, skip);
  return hipGetLastError();
}

// Unweighted row sum: work[row] = (float)degree (jaccard.cpp:257-258).
__global__ void k_rowsum_deg(int32_t n, const int32_t* __restrict__ off, float* __restrict__ work) {
  for (int32_t u = blockIdx.x * blockDim.x + threadIdx.x; u < n; u += gridDim.x * blockDim.x)
    work[u] = (float)(off[u + 1] - off[u]);
}

// Weighted row sum over column weights: sum_{k in row u} v[ind[k]] (ind may be
// nullptr: identity index, i.e. the row's own edge weights, as main.cpp:216-257
// arranges with its presumInd buffer). By row length: rows of at most
// kRowShort entries by groups of 4 lanes (k_rowsum_w), rows up to kRowWave
// entries one wave per row from a list (k_rowsum_w_med), longer rows one
// workgroup per row from a list (k_rowsum_w_long). Loads are unrolled 4x per
// lane.
#ifndef JC_ROW_WAVE
#define JC_ROW_WAVE 2048
#endif
constexpr int kRowWave = JC_ROW_WAVE;
constexpr int kRowU = 4;

// Loads of one unrolled step are unconditional (clamped index) so they are
// all in flight together; IDX selects v[ind[p]] (column weights) or v[p]
// (the row's own edge weights).
template <bool IDX, int U>
__device__ __forceinline__ void gather_step(const int32_t* __restrict__ ind, const float* __restrict__ v, int p0,
                                            int stride, int lane, int end, float (&x)[U]) {
  int q[U];
#pragma unroll
  for (int t = 0; t < U; ++t) q[t] = min(p0 + t * stride + lane, end - 1);
  if constexpr (IDX) {
#pragma unroll
    for (int t = 0; t < U; ++t) q[t] = ind[q[t]];
  }
#pragma unroll
  for (int t = 0; t < U; ++t) x[t] = v[q[t]];
#pragma unroll
  for (int t = 0; t < U; ++t)
    if (p0 + t * stride + lane >= end) x[t] = 0.0f;
}

// Rows of at most kRowShort entries (most rows of power-law graphs), 16
// consecutive rows per wave and iteration, each summed by its own group of 4
// lanes (groups of 8 measured the same or slightly slower). (One wave per row
// leaves most lanes idle and pays a row's load latency per row.) Rows of up
// to kRowWave entries are listed by k_collect_rows and summed one wave per
// row by k_rowsum_w_med: summed here one after another by the whole wave,
// they made the waves that met many of them (power-law graphs put them at
// structured ids) the kernel's tail (RMAT-22: gathered sums 1.52 -> 0.83 ms,
// vertex weights 0.63 -> 0.41 ms with the lists). The double-double sums are
// exact, so the lane split does not change the result.
constexpr int kRowShort = 64;
#ifndef JC_ROW_GROUP
#define JC_ROW_GROUP 4
#endif
constexpr int kRowGroup = JC_ROW_GROUP;

template <typename OutT, bool IDX>
__global__ void k_rowsum_w(int32_t n, const int32_t* __restrict__ off, const int32_t* __restrict__ ind,
                           const float* __restrict__ v, OutT* __restrict__ out, const int* skip) {
  if (skip && *skip) return;
  constexpr int R = kWave / kRowGroup;  // rows per wave and iteration
  const int lane = lane_id();
  const int gl = lane % kRowGroup;
  const int nw = gridDim.x * (blockDim.x / kWave);
  for (int32_t base = (blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave) * R; base < n; base += nw * R) {
    const int32_t u = base + lane / kRowGroup;
    int o = 0, d = 0;
    if (u < n) {
      o = off[u];
      d = off[u + 1] - o;
    }
    const bool short_row = u < n && d <= kRowShort;
    {
      const int ds = short_row ? d : 0;
      DD2 acc{0.0, 0.0};
      for (int p0 = o; p0 < o + ds; p0 += kRowGroup * kRowU) {
        float x[kRowU];
        gather_step<IDX, kRowU>(ind, v, p0, kRowGroup, gl, o + ds, x);
#pragma unroll
        for (int t = 0; t < kRowU; ++t) acc = add_d(acc, (double)x[t]);
      }
#pragma unroll
      for (int sh = 1; sh < kRowGroup; sh <<= 1)
        acc = add_dd(acc, DD2{__shfl_xor(acc.hi, sh), __shfl_xor(acc.lo, sh)});
      if (short_row && gl == 0) out[u] = (OutT)acc.hi;
    }
  }
}

// Rows of kRowShort + 1 .. kRowWave entries, one wave per row; wave w of the
// grid takes the list's entries w, w + waves, ..., and the grid has several
// times the waves the device holds at once, so the dispatcher balances the
// rows' unequal lengths (an atomic cursor shared by every wave serialises on
// its one address: measured slower). The list is stored from the end of
// `list` backwards (k_collect_rows).
#ifndef JC_MED_U
#define JC_MED_U 4
#endif
constexpr int kMedU = JC_MED_U;

template <typename OutT, bool IDX>
__global__ void k_rowsum_w_med(int32_t n, const int32_t* __restrict__ off, const int32_t* __restrict__ ind,
                               const float* __restrict__ v, OutT* __restrict__ out, const int* __restrict__ list,
                               const int* __restrict__ counters) {
  const int lane = lane_id();
  const int count = counters[2];
  const int nw = gridDim.x * (blockDim.x / kWave);
  for (int r = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; r < count; r += nw) {
    const int32_t u = list[n - 1 - r];
    const int o = off[u], d = off[u + 1] - o;
    DD2 acc{0.0, 0.0};
    for (int p0 = o; p0 < o + d; p0 += kWave * kMedU) {
      float x[kMedU];
      gather_step<IDX, kMedU>(ind, v, p0, kWave, lane, o + d, x);
#pragma unroll
      for (int t = 0; t < kMedU; ++t) acc = add_d(acc, (double)x[t]);
    }
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) acc = add_dd(acc, DD2{__shfl_xor(acc.hi, sh), __shfl_xor(acc.lo, sh)});
    if (lane == 0) out[u] = (OutT)acc.hi;
  }
}

// Rows longer than kRowWave fill list[0 ..) (counters[0]), taken from an
// atomic cursor (counters[1]) by a persistent grid of 1024-thread
// workgroups, one row each. (A static row-to-workgroup map is not used: in
// power-law graphs the long rows sit at structured ids -- RMAT hubs have many
// trailing zero bits -- and any fixed stride piles them onto a few
// workgroups.) Rows of kRowShort + 1 .. kRowWave entries fill
// list[n-1] downwards (counters[2]) for k_rowsum_w_med. The lists are
// disjoint, so n entries hold both. Each workgroup takes a contiguous range
// of rows: it counts them, scans the counts over its threads and reserves
// its places with one atomic per list, then writes (one atomic per wave on
// one counter serialised: 0.22 ms on RMAT-22).
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_collect_rows(int32_t n, const int32_t* __restrict__ off,
                                                        int* __restrict__ list, int* __restrict__ counters,
                                                        const int* skip) {
  if (skip && *skip) return;  // empty lists: the kernels over them end at once
  constexpr int NW = BLOCK / kWave;
  __shared__ int s_w[2][NW];
  __shared__ int s_base[2];
  const int lane = lane_id(), w = threadIdx.x / kWave;
  const int64_t per = ((int64_t)n + gridDim.x - 1) / gridDim.x;
  const int64_t b0 = per * blockIdx.x, b1 = b0 + per;
  const int32_t r0 = (int32_t)(b0 < n ? b0 : n);
  const int32_t r1 = (int32_t)(b1 < n ? b1 : n);
  int cl = 0, cm = 0;
  for (int32_t u = r0 + threadIdx.x; u < r1; u += BLOCK) {
    const int d = off[u + 1] - off[u];
    cl += d > kRowWave ? 1 : 0;
    cm += d > kRowShort && d <= kRowWave ? 1 : 0;
  }
  // inclusive scans over the wave, then over the waves
  int il = cl, im = cm;
#pragma unroll
  for (int sh = 1; sh < kWave; sh <<= 1) {
    const int tl = __shfl_up(il, sh), tm = __shfl_up(im, sh);
    if (lane >= sh) {
      il += tl;
      im += tm;
    }
  }
  if (lane == kWave - 1) {
    s_w[0][w] = il;
    s_w[1][w] = im;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int tl = 0, tm = 0;
    for (int k = 0; k < NW; ++k) {
      const int a = s_w[0][k], b = s_w[1][k];
      s_w[0][k] = tl;
      s_w[1][k] = tm;
      tl += a;
      tm += b;
    }
    s_base[0] = tl ? atomicAdd(&counters[0], tl) : 0;
    s_base[1] = tm ? atomicAdd(&counters[2], tm) : 0;
  }
  __syncthreads();
  int pl = s_base[0] + s_w[0][w] + il - cl;
  int pm = s_base[1] + s_w[1][w] + im - cm;
  for (int32_t u = r0 + threadIdx.x; u < r1; u += BLOCK) {
    const int d = off[u + 1] - off[u];
    if (d > kRowWave) list[pl++] = u;
    else if (d > kRowShort) list[n - 1 - pm++] = u;
  }
}

template <typename OutT, bool IDX, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_rowsum_w_long(const int32_t* __restrict__ off,
                                                         const int32_t* __restrict__ ind,
                                                         const float* __restrict__ v, OutT* __restrict__ out,
                                                         const int* __restrict__ list, int* counters) {
  __shared__ double part[2][BLOCK / kWave];
  __shared__ int s_row;
  const int count = counters[0];
  for (;;) {
    if (threadIdx.x == 0) {
      const int r = atomicAdd(&counters[1], 1);
      s_row = r < count ? list[r] : -1;
    }
    __syncthreads();
    const int32_t u = s_row;
    if (u < 0) return;
    const int o = off[u], d = off[u + 1] - o;
    DD2 acc{0.0, 0.0};
    for (int p0 = o; p0 < o + d; p0 += BLOCK * kRowU) {
      float x[kRowU];
      gather_step<IDX, kRowU>(ind, v, p0, BLOCK, threadIdx.x, o + d, x);
#pragma unroll
      for (int t = 0; t < kRowU; ++t) acc = add_d(acc, (double)x[t]);
    }
    for (int s = 1; s < kWave; s <<= 1) acc = add_dd(acc, DD2{__shfl_xor(acc.hi, s), __shfl_xor(acc.lo, s)});
    if (lane_id() == 0) {
      part[0][threadIdx.x / kWave] = acc.hi;
      part[1][threadIdx.x / kWave] = acc.lo;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      DD2 t{0.0, 0.0};
      for (int w = 0; w < BLOCK / kWave; ++w) t = add_dd(t, DD2{part[0][w], part[1][w]});
      out[u] = (OutT)t.hi;
    }
    __syncthreads();
  }
}

// Row sums of all but the largest graphs in one launch: the five launches of
// the way above take 40 us however small the graph, this 6 to 8 (9001 vertices,
// 2.4e5 entries). A workgroup takes 64 rows: rows up to kRowShort entries by 4
// lanes each, up to kOneWave by a wave, longer ones by the workgroup (and those
// above kHubRow by one of k_rowsum_hubs). Fewer rows, down to 8, where 64 would
// leave less than four workgroups per CU and have more than 2048 entries (3000
// rows of 780 entries 36 -> 10 us, 20000 of 100 27 -> 12). EX: facts[workgroup]
// receives the range facts of v and of its sums (k_exact_scan); added up by
// atomics on one line they took 60 us on 150000 vertices. Pairs of rows come in an
// order that scatters them (step): hubs are neighbours in graphs sorted by
// degree, and in RMAT-like ones their ids have many trailing zeros, so with
// consecutive rows or with a fixed stride they meet in a few workgroups
// (RMAT-18 gathered sums 86 us with a stride, 56 so; Chung-Lu of 8.4M entries
// 134 us in runs of 16 rows, 43 in pairs). Single rows measured
// a little better still on those and a little worse on uniform random ones.
constexpr int kOneWave = 1024;
constexpr int kOneRun = 2;   // consecutive rows that stay together
constexpr int kHubRow = 32768;
constexpr int kOneU = 8;  // loads in flight per thread in those
// Above, hub rows outlast one workgroup. Vertex weights / gathered sums, one
// launch and five, us: RMAT of 5.8M entries 23 / 34 and 45 / 59, 11.7M 40 / 63
// and 64 / 94, 17.8M 58 / 94 and 90 / 128, 31M 104 / 232 and 121 / 201; Chung-Lu
// 8.4M 31 / 43 and 45 / 61, 19.2M 60 / 107 and 69 / 108; uniform random 16M 36 /
// 104 and 52 / 112.
constexpr int64_t kOneMaxEdges = 20 << 20;
// Above, the scattered order costs more than the launches: uniform random, 1M
// vertices and 2M entries 29 / 41 us and 42 / 46, 4M and 8M 103 / 225 and 84 / 147.
constexpr int32_t kOneMaxRows = 2 << 20;

__device__ __forceinline__ void exact_fact(float w, int& lsb, int& bad) {
  const uint32_t b = __float_as_uint(w);
  const uint32_t ex = (b >> 23) & 0xFFu, man = b & 0x7FFFFFu;
  if ((b >> 31) && (b << 1)) bad = 1;  // negative (-0 is harmless)
  if (ex == 0xFFu) {
    bad = 1;
  } else if (ex != 0 || man != 0) {
    const uint32_t full = ex ? (man | 0x800000u) : man;
    lsb = min(lsb, (ex ? (int)ex - 150 : -149) + __builtin_ctz(full));
  }
}

__device__ __forceinline__ void exact_sum_fact(double sv, int& mx, int& bad) {
  if (!(sv >= 0.0) || isinf(sv))
    bad = 1;
  else if (sv > 0.0)
    mx = max(mx, ilogb(sv) + 1);
}

template <typename OutT, bool IDX, bool EX>
__global__ __launch_bounds__(256) void k_rowsum_one(int32_t n, const int32_t* __restrict__ off,
                                                    const int32_t* __restrict__ ind, const float* __restrict__ v,
                                                    OutT* __restrict__ out, ExactInfo* facts, uint32_t step, int rows,
                                                    const int* skip) {
  if (skip && *skip) return;
  constexpr int BLOCK = 256, NW = BLOCK / kWave, R = BLOCK / kRowGroup;
  __shared__ int s_long[R], s_nlong;
  __shared__ double part[2][NW];
  __shared__ int s_r[3][NW];
  const int tid = threadIdx.x, lane = lane_id(), w = tid / kWave, gl = lane % kRowGroup;
  int lsb = INT32_MAX, mx = INT32_MIN, bad = 0;
  auto put = [&](int32_t u, double sum) {
    out[u] = (OutT)sum;
    if constexpr (EX) exact_sum_fact(sum, mx, bad);
  };
  const uint32_t runs = ((uint32_t)n + kOneRun - 1) / kOneRun;
  for (int64_t i0 = (int64_t)blockIdx.x * rows; i0 < n; i0 += (int64_t)gridDim.x * rows) {
    if (tid == 0) s_nlong = 0;
    __syncthreads();
    const uint32_t run = (uint32_t)(i0 / kOneRun) + tid / (kOneRun * kRowGroup);
    const uint32_t at = (uint32_t)((uint64_t)run * step % runs) * kOneRun + tid / kRowGroup % kOneRun;
    const int32_t u = (int32_t)at;
    int o = 0, d = 0;
    const bool live = tid / kRowGroup < rows && run < runs && at < (uint32_t)n;
    if (live) {
      o = off[u];
      d = off[u + 1] - o;
      if constexpr (EX) {
        if (gl == 0) exact_fact(v[u], lsb, bad);
      }
    }
    const int ds = live && d <= kRowShort ? d : 0;
    DD2 acc{0.0, 0.0};
    for (int p0 = o; p0 < o + ds; p0 += kRowGroup * kRowU) {
      float x[kRowU];
      gather_step<IDX, kRowU>(ind, v, p0, kRowGroup, gl, o + ds, x);
#pragma unroll
      for (int t = 0; t < kRowU; ++t) acc = add_d(acc, (double)x[t]);
    }
#pragma unroll
    for (int sh = 1; sh < kRowGroup; sh <<= 1) acc = add_dd(acc, DD2{__shfl_xor(acc.hi, sh), __shfl_xor(acc.lo, sh)});
    if (live && gl == 0) {
      if (d <= kRowShort) put(u, acc.hi);
      else if (d <= kHubRow) s_long[atomicAdd(&s_nlong, 1)] = u;
    }
    __syncthreads();
    const int nl = s_nlong;
    for (int j = w; j < nl; j += NW) {
      const int32_t q = s_long[j];
      const int qo = off[q], qe = off[q + 1];
      if (qe - qo > kOneWave) continue;
      DD2 a2{0.0, 0.0};
      for (int p0 = qo; p0 < qe; p0 += kWave * kRowU) {
        float x[kRowU];
        gather_step<IDX, kRowU>(ind, v, p0, kWave, lane, qe, x);
#pragma unroll
        for (int t = 0; t < kRowU; ++t) a2 = add_d(a2, (double)x[t]);
      }
#pragma unroll
      for (int sh = 1; sh < kWave; sh <<= 1) a2 = add_dd(a2, DD2{__shfl_xor(a2.hi, sh), __shfl_xor(a2.lo, sh)});
      if (lane == 0) put(q, a2.hi);
    }
    for (int j = 0; j < nl; ++j) {
      const int32_t q = s_long[j];
      const int qo = off[q], qe = off[q + 1];
      if (qe - qo <= kOneWave) continue;  // uniform over the workgroup
      DD2 a2{0.0, 0.0};
      for (int p0 = qo; p0 < qe; p0 += BLOCK * kOneU) {
        float x[kOneU];
        gather_step<IDX, kOneU>(ind, v, p0, BLOCK, tid, qe, x);
#pragma unroll
        for (int t = 0; t < kOneU; ++t) a2 = add_d(a2, (double)x[t]);
      }
#pragma unroll
      for (int sh = 1; sh < kWave; sh <<= 1) a2 = add_dd(a2, DD2{__shfl_xor(a2.hi, sh), __shfl_xor(a2.lo, sh)});
      if (lane == 0) {
        part[0][w] = a2.hi;
        part[1][w] = a2.lo;
      }
      __syncthreads();
      if (tid == 0) {
        DD2 t{0.0, 0.0};
        for (int k = 0; k < NW; ++k) t = add_dd(t, DD2{part[0][k], part[1][k]});
        put(q, t.hi);
      }
      __syncthreads();
    }
    __syncthreads();  // the list is read before it is begun again
  }
  if constexpr (EX) {
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      lsb = min(lsb, __shfl_xor(lsb, o));
      mx = max(mx, __shfl_xor(mx, o));
      bad |= __shfl_xor(bad, o);
    }
    if (lane == 0) {
      s_r[0][w] = lsb;
      s_r[1][w] = mx;
      s_r[2][w] = bad;
    }
    __syncthreads();
    if (tid == 0) {
      for (int k = 1; k < NW; ++k) {
        lsb = min(lsb, s_r[0][k]);
        mx = max(mx, s_r[1][k]);
        bad |= s_r[2][k];
      }
      facts[blockIdx.x] = ExactInfo{lsb, mx, bad, 0};
    }
  }
}

// Rows above kHubRow entries: a workgroup of 1024 threads has twice the loads in
// flight, and 63 other rows do not wait for it. Such rows are told apart by the
// stretch of kHubRow entries that they start in, and cover the end of it, so one
// workgroup per stretch finds its row by searching the offsets, 64 at a time. EX:
// the last one also gathers the nfacts facts of k_rowsum_one's workgroups.
// Gathered sums, us, five launches / in k_rowsum_one / here: one row of 1M
// entries 244 / 391 / 204, of 2M 460 / 768 / 401, three of 300K 92 / 223 / 67,
// eight of 500K 137 / 404 / 107; 3 us where there is none.
template <typename OutT, bool IDX, bool EX>
__global__ __launch_bounds__(1024) void k_rowsum_hubs(int32_t n, const int32_t* __restrict__ off,
                                                      const int32_t* __restrict__ ind, const float* __restrict__ v,
                                                      OutT* __restrict__ out, const ExactInfo* facts, int nfacts,
                                                      ExactInfo* info, const int* skip) {
  if (skip && *skip) return;
  constexpr int BLOCK = 1024;
  __shared__ double part[2][BLOCK / kWave];
  const int lane = lane_id(), w = threadIdx.x / kWave;
  if constexpr (EX) {
    if (blockIdx.x == gridDim.x - 1) gather_facts(facts, nfacts, info);
  }
  const int m = off[n];
  for (int64_t s = blockIdx.x; (s + 1) * kHubRow < m; s += gridDim.x) {
    const int at = (int)((s + 1) * kHubRow);
    // the last row that starts at or before `at`; every wave for itself
    int u = 0;
    for (int len = n; len > 1;) {
      const int stride = (len + kWave - 1) / kWave;
      const int k = lane * stride;
      u += stride * (popc64(ballot(k < len && off[u + min(k, len - 1)] <= at)) - 1);
      len = min(stride, n - u);
    }
    const int o = off[u], e = off[u + 1];
    if (e - o <= kHubRow || o < at - kHubRow || o >= at) continue;  // uniform
    DD2 acc{0.0, 0.0};
    for (int p0 = o; p0 < e; p0 += BLOCK * kOneU) {
      float x[kOneU];
      gather_step<IDX, kOneU>(ind, v, p0, BLOCK, threadIdx.x, e, x);
#pragma unroll
      for (int t = 0; t < kOneU; ++t) acc = add_d(acc, (double)x[t]);
    }
#pragma unroll
    for (int t = 1; t < kWave; t <<= 1) acc = add_dd(acc, DD2{__shfl_xor(acc.hi, t), __shfl_xor(acc.lo, t)});
    if (lane == 0) {
      part[0][w] = acc.hi;
      part[1][w] = acc.lo;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      DD2 t{0.0, 0.0};
      for (int k = 0; k < BLOCK / kWave; ++k) t = add_dd(t, DD2{part[0][k], part[1][k]});
      out[u] = (OutT)t.hi;
      if constexpr (EX) {
        int mx = INT32_MIN, bad = 0;
        exact_sum_fact(t.hi, mx, bad);
        if (mx > *(volatile int*)&info->max_exp) atomicMax(&info->max_exp, mx);
        if (bad) atomicOr(&info->bad, 1);
      }
    }
    __syncthreads();
  }
}

// Rows of a workgroup, see above.
int rows_one(int32_t n, int64_t m) {
  int rows = 64;
  while (rows > 8 && n < (int64_t)device_cu_count() * 4 * rows && m * rows > 2048ll * n) rows /= 2;
  return rows;
}

// A second round of rows would make the workgroups that met the long ones the
// tail (11.7M entries, 4097 workgroups: 84 us and not 39).
int grid_one(int32_t n, int rows) { return grid_rows((n + rows - 1) / rows, 1, 256); }

// Run k of the order is run k * step_one(n) mod runs: runs / golden ratio, less
// what it takes to share no factor with them.
uint32_t step_one(int32_t n) {
  const uint32_t runs = ((uint32_t)n + kOneRun - 1) / kOneRun;
  uint32_t p = (uint32_t)(runs * 0.6180339887498949);
  while (p > 1 && std::gcd(p, runs) != 1) --p;
  return std::max(p, 1u);
}

bool rowsum_one_launch(int32_t n, int64_t m) { return m <= kOneMaxEdges && n <= kOneMaxRows; }

template <typename OutT, bool IDX, bool EX>
static hipError_t rowsum_one(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* v, OutT* out,
                             ExactInfo* facts, int* nfacts, ExactInfo* info, hipStream_t s, const int* skip) {
  const int rows = rows_one(n, m), g = grid_one(n, rows);
  hipLaunchKernelGGL((k_rowsum_one<OutT, IDX, EX>), dim3(g), dim3(256), 0, s, n, off, ind, v, out, facts, step_one(n),
                     rows, skip);
  if (EX) *nfacts = n > kHubRow ? 0 : g;
  if (n > kHubRow)  // a row has at most n entries
    hipLaunchKernelGGL((k_rowsum_hubs<OutT, IDX, EX>), dim3(device_cu_count() * 3), dim3(1024), 0, s, n, off, ind, v,
                       out, facts, g, info, skip);
  return hipGetLastError();
}

hipError_t launch_rowsum_exact(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* v, double* S,
                               void* scratch, int* nfacts, ExactInfo* info, hipStream_t s, const int* skip) {
  ProfScope ps_("rowsum", s);
  // (one per workgroup, of eight rows at least: a part of rowsum_scratch_bytes)
  return rowsum_one<double, true, true>(n, m, off, ind, v, S, static_cast<ExactInfo*>(scratch), nfacts, info, s, skip);
}

// Sentinel fill of the result (when x is not null) and the start values of a
// pass's counters and range facts, in one launch.
__global__ void k_prepare(uint32_t* __restrict__ x, int64_t n, uint32_t v, int* __restrict__ z, int nz, ExactInfo* info,
                          const int* skip) {
  if (skip && *skip) x = nullptr;  // (the counters are read all the same)
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (x)
    for (int64_t i = t; i < n; i += (int64_t)gridDim.x * blockDim.x) x[i] = v;
  if (blockIdx.x == 0) {
    for (int i = threadIdx.x; i < nz; i += blockDim.x) z[i] = 0;
    if (info && threadIdx.x == 0) *info = ExactInfo{INT32_MAX, INT32_MIN, 0, 0};
  }
}

hipError_t launch_prepare(uint32_t* x, int64_t n, uint32_t v, int* zero, int nzero, ExactInfo* info, hipStream_t s,
                          const int* skip) {
  ProfScope ps_("fill", s);
  hipLaunchKernelGGL(k_prepare, dim3(x ? grid_for(n, 256 * 4, 32) : 1), dim3(256), 0, s, x, n, v, zero, nzero, info, skip);
  return hipGetLastError();
}

size_t rowsum_scratch_bytes(int32_t n) { return ((size_t)std::max(n, 1) + 4) * sizeof(int); }

// scratch: rowsum_scratch_bytes(n) bytes, or nullptr to use a stream-ordered
// allocation for the call.
template <typename OutT>
static hipError_t rowsum_both(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* v, OutT* out,
                              void* scratch, hipStream_t s, const int* skip = nullptr) {
  if (rowsum_one_launch(n, m)) {
    return ind ? rowsum_one<OutT, true, false>(n, m, off, ind, v, out, nullptr, nullptr, nullptr, s, skip)
               : rowsum_one<OutT, false, false>(n, m, off, ind, v, out, nullptr, nullptr, nullptr, s, skip);
  }
  CallBuf own;
  if (!scratch) {
    const hipError_t err = own.get(rowsum_scratch_bytes(n), s);
    if (err != hipSuccess) return err;
    scratch = own.p;
  }
  int* counters = static_cast<int*>(scratch);
  int* list = counters + 4;
  const int cus = device_cu_count();
  hipLaunchKernelGGL(k_fill<uint32_t>, dim3(1), dim3(64), 0, s, reinterpret_cast<uint32_t*>(counters), (int64_t)4, 0u,
                     (const int*)nullptr);
  hipLaunchKernelGGL(k_collect_rows<256>, dim3(grid_for(n, 256 * 4, 4)), dim3(256), 0, s, n, off, list, counters,
                     skip);
  const int gs = grid_rows((n + kWave / kRowGroup - 1) / (kWave / kRowGroup), 4, 64);
  const int gm = grid_rows(n, 4, 64);  // at most n listed rows, one per wave
  if (ind) {
    hipLaunchKernelGGL((k_rowsum_w<OutT, true>), dim3(gs), dim3(256), 0, s, n, off, ind, v, out, skip);
    hipLaunchKernelGGL((k_rowsum_w_med<OutT, true>), dim3(gm), dim3(256), 0, s, n, off, ind, v, out, list,
                       counters);
    hipLaunchKernelGGL((k_rowsum_w_long<OutT, true, 1024>), dim3(cus * 2), dim3(1024), 0, s, off, ind, v, out,
                       list, counters);
  } else {
    hipLaunchKernelGGL((k_rowsum_w<OutT, false>), dim3(gs), dim3(256), 0, s, n, off, ind, v, out, skip);
    hipLaunchKernelGGL((k_rowsum_w_med<OutT, false>), dim3(gm), dim3(256), 0, s, n, off, ind, v, out, list,
                       counters);
    hipLaunchKernelGGL((k_rowsum_w_long<OutT, false, 1024>), dim3(cus * 2), dim3(1024), 0, s, off, ind, v, out,
                       list, counters);
  }
  return hipGetLastError();
}

hipError_t launch_rowsum_f32(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* v,
                             float* work, void* scratch, hipStream_t s) {
  ProfScope ps_("rowsum", s);
  if (n <= 0) return hipSuccess;
  if (v == nullptr) {
    hipLaunchKernelGGL(k_rowsum_deg, dim3(grid_for(n, 256, 32)), dim3(256), 0, s, n, off, work);
    return hipGetLastError();
  }
  return rowsum_both<float>(n, m, off, ind, v, work, scratch, s);
}

hipError_t launch_rowsum_f64(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* v,
                             double* S, void* scratch, hipStream_t s, const int* skip) {
  ProfScope ps_("rowsum", s);
  if (n <= 0) return hipSuccess;
  return rowsum_both<double>(n, m, off, ind, v, S, scratch, s, skip);
}

hipError_t launch_vertex_weights(int32_t n, int64_t m, const int32_t* off, const float* edge_w, float* W,
                                 void* scratch, hipStream_t s) {
  ProfScope ps_("vertex_weights", s);
  if (n <= 0) return hipSuccess;
  return rowsum_both<float>(n, m, off, nullptr, edge_w, W, scratch, s);
}

// Jaccard weight: weight_j = Wi / (Ws - Wi) (jaccard.cpp:614-619).
__global__ void k_jw_f32(int64_t m, const float* __restrict__ wi, const float* __restrict__ ws,
                         float* __restrict__ out) {
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < m; j += (int64_t)gridDim.x * blockDim.x) {
    const float Wi = wi[j];
    const float Ws = ws[j];
    out[j] = Wi / (Ws - Wi);
  }
}

__global__ void k_jw_f64(int64_t m, const double* __restrict__ wi, const double* __restrict__ ws,
                         float* __restrict__ out) {
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < m; j += (int64_t)gridDim.x * blockDim.x) {
    const double Wi = wi[j];
    const double Ws = ws[j];
    out[j] = (float)(Wi / (Ws - Wi));
  }
}

hipError_t launch_jw_f32(int64_t m, const float* wi, const float* ws, float* out, hipStream_t s) {
  ProfScope ps_("jw", s);
  if (m <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_jw_f32, dim3(grid_for(m, 256 * 4, 32)), dim3(256), 0, s, m, wi, ws, out);
  return hipGetLastError();
}

hipError_t launch_jw_f64(int64_t m, const double* wi, const double* ws, float* out, hipStream_t s) {
  ProfScope ps_("jw", s);
  if (m <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_jw_f64, dim3(grid_for(m, 256 * 4, 32)), dim3(256), 0, s, m, wi, ws, out);
  return hipGetLastError();
}

// Row expansion: dest[k] = row(k), weight_j[k] = 0. One wave per row, so the
// writes of a row are coalesced (the reference writes a row with one thread).
__global__ void k_ec_scan(int32_t n, const int32_t* __restrict__ off, int32_t* __restrict__ dest,
                          float* __restrict__ wj) {
  const int nw = gridDim.x * (blockDim.x / kWave);
  for (int32_t u = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; u < n; u += nw) {
    const int o = off[u], e = off[u + 1];
    for (int p = o + lane_id(); p < e; p += kWave) {
      dest[p] = u;
      wj[p] = 0.0f;
    }
  }
}

hipError_t launch_ec_scan(int32_t n, const int32_t* off, int32_t* dest, float* wj, hipStream_t s) {
  ProfScope ps_("ec_scan", s);
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_ec_scan, dim3(grid_rows(n, 4, 64)), dim3(256), 0, s, n, off, dest, wj);
  return hipGetLastError();
}

__global__ void k_count_above(int64_t m, const float* __restrict__ x, float thresh,
                              unsigned long long* cnt) {
  unsigned long long c = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
    c += x[i] > thresh ? 1u : 0u;
  for (int s = 1; s < kWave; s <<= 1) c += __shfl_xor(c, s);
  if (lane_id() == 0 && c) atomicAdd(cnt, c);
}

hipError_t launch_count_above(int64_t m, const float* x, float thresh, unsigned long long* cnt,
                              hipStream_t s) {
  ProfScope ps_("count_above", s);
  if (m <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_count_above, dim3(grid_for(m, 256 * 8, 16)), dim3(256), 0, s, m, x, thresh, cnt);
  return hipGetLastError();
}

// CSR validation. flags[0]: offsets bad (offsets[0] != 0, decreasing, or
// offsets[n] != m, or out of [0, m]); flags[1]: a column out of [0, n);
// flags[2]: a row not strictly increasing (unsorted or duplicate columns).
// Every read is bounds-checked before it is made.
__global__ void k_validate(int32_t n, int64_t m, const int32_t* __restrict__ off,
                           const int32_t* __restrict__ ind, int* flags) {
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nt = (int64_t)gridDim.x * blockDim.x;
  if (tid == 0 && (off[0] != 0 || (int64_t)off[n] != m)) atomicOr(&flags[0], 1);
  for (int64_t u = tid; u < n; u += nt) {
    const int32_t a = off[u], b = off[u + 1];
    if (a < 0 || b < a || (int64_t)b > m) atomicOr(&flags[0], 1);
  }
  for (int64_t k = tid; k < m; k += nt) {
    const int32_t c = ind[k];
    if (c < 0 || c >= n) atomicOr(&flags[1], 1);
  }
}

// Second pass (only run when the offsets are valid): sortedness per row.
__global__ void k_validate_rows(int32_t n, const int32_t* __restrict__ off,
                                const int32_t* __restrict__ ind, int* flags) {
  const int nw = gridDim.x * (blockDim.x / kWave);
  for (int32_t u = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; u < n; u += nw) {
    const int o = off[u], e = off[u + 1];
    bool bad = false;
    for (int p = o + 1 + lane_id(); p < e; p += kWave) bad |= ind[p] <= ind[p - 1];
    if (ballot(bad) && lane_id() == 0) atomicOr(&flags[2], 1);
  }
}

hipError_t launch_validate(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, int* flags,
                           hipStream_t s) {
  hipLaunchKernelGGL(k_validate, dim3(grid_for(std::max<int64_t>(n, m), 256 * 4, 16)), dim3(256), 0, s, n, m,
                     off, ind, flags);
  return hipGetLastError();
}

hipError_t launch_validate_rows(int32_t n, const int32_t* off, const int32_t* ind, int* flags,
                                hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_validate_rows, dim3(grid_rows(n, 4, 64)), dim3(256), 0, s, n, off, ind, flags);
  return hipGetLastError();
}

// Symmetry check: flag if some stored (u, v) has no stored (v, u).
__global__ void k_symcheck(int32_t n, const int32_t* __restrict__ off, const int32_t* __restrict__ ind,
                           int* flag) {
  const int nw = gridDim.x * (blockDim.x / kWave);
  for (int32_t u = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; u < n; u += nw) {
    bool bad = false;
    for (int p = off[u] + lane_id(); p < off[u + 1]; p += kWave) {
      const int32_t v = ind[p];
      const int lo = off[v], hi = off[v + 1];
      const int q = lane_lower_bound(ind, lo, hi, u);
      bad |= !(q < hi && ind[q] == u);
    }
    if (ballot(bad) && lane_id() == 0) atomicOr(flag, 1);
  }
}

hipError_t launch_symcheck(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, int* flag,
                           hipStream_t s) {
  (void)m;
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_symcheck, dim3(grid_rows(n, 4, 64)), dim3(256), 0, s, n, off, ind, flag);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Range facts of vertex weights and row sums (ExactInfo): smallest exponent
// of a set bit over all weights, bound exponent of the largest row sum, and
// whether any weight or sum is negative or not finite.
__global__ void k_exact_init(ExactInfo* e) {
  if (threadIdx.x == 0) *e = ExactInfo{INT32_MAX, INT32_MIN, 0, 0};
}

__global__ __launch_bounds__(256) void k_exact_scan(int32_t n, const float* __restrict__ vw,
                                                    const double* __restrict__ S, ExactInfo* info,
                                                    const int* skip) {
  if (skip && *skip) return;
  int lsb = INT32_MAX, mx = INT32_MIN, bad = 0;
  for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    exact_fact(vw[i], lsb, bad);
    exact_sum_fact(S[i], mx, bad);
  }
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    lsb = min(lsb, __shfl_xor(lsb, o));
    mx = max(mx, __shfl_xor(mx, o));
    bad |= __shfl_xor(bad, o);
  }
  // one set of atomics per workgroup (per wave, the few counters serialise)
  __shared__ int s_r[3][256 / kWave];
  const int w = threadIdx.x / kWave;
  if (lane_id() == 0) {
    s_r[0][w] = lsb;
    s_r[1][w] = mx;
    s_r[2][w] = bad;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < (int)(blockDim.x / kWave); ++k) {
      lsb = min(lsb, s_r[0][k]);
      mx = max(mx, s_r[1][k]);
      bad |= s_r[2][k];
    }
    if (lsb != INT32_MAX) atomicMin(&info->min_lsb, lsb);
    if (mx != INT32_MIN) atomicMax(&info->max_exp, mx);
    if (bad) atomicOr(&info->bad, 1);
  }
}

hipError_t launch_exact_info(int32_t n, const float* vw, const double* S, ExactInfo* info, hipStream_t s,
                             const int* skip) {
  hipLaunchKernelGGL(k_exact_init, dim3(1), dim3(64), 0, s, info);
  if (n > 0) hipLaunchKernelGGL(k_exact_scan, dim3(grid_for(n, 256 * 4, 4)), dim3(256), 0, s, n, vw, S, info,
                                skip);
  return hipGetLastError();
}

int device_cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    cached[dev] = v;
  }
  return cached[dev];
}

}  // namespace jc
