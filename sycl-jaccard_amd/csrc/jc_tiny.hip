// Graphs whose whole CSR fits the LDS of a CU, in one launch.
//
// What such a graph costs is launches and chains of dependent reads: the owner
// engine's ten launches took 63 us on 700 vertices and 7966 entries, with 27
// of them in one wave's walk over a 128-entry row. Here every workgroup copies
// the offsets and columns (weighted: the weights too, from which it forms the
// row sums) to LDS, with all reads in flight at once, and its groups of 16
// lanes take stored entries: the shorter row's columns are searched in the
// longer row (jaccard.cpp:711-742, the reference's loop, in LDS). Each stored
// entry is computed by itself, so no fill, no schedule and no fix-up of
// asymmetric entries. Measured (whole calls): 700 vertices unweighted 66.8 ->
// 10.3 us, weighted 93 -> 21.
//
// Sums are double-double like the other paths', exact where theirs are.
#include <algorithm>

#include "jc_device.hpp"
#include "jc_internal.hpp"
#include "jc_profile.hpp"

namespace jc {

namespace {

constexpr int kTinyBlock = 1024;
constexpr int kTinyGroup = 16;
constexpr size_t kTinyLds = 150 * 1024;

struct Sum2 {
  double hi, lo;
};

__device__ __forceinline__ Sum2 add2(Sum2 a, Sum2 b) {
  const double s = a.hi + b.hi;
  const double bb = s - a.hi;
  const double e = (a.hi - (s - bb)) + (b.hi - bb);
  double t = a.lo + b.lo;
  t += e;
  const double hi = s + t;
  return Sum2{hi, t - (hi - s)};
}

__device__ __forceinline__ Sum2 group_sum(Sum2 v) {
#pragma unroll
  for (int o = 1; o < kTinyGroup; o <<= 1) v = add2(v, Sum2{__shfl_xor(v.hi, o), __shfl_xor(v.lo, o)});
  return v;
}

size_t tiny_bytes(int32_t n, int64_t m, bool weighted) {
  return (weighted ? (size_t)n * (sizeof(double) + sizeof(float)) : 0) + ((size_t)n + 1 + (size_t)m) * sizeof(int32_t);
}

// LDS: [row sums n x fp64, weights n x fp32,] offsets n + 1, columns m
template <bool W>
__global__ __launch_bounds__(kTinyBlock) void k_tiny(int32_t n, int32_t m, const int32_t* __restrict__ off,
                                                     const int32_t* __restrict__ ind, const float* __restrict__ vw,
                                                     float* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem[];
  double* const s_S = reinterpret_cast<double*>(smem);
  float* const s_w = reinterpret_cast<float*>(smem + (W ? (size_t)n * sizeof(double) : 0));
  int32_t* const s_off = reinterpret_cast<int32_t*>(s_w + (W ? n : 0));
  int32_t* const s_ind = s_off + n + 1;
  const int tid = threadIdx.x, gl = tid % kTinyGroup, grp = tid / kTinyGroup;
  constexpr int NG = kTinyBlock / kTinyGroup;
  // four reads per thread in flight
  auto stage = [&](auto* dst, const auto* src, int cnt) {
    for (int i = tid; i < cnt; i += 4 * kTinyBlock) {
      decltype(src[0] + src[0]) x[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) x[t] = src[min(i + t * kTinyBlock, cnt - 1)];
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (i + t * kTinyBlock < cnt) dst[i + t * kTinyBlock] = x[t];
    }
  };
  stage(s_off, off, n + 1);
  stage(s_ind, ind, m);
  if constexpr (W) stage(s_w, vw, n);
  __syncthreads();
  if constexpr (W) {
    for (int u = grp; u < n; u += NG) {
      const int o = s_off[u], e = s_off[u + 1];
      Sum2 acc{0.0, 0.0};
      for (int p = o + gl; p < e; p += kTinyGroup) acc = add2(acc, Sum2{(double)s_w[s_ind[p]], 0.0});
      acc = group_sum(acc);
      if (gl == 0) s_S[u] = acc.hi;
    }
    __syncthreads();
  }
  for (int k = blockIdx.x * NG + grp; k < m; k += gridDim.x * NG) {
    // the row of entry k: the last whose offset is at most k
    int lo = 0, len = n;
    while (len > 0) {
      const int half = len >> 1;
      if (s_off[lo + half + 1] <= k) {
        lo += half + 1;
        len -= half + 1;
      } else {
        len = half;
      }
    }
    const int u = lo, x = s_ind[k];
    const int ou = s_off[u], du = s_off[u + 1] - ou;
    const int ox = s_off[x], dx = s_off[x + 1] - ox;
    const bool u_long = du > dx;
    const int oL = u_long ? ou : ox, dL = u_long ? du : dx;
    const int oS = u_long ? ox : ou, dS = u_long ? dx : du;
    int cnt = 0;
    Sum2 acc{0.0, 0.0};
    for (int p = gl; p < dS; p += kTinyGroup) {
      const int32_t y = s_ind[oS + p];
      int a = oL, l = dL;
      while (l > 0) {
        const int half = l >> 1;
        if (s_ind[a + half] < y) {
          a += half + 1;
          l -= half + 1;
        } else {
          l = half;
        }
      }
      if (a < oL + dL && s_ind[a] == y) {
        ++cnt;
        if constexpr (W) acc = add2(acc, Sum2{(double)s_w[y], 0.0});
      }
    }
    if constexpr (W) {
      acc = group_sum(acc);
      if (gl == 0) out[k] = (float)(acc.hi / ((s_S[u] + s_S[x]) - acc.hi));
    } else {
#pragma unroll
      for (int o = 1; o < kTinyGroup; o <<= 1) cnt += __shfl_xor(cnt, o);
      const float fI = (float)cnt;
      if (gl == 0) out[k] = fI / ((float)(du + dx) - fI);
    }
  }
}

}  // namespace

bool tiny_fits(int32_t n, int64_t m, bool weighted) { return tiny_bytes(n, m, weighted) <= kTinyLds; }

hipError_t run_tiny(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* vw, float* out,
                    hipStream_t s) {
  ProfScope ps("tiny", s);
  const bool weighted = vw != nullptr;
  const size_t lds = tiny_bytes(n, m, weighted);
  const void* f = weighted ? reinterpret_cast<const void*>(k_tiny<true>) : reinterpret_cast<const void*>(k_tiny<false>);
  if (lds > 64 * 1024) {
    const hipError_t err = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTinyLds);
    if (err != hipSuccess) return err;
  }
  const int g = (int)std::min<int64_t>((m + 63) / 64, device_cu_count());
  if (weighted)
    hipLaunchKernelGGL(k_tiny<true>, dim3(g), dim3(kTinyBlock), lds, s, n, (int32_t)m, off, ind, vw, out);
  else
    hipLaunchKernelGGL(k_tiny<false>, dim3(g), dim3(kTinyBlock), lds, s, n, (int32_t)m, off, ind, vw, out);
  return hipGetLastError();
}

}  // namespace jc
