// Pair list: the intersection of two arbitrary rows per pair.
//
// The shorter row's entries are looked for in the longer row, 64 at a time.
// Rows of power-law graphs differ by orders of magnitude, and a pair drawn
// from the edges has a hub more often than not, so a workgroup takes a few
// pairs, cuts the rows into units of 128 entries and deals those to its
// waves: one wave per pair spent half its time waiting for the largest row.
// A binary search in memory costs one gather per step; the first six steps are
// taken in registers instead, over 64 evenly spaced entries of the longer row
// (one per lane, loaded once per unit), and two searches per lane are in flight
// together (four: 0.126 ms where two take 0.115).
//
// Weighted pairs need the two row sums as well. Summed anew for each pair they
// are most of the gathers (RMAT-18, 65536 pairs: 8.3e7 against 9.2e6 entries
// of shorter rows), so the caller hands over the sums of all rows where it
// has them or the list is long (launch in run_pairs); short lists sum their
// rows here, in units of 1024 entries.
//
// What bounds it then is the gathers of the search's last steps. Measured on
// RMAT of 2^18 vertices (7.6M entries), half edges and half random pairs, one
// wave per pair before: 64 pairs 48 -> 14 us unweighted, 102 -> 19 weighted;
// 1000 pairs 121 -> 18 and 191 -> 32; 65536 pairs 286 -> 115 and 568 -> 197.
#include "jc_engine.hpp"

namespace jc {

namespace {

constexpr int kPairB = 512;
constexpr int kPairNW = kPairB / kWave;
constexpr int kPairK = 2;                   // entries of the shorter row per lane and unit
constexpr int kPairUnit = kWave * kPairK;
constexpr int kSumUnit = kWave * 16;        // entries of a row sum's unit
constexpr int kPairPart = 512;              // sums of units held at a time

struct PairArgs {
  int32_t n;
  const int32_t* off;
  const int32_t* ind;
  const float* vw;
  const float* work32;
  const double* S;      // row sums, or nullptr
  int64_t np;
  int per;              // pairs of a workgroup
  const int32_t* first;
  const int32_t* second;
  float* out32;
  float* ws32;
  int accumulate;
};

// A row to look for in a longer one, or (len_l < 0) to sum.
struct PairJob {
  int o, d;        // entries [o, o + d)
  int o_l, d_l;    // the longer row
};

template <bool W>
struct PairSum;
template <>
struct PairSum<false> {
  int cnt[kWave];
};
template <>
struct PairSum<true> {
  DD part[kPairPart];
};

// Entries [r, min(r + K * 64, d)) of the job's row in its longer row: the number found
// (the same in every lane), and per lane the sum of their weights.
template <bool W, int K>
__device__ __forceinline__ int pair_unit(const PairArgs& a, const PairJob& j, int r, DD& acc) {
  const int lane = lane_id();
  const int stride = (j.d_l + kWave - 1) / kWave;
  const int32_t* row = a.ind + j.o_l;
  const int32_t piv = lane * stride < j.d_l ? row[lane * stride] : INT32_MAX;
  int32_t y[K];
  int lo[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int p = r + k * kWave + lane;
    y[k] = p < j.d ? a.ind[j.o + p] : -1;  // (no entry is negative)
    lo[k] = 0;
  }
#pragma unroll
  for (int s = kWave / 2; s > 0; s >>= 1)
#pragma unroll
    for (int k = 0; k < K; ++k) lo[k] += __shfl(piv, lo[k] + s) <= y[k] ? s : 0;
#pragma unroll
  for (int k = 0; k < K; ++k) lo[k] *= stride;  // (a lane without a pivot is never chosen)
  for (int len = stride; len > 1;) {
    const int half = len >> 1;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int at = lo[k] + half;
      lo[k] = at < j.d_l && row[at] <= y[k] ? at : lo[k];
    }
    len -= half;
  }
  int cnt = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const bool hit = row[lo[k]] == y[k];
    cnt += popc64(ballot(hit));
    if constexpr (W) {
      if (hit) acc = dd_add1(acc, (double)a.vw[y[k]]);
    }
  }
  return cnt;
}

// Weights of entries [r, min(r + kSumUnit, d)) of the job's row, per lane.
__device__ __forceinline__ DD sum_unit(const PairArgs& a, const PairJob& j, int r) {
  DD acc{0.0, 0.0};
  const int end = min(r + kSumUnit, j.d);
  for (int p = r + lane_id(); p < end; p += 4 * kWave) {
    float x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] = p + k * kWave < end ? a.vw[a.ind[j.o + p + k * kWave]] : 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) acc = dd_add1(acc, (double)x[k]);
  }
  return acc;
}

// DIRECT: the row sums are formed here. Job p of the first `per` is pair p's
// intersection, then (DIRECT) the first rows of all pairs, then the second.
template <int MODE, bool W, bool DIRECT>
__global__ __launch_bounds__(kPairB) void k_pairs(PairArgs a) {
  __shared__ PairJob job[kWave];
  __shared__ int begin[kWave + 1];  // first unit of every job
  __shared__ PairSum<W> sum;
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int jobs = a.per * (DIRECT ? 3 : 1);
  const int64_t i = (int64_t)blockIdx.x * a.per + lane % a.per;
  int32_t pa = -1, pb = -1;
  bool valid = false;
  if (wave == 0) {
    PairJob j{0, 0, 0, -1};
    int units = 0;
    if (lane < jobs && i < a.np) {
      pa = a.first[i];
      pb = a.second[i];
      valid = pa >= 0 && pa < a.n && pb >= 0 && pb < a.n;
      if (valid) {
        const int oa = a.off[pa], da = a.off[pa + 1] - oa;
        const int ob = a.off[pb], db = a.off[pb + 1] - ob;
        const int kind = lane / a.per;
        if (kind == 0) {
          const bool a_long = da > db || (da == db && pa >= pb);
          j = a_long ? PairJob{ob, db, oa, da} : PairJob{oa, da, ob, db};
          units = (j.d + kPairUnit - 1) / kPairUnit;
        } else {
          j.o = kind == 1 ? oa : ob;
          j.d = kind == 1 ? da : db;
          units = (j.d + kSumUnit - 1) / kSumUnit;
        }
      }
    }
    job[lane] = j;
    if constexpr (!W) sum.cnt[lane] = 0;
    int incl = units;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
      const int t = __shfl_up(incl, s);
      if (lane >= s) incl += t;
    }
    begin[lane + 1] = incl;
    if (lane == 0) begin[0] = 0;
  }
  __syncthreads();
  const int total = begin[kWave];
  const int mine = begin[lane];
  DD acc{0.0, 0.0};  // (weighted) of job `lane`, in wave 0
  for (int base = 0; base < total; base += W ? kPairPart : total) {
    const int stop = W ? min(base + kPairPart, total) : total;
    for (int u = base + wave; u < stop; u += kPairNW) {
      const int at = popc64(ballot(mine <= u)) - 1;
      const PairJob j = job[at];
      const int q = u - begin[at];
      DD s{0.0, 0.0};
      bool any = true;
      if (!DIRECT || j.d_l >= 0) {
        const int r = q * kPairUnit;
        const int c = j.d - r <= kWave ? pair_unit<W, 1>(a, j, r, s) : pair_unit<W, kPairK>(a, j, r, s);
        any = c != 0;
        if constexpr (!W) {
          if (lane == 0 && any) atomicAdd(&sum.cnt[at], c);
        }
      } else {
        s = sum_unit(a, j, q * kSumUnit);
      }
      if constexpr (W) {
        if (any) s = wave_sum_dd(s);
        if (lane == 0) sum.part[u - base] = s;
      }
    }
    __syncthreads();
    if constexpr (W) {
      // in the order of the row, whichever wave summed what
      if (wave == 0) {
        const int e = min(begin[lane + 1], stop);
        for (int u = max(mine, base); u < e; ++u) acc = dd_add(acc, sum.part[u - base]);
      }
      __syncthreads();
    }
  }
  if (wave != 0) return;
  double sa = 0.0, sb = 0.0;
  if constexpr (DIRECT) {
    sa = __shfl(acc.hi, min(lane + a.per, kWave - 1));
    sb = __shfl(acc.hi, min(lane + 2 * a.per, kWave - 1));
  }
  if (lane >= a.per || i >= a.np) return;
  if (!valid) {
    a.out32[i] = __int_as_float(0x7fc00000);
    if (MODE == kModeIsF32) a.ws32[i] = __int_as_float(0x7fc00000);
    return;
  }
  float cnt = 0.0f;
  if constexpr (!W) cnt = (float)(uint32_t)sum.cnt[lane];
  if constexpr (MODE == kModeEcU) {
    const int da = a.off[pa + 1] - a.off[pa], db = a.off[pb + 1] - a.off[pb];
    a.out32[i] = cnt / ((float)(da + db) - cnt);
  } else if constexpr (MODE == kModeEcW) {
    if constexpr (!DIRECT) {
      sa = a.S[pa];
      sb = a.S[pb];
    }
    a.out32[i] = (float)(acc.hi / ((sa + sb) - acc.hi));
  } else {
    a.out32[i] = (a.accumulate ? a.out32[i] : 0.0f) + (W ? (float)acc.hi : cnt);
    a.ws32[i] = a.work32[pa] + a.work32[pb];
  }
}

}  // namespace

hipError_t run_pairs(int mode, bool weighted, int32_t n, const int32_t* off, const int32_t* ind,
                     const float* vw, const float* work32, const double* S, int64_t np, const int32_t* first,
                     const int32_t* second, float* out32, float* ws32, int accumulate,
                     hipStream_t stream) {
  if (np <= 0) return hipSuccess;
  if (mode != kModeIsF32 && mode != (weighted ? kModeEcW : kModeEcU)) return hipErrorInvalidValue;
  const bool direct = mode == kModeEcW && !S;
  // as few pairs per workgroup as keep a few thousand workgroups: the rows'
  // lengths even out over the CUs, and a lone hub pair has eight waves
  const int per = (int)std::min<int64_t>(std::max<int64_t>(np / ((int64_t)device_cu_count() * 16), 1),
                                         direct ? kWave / 3 : kWave);
  const PairArgs a{n, off, ind, vw, work32, S, np, per, first, second, out32, ws32, accumulate};
  const dim3 g((unsigned)((np + per - 1) / per)), b(kPairB);
  ProfScope ps("pairs", stream);
  if (mode == kModeEcU) hipLaunchKernelGGL((k_pairs<kModeEcU, false, false>), g, b, 0, stream, a);
  else if (direct) hipLaunchKernelGGL((k_pairs<kModeEcW, true, true>), g, b, 0, stream, a);
  else if (mode == kModeEcW) hipLaunchKernelGGL((k_pairs<kModeEcW, true, false>), g, b, 0, stream, a);
  else if (weighted) hipLaunchKernelGGL((k_pairs<kModeIsF32, true, false>), g, b, 0, stream, a);
  else hipLaunchKernelGGL((k_pairs<kModeIsF32, false, false>), g, b, 0, stream, a);
  return hipGetLastError();
}

}  // namespace jc
