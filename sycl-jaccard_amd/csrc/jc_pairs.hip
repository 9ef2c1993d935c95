// Pair list: the intersection of two arbitrary rows per pair.
//
// The shorter row's entries are looked for in the longer row, 64 at a time. Pairs of
// rows of up to kPairShort entries are a wave's each. Rows of power-law graphs
// differ by orders of magnitude, and a pair drawn from the edges has a hub more
// often than not, so a workgroup lists its other pairs, cuts their rows into units
// of 128 entries and deals those to its waves: with one wave per pair half the
// time went by waiting for the largest row. (With units alone, pairs of short rows
// waited for each other: 16384 weighted pairs of uniform rows 31 us where a
// wave each takes 14.)
// A binary search in memory costs one gather per step; the first six steps are
// taken in registers instead, over 64 evenly spaced entries of the longer row
// (one per lane, loaded once per pair or unit), and two searches per lane are in flight
// together (four: 0.126 ms where two take 0.115).
//
// Weighted pairs need the two row sums as well. Summed anew for each pair they
// are most of the gathers where pairs name hubs (RMAT-18, 65536 pairs: 8.3e7
// against 9.2e6 entries of shorter rows), so the caller hands over the sums of all
// rows where that is less work; else the rows are summed here, in units of 1024
// entries.
//
// What bounds it then is the gathers of the search's last steps. Measured in us on
// RMAT of 2^18 vertices (7.6M entries), half edges and half random pairs, one
// wave per pair before: 1000 pairs 48 -> 11 unweighted, 109 -> 24 weighted; 65536
// pairs 461 -> 111 and 763 -> 211; uniform random, 20 to 100 entries a row, 65536
// random pairs 24 to 53 -> 16 to 29 and 59 to 92 -> 34 to 48.
#include "jc_engine.hpp"

namespace jc {

namespace {

constexpr int kPairB = 512;
constexpr int kPairNW = kPairB / kWave;
constexpr int kPairK = 2;                   // entries of the shorter row per lane and unit
constexpr int kPairUnit = kWave * kPairK;
constexpr int kSumUnit = kWave * 16;        // entries of a row sum's unit
constexpr int kPairPart = 512;              // sums of units held at a time
constexpr int kPairShort = 512;             // pairs of rows up to this by one wave
static_assert(kPairShort <= kSumUnit, "one step");

struct PairArgs {
  int32_t n;
  const int32_t* off;
  const int32_t* ind;
  const float* vw;
  const float* work32;
  const double* S;      // row sums, or nullptr
  const int* no_S;      // (device) not 0: they were not formed after all; or nullptr
  int64_t np;
  int per;              // pairs of a workgroup
  const int32_t* first;
  const int32_t* second;
  float* out32;
  float* ws32;
  int accumulate;
};

// A row to look for in a longer one, or (d_l < 0) to sum.
struct PairJob {
  int o, d;        // entries [o, o + d)
  int o_l, d_l;    // the longer row
};

// A pair that is cut into units: its place in the workgroup, ids, rows.
struct PairLong {
  int q;
  int32_t pa, pb;
  int oa, da, ob, db;
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

// What a wave keeps of a longer row: 64 evenly spaced entries, one per lane.
struct PairRow {
  const int32_t* row;
  int d, stride;
  int32_t piv, last;
  __device__ __forceinline__ PairRow(const PairArgs& a, const PairJob& j) : row(a.ind + j.o_l), d(j.d_l) {
    stride = (d + kWave - 1) / kWave;
    piv = lane_id() * stride < d ? row[lane_id() * stride] : INT32_MAX;
    last = stride == 1 ? __builtin_amdgcn_readlane(piv, d - 1) : row[d - 1];
  }
};

// Entries [r, min(r + K * 64, d)) of the job's row in its longer row: the number found
// (the same in every lane), and per lane the sum of their weights.
template <bool W, int K>
__device__ __forceinline__ int pair_unit(const PairArgs& a, const PairJob& j, const PairRow& l, int r, DD& acc) {
  const int lane = lane_id();
  int32_t y[K];
  int lo[K];
  bool near = false;
  const int32_t begin = __builtin_amdgcn_readfirstlane(l.piv);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int p = r + k * kWave + lane;
    y[k] = p < j.d ? a.ind[j.o + p] : -1;  // (no entry is negative)
    near |= y[k] >= begin && y[k] <= l.last;
    lo[k] = 0;
  }
  if (!ballot(near)) return 0;  // most pairs of vertices that are far apart
#pragma unroll
  for (int s = kWave / 2; s > 0; s >>= 1)
#pragma unroll
    for (int k = 0; k < K; ++k) lo[k] += __shfl(l.piv, lo[k] + s) <= y[k] ? s : 0;
  bool hit[K];
  if (l.stride == 1) {
#pragma unroll
    for (int k = 0; k < K; ++k) hit[k] = __shfl(l.piv, lo[k]) == y[k];
  } else {
#pragma unroll
    for (int k = 0; k < K; ++k) lo[k] *= l.stride;  // (a lane without a pivot is never chosen)
    for (int len = l.stride; len > 1;) {
      const int half = len >> 1;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int at = lo[k] + half;
        lo[k] = at < l.d && l.row[at] <= y[k] ? at : lo[k];
      }
      len -= half;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) hit[k] = l.row[lo[k]] == y[k];
  }
  int cnt = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    cnt += popc64(ballot(hit[k]));
    if constexpr (W) {
      if (hit[k]) acc = dd_add1(acc, (double)a.vw[y[k]]);
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

// The result of pair i = (pa, pb), by one lane. sa, sb: the row sums (kModeEcW).
template <int MODE, bool W>
__device__ __forceinline__ void put_pair(const PairArgs& a, int64_t i, int32_t pa, int32_t pb, int da, int db,
                                         uint32_t cnt, double sum, double sa, double sb) {
  const float fI = (float)cnt;
  if constexpr (MODE == kModeEcU) {
    a.out32[i] = fI / ((float)(da + db) - fI);
  } else if constexpr (MODE == kModeEcW) {
    a.out32[i] = (float)(sum / ((sa + sb) - sum));
  } else {
    a.out32[i] = (a.accumulate ? a.out32[i] : 0.0f) + (W ? (float)sum : fI);
    a.ws32[i] = a.work32[pa] + a.work32[pb];
  }
}

// DIRECT: the row sums are formed here, unless S has them. Pairs of short rows first, one wave
// each; the others are listed. Of those, job p of the first nl is pair p's
// intersection, then (DIRECT) come the first rows of all, then the second.
template <int MODE, bool W, bool DIRECT>
__global__ __launch_bounds__(kPairB) void k_pairs(PairArgs a) {
  constexpr int kList = DIRECT ? kWave / 3 : kWave;
  __shared__ PairJob job[kWave];
  __shared__ int begin[kWave + 1];  // first unit of every job
  __shared__ PairSum<W> sum;
  __shared__ PairLong s_long[kList];
  __shared__ int s_nl;
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t base_i = (int64_t)blockIdx.x * a.per;
  const bool sums = DIRECT && (!a.no_S || *a.no_S != 0);
  if (threadIdx.x == 0) s_nl = 0;
  {
    // a wave's pairs, one per lane up to here
    const int chunk = (a.per + kPairNW - 1) / kPairNW;
    const int64_t i = base_i + wave * chunk + lane;
    const bool live = lane < chunk && wave * chunk + lane < a.per && i < a.np;
    int32_t pa = -1, pb = -1;
    int oa = 0, da = 0, ob = 0, db = 0;
    if (live) {
      pa = a.first[i];
      pb = a.second[i];
    }
    const bool valid = pa >= 0 && pa < a.n && pb >= 0 && pb < a.n;
    if (valid) {
      oa = a.off[pa];
      da = a.off[pa + 1] - oa;
      ob = a.off[pb];
      db = a.off[pb + 1] - ob;
    }
    __syncthreads();  // s_nl is 0
    const bool single = max(da, db) <= kPairShort || (!sums && min(da, db) <= kPairUnit);
    if (valid && !single) s_long[atomicAdd(&s_nl, 1)] = PairLong{wave * chunk + lane, pa, pb, oa, da, ob, db};
    uint32_t cnt = 0;
    double sum = 0.0, sa = 0.0, sb = 0.0;
    for (uint64_t todo = ballot(valid && single); todo; todo &= todo - 1) {
      const int q = __ffsll((unsigned long long)todo) - 1;
      const int qoa = __builtin_amdgcn_readlane(oa, q), qda = __builtin_amdgcn_readlane(da, q);
      const int qob = __builtin_amdgcn_readlane(ob, q), qdb = __builtin_amdgcn_readlane(db, q);
      const PairJob j = qda > qdb ? PairJob{qob, qdb, qoa, qda} : PairJob{qoa, qda, qob, qdb};
      int c = 0;
      DD acc{0.0, 0.0};
      if (j.d > 0) {
        const PairRow l(a, j);
        int r = 0;
        for (; j.d - r > kWave; r += kPairUnit) c += pair_unit<W, kPairK>(a, j, l, r, acc);
        if (r < j.d) c += pair_unit<W, 1>(a, j, l, r, acc);
      }
      if constexpr (W) {
        if (c > 0) acc = wave_sum_dd(acc);
      }
      DD xa{0.0, 0.0}, xb{0.0, 0.0};
      if (sums) {
        xa = sum_unit(a, PairJob{qoa, qda, 0, -1}, 0);
        xb = sum_unit(a, PairJob{qob, qdb, 0, -1}, 0);
        xa = wave_sum_dd(xa);
        xb = wave_sum_dd(xb);
      }
      if (lane == q) {
        cnt = (uint32_t)c;
        sum = acc.hi;
        sa = xa.hi;
        sb = xb.hi;
      }
    }
    if (valid && single) {
      if (MODE == kModeEcW && !sums) {
        sa = a.S[pa];
        sb = a.S[pb];
      }
      put_pair<MODE, W>(a, i, pa, pb, da, db, cnt, sum, sa, sb);
    } else if (live && !valid) {
      a.out32[i] = __int_as_float(0x7fc00000);
      if (MODE == kModeIsF32) a.ws32[i] = __int_as_float(0x7fc00000);
    }
  }
  __syncthreads();
  const int nl = s_nl;
  if (nl == 0) return;
  const int jobs = nl * (sums ? 3 : 1);
  int32_t pa = 0, pb = 0;
  int da = 0, db = 0;
  int64_t i = 0;
  if (wave == 0) {
    PairJob j{0, 0, 0, -1};
    int units = 0;
    if (lane < jobs) {
      const PairLong l = s_long[lane % nl];
      i = base_i + l.q;
      pa = l.pa;
      pb = l.pb;
      da = l.da;
      db = l.db;
      const int oa = l.oa, ob = l.ob;
      const int kind = lane / nl;
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
        const PairRow l(a, j);
        const int c = j.d - r <= kWave ? pair_unit<W, 1>(a, j, l, r, s) : pair_unit<W, kPairK>(a, j, l, r, s);
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
  if (sums) {
    sa = __shfl(acc.hi, min(lane + nl, kWave - 1));
    sb = __shfl(acc.hi, min(lane + 2 * nl, kWave - 1));
  }
  if (lane >= nl) return;
  if (MODE == kModeEcW && !sums) {
    sa = a.S[pa];
    sb = a.S[pb];
  }
  uint32_t cnt = 0;
  if constexpr (!W) cnt = (uint32_t)sum.cnt[lane];
  put_pair<MODE, W>(a, i, pa, pb, da, db, cnt, acc.hi, sa, sb);
}

// *no_S = 1 where the rows of the pairs, by a sample, have less than 1.5 times the
// entries of the graph: summed for each pair they are then the smaller work (a ring
// with 96 a row, at 1.3 times 95 us for each pair and 121 of all; uniform random
// rows of 100 at 6.6 times 64 and 48).
__global__ __launch_bounds__(1024) void k_pairs_want(PairArgs a, int64_t m, int* no_S) {
  __shared__ unsigned long long s_sum;
  if (threadIdx.x == 0) s_sum = 0ull;
  __syncthreads();
  const int64_t i = (int64_t)threadIdx.x * a.np / 1024;
  const int32_t pa = a.first[i], pb = a.second[i];
  long long d = 0;
  if (pa >= 0 && pa < a.n && pb >= 0 && pb < a.n) d = (long long)(a.off[pa + 1] - a.off[pa]) + (a.off[pb + 1] - a.off[pb]);
#pragma unroll
  for (int t = 1; t < kWave; t <<= 1) d += __shfl_xor(d, t);
  if (lane_id() == 0) atomicAdd(&s_sum, (unsigned long long)d);
  __syncthreads();
  if (threadIdx.x == 0) *no_S = (double)s_sum / 1024.0 * (double)a.np < 1.5 * (double)m;
}

}  // namespace

hipError_t launch_pairs_want(int32_t n, int64_t m, const int32_t* off, int64_t np, const int32_t* first,
                             const int32_t* second, int* no_S, hipStream_t stream) {
  PairArgs a{};
  a.n = n;
  a.off = off;
  a.np = np;
  a.first = first;
  a.second = second;
  hipLaunchKernelGGL(k_pairs_want, dim3(1), dim3(1024), 0, stream, a, m, no_S);
  return hipGetLastError();
}

hipError_t run_pairs(int mode, bool weighted, int32_t n, const int32_t* off, const int32_t* ind,
                     const float* vw, const float* work32, const double* S, int64_t np, const int32_t* first,
                     const int32_t* second, float* out32, float* ws32, int accumulate,
                     hipStream_t stream, const int* no_S) {
  if (np <= 0) return hipSuccess;
  if (mode != kModeIsF32 && mode != (weighted ? kModeEcW : kModeEcU)) return hipErrorInvalidValue;
  const bool direct = mode == kModeEcW && (!S || no_S);
  // a pair per wave; fewer for short lists, so that there is a workgroup for every
  // CU and a lone hub pair has eight waves, more for very long ones
  const int64_t cus = device_cu_count();
  const int per = (int)std::min<int64_t>(
      std::max({np / (cus * 16), std::min<int64_t>(np / cus, kPairNW), int64_t(1)}), direct ? kWave / 3 : kWave);
  const PairArgs a{n, off, ind, vw, work32, S, no_S, np, per, first, second, out32, ws32, accumulate};
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
