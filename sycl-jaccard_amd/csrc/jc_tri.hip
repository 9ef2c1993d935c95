// Oriented engine: every intersection of a symmetric graph from its triangles.
//
// The owner engine (jc_engine.hpp) streams, for each pair {u, x}, the whole
// shorter row: sum over pairs of min(d_u, d_x) entries (4.3e10 on RMAT-22).
// I(u, v) is also the weight of the triangles over the edge {u, v}, and one
// triangle serves three edges. Ranking the vertices by degree (rank 0 the
// largest) and keeping of each row only the neighbours of lower rank,
// R(u), leaves rows of at most sqrt(2m) entries, and every triangle
// {w < v < u by rank} once: v, w in R(u), w in R(v). That is
// sum |R(u)|^2 / 2 tests (7.2e9 on RMAT-22, a sixth), each against a bitmap
// over the ranks below v, which for the vertices that matter is a few KiB.
//
//   rank     degree-bucket counting sort of the vertices
//            (a batch of small graphs, EngineArgs::members: the disjoint parts
//            are found from the reach of the rows, and each is ranked by
//            itself, so that its 16-bit ranks start at its own first)
//   orient   per row: R(u) sorted by rank (32-bit and, saturated, 16-bit
//            copies, at the row's own offset), the row sum of the weights,
//            and emap[k], the oriented slot of a stored entry (u, v in R(u))
//   plan     places in the bit matrix, task lists
//   wedge    per v: the bitmap of R(v) in LDS; for every u with v in R(u) (the
//            entries of v's own row that are not in R(v); the position p of v
//            in R(u) by binary search, which also fills emap for the entry
//            and proves the entry has its mirror) the p entries before v are
//            tested. Hits go two ways: into the LDS sum of the pair (v, w),
//            weight W[u], and as one bit each into row p of u's bit matrix
//   reduce   per u: the symmetric bit matrix M over R(u) times the weights
//            gives the parts of the pairs (u, v) that have the third vertex
//            in R(u); with the LDS sums of wedge that is the whole
//            intersection, and the quotient is formed
//   deliver  result[k] = value[emap[k]]
//
// No part depends on the order of the sums: counts are integers, and weights
// are added in fp64 only when ExactInfo shows that every sum is exact. What
// the engine cannot do it refuses before anything is written to the result
// (refuse): a graph that is not symmetric, has self loops or rows out of
// order, weights
// whose fp64 sums may round, a bit matrix larger than its budget, an |R(u)|
// above kTriMaxOut. The owner engine, launched after it, then runs; when the
// oriented engine has delivered, the owner engine's kernels return at once.
//
// Measured against the owner engine (whole calls): RMAT-22 weighted 58.2 ->
// 15.9 ms, RMAT of 200003 vertices weighted vertex-centric 1.58 -> 0.72 ms,
// Chung-Lu 2^20 4.00 -> 2.86 ms.
#include <stddef.h>

#include <type_traits>

#include "jc_device.hpp"
#include "jc_hash.hpp"
#include "jc_internal.hpp"
#include "jc_profile.hpp"

namespace jc {

namespace {

constexpr int kTriBuckets = 1024;
constexpr int kSamples = 1024;     // entries looked at before the engine is chosen
constexpr int kSampleCap = 512;
constexpr int kTriParts = 1024;    // vertex ranges of the rank kernels, at most
constexpr int kPartMax = kTriPart; // vertices of a disjoint part
constexpr int kTriMaxOut = 4096;   // largest |R(u)|: the sort and reduce buffers in LDS
constexpr int kTriRowWave = 1024;  // rows up to this many entries are oriented by one wave
constexpr int kSat16 = 65535;      // 16-bit ranks saturate here
constexpr int kPivotMin = 16;      // rows up to this are searched whole
constexpr int kWgMinDeg = 192;     // rows of at least this many entries get a workgroup in wedge
constexpr int kWedgeB = 512;       // threads of a wedge workgroup, entries of a wedge task
constexpr int kGroupMax = 512;     // shorter rows are taken several to a workgroup
constexpr int kGroupRows = 64;     // at most that many
constexpr int kTabA = 2048;        // bitmap words of the 16-bit wedge kernel (65536 ranks)
constexpr int kAccA = 1408;        // largest |R(v)| of the 16-bit wedge kernel
constexpr int kTabB = 8192;        // the same for the 32-bit wedge kernel (262144 ranks)
constexpr int kAccB = kTriMaxOut;
constexpr int kWaveTab = 256;      // largest |R(v)| hashed in LDS by the one-wave wedge kernel
constexpr int kRedWave = 256;      // |R(u)| that reduce takes by one wave
constexpr int kRedWg = 1280;       // by a workgroup with that many weights in LDS; above, kTriMaxOut

// Monotone in the degree: exact below 512, 16 steps per octave above.
__device__ __forceinline__ int deg_bucket(int d) {
  if (d < 512) return d;
  const int e = 31 - __clz(d);  // >= 9
  return 512 + (e - 9) * 16 + ((d >> (e - 4)) & 15);
}

// Words of the bit matrix rows of 0 .. L-1 columns: sum of ceil(l / 32).
__device__ __forceinline__ uint32_t tri_words(int L) {
  const uint32_t t = (uint32_t)max(L - 1, 0), k = t >> 5;
  return (k + 1u) * (t - 16u * k);
}

// Row u of the 16-bit ranks, in units of 16 bytes: a header of two units, then
// the entries, eight to a unit, and at least eight more, which hold kSat16 (no
// bitmap has that bit), so a group of eight may be read past the end. The
// header is what wedge needs of u: row offset, |R(u)|, first word of its bit
// matrix, weight bits; then the ranks at |R| k / 8, k = 1 .. 7, for the search.
// An entry that leads to u carries the header's place (emap). Rows start on
// 128-byte lines, the unit of what the cache fetches: wedge is bound by the
// lines it touches (RMAT-22: 34.5 GB at 5.5 TB/s with rows on 16 bytes).
__host__ __device__ __forceinline__ uint64_t row16_line(uint64_t o, uint64_t u) { return ((o + 24 * u) >> 6) + u; }
__device__ __forceinline__ uint32_t row16(int o, int32_t u) { return 8u * (uint32_t)row16_line((uint64_t)o, (uint64_t)u); }
constexpr int kHead = 2;
// In place of row16 where a row is empty: such a row gets no header, so no
// entry may lead to one. In a symmetric graph none does; orient refuses the
// graph at the first that would.
constexpr int kNoRow = -1;

// A task of the bitmap wedge kernels.
struct __attribute__((aligned(32))) TriTask {
  int32_t r, o, d, dp;  // v: rank (16-bit kernel: in its part), row offset, row entries, |R(v)|
  int32_t piece;        // entries [piece * kWedgeB, ...) of v's row
  int32_t row;          // row16 of v
  int32_t pad[2];
};

}  // namespace

// A counter on a cache line of its own. Atomics on a line and reads of it wait
// for each other, over the XCDs some 40 ns each: with the counters side by side
// reduce by workgroup took 2.31 ms on RMAT-22, and 0.92 without.
template <typename T>
struct alignas(256) Own {
  T v;
};

// Why the engine may refuse a graph is found out in stages, each with a
// word of its own: a kernel reads the words of the stages before its own, which
// no kernel in flight writes, and writes only its own stage's. So all waves of a
// workgroup see the same and end together or not at all; with one word for all,
// waves that found it set while the launch was under way left the others at
// barriers and on LDS that nobody had filled.
enum TriStage { kStLook, kStCount, kStRank, kStOrient, kStWedge, kStReduce };

struct TriCtl {
  int pad;
  int done;
  int bad[kStReduce];
  Own<int> lsb, maxexp;             // exactness of the weights (see ExactInfo)
  Own<int> wexp;                    // every weight is below 2^wexp
  Own<double> sampled_w;            // weights of the sampled entries' vertices
  Own<unsigned long long> out_total;  // sum of |R(u)|
  Own<unsigned long long> bits;     // words of the bit matrix handed out
  Own<int> num_big;                 // rows oriented by a workgroup
  Own<int> num_mid;                 // rows oriented by a wave
  Own<int> num_task[2];             // wedge tasks: 16-bit, 32-bit
  Own<int> num_wave, num_s16, num_s64;
  Own<int> num_red[2];              // reduce by workgroup: up to kRedWg entries, more
  Own<int> num_part;                // disjoint parts (members)
  Own<int> num_group;               // group tasks of wedge: rows of fewer than kGroupMax entries
  // taken off the lists, beyond what every workgroup takes without asking
  Own<int> cur_big, cur_task[2], cur_red[2], cur_part, cur_group;
  int grp_task[kGroupMax];       // first task of the rows of each length
  int grp_rank[kGroupMax];       // first rank among them that is taken in groups
  int hist[kTriBuckets];
  int cur[kTriBuckets];
  int reach[kTriParts], nstart[kTriParts];  // per vertex range: largest neighbour id (then of all ranges before), parts begun
};
// (where the tests look to see what ran)
static_assert(offsetof(TriCtl, done) == 4 && offsetof(TriCtl, num_task) == 9 * 256 &&
                  offsetof(TriCtl, num_wave) == 11 * 256 && offsetof(TriCtl, num_red) == 14 * 256,
              "places of the counters");

namespace {

struct TriArgs {
  int32_t n;
  int64_t m;
  const int32_t* off;
  const int32_t* ind;
  const float* vw;
  TriCtl* ctl;
  int4* rw;         // per vertex: rank, weight bits, place of its 16-bit row (kNoRow: it has no entries), first rank of its part
  int32_t* vtx;     // per rank: vertex
  float* wr;        // per rank: weight
  double* sr;       // per rank: row sum of the weights (unweighted: unused)
  int32_t* dr;      // per rank: degree
  int32_t* ord;     // vertices and their degrees by descending degree bucket: vtx
  int32_t* dord;    // and dr, but for disjoint parts, whose ranks are in id order
  int always;       // whatever the rows' lengths
  int members;      // rank disjoint parts by themselves
  int32_t grp_from; // place in ord from which longer rows than kWgMinDeg are taken in groups too
  int32_t* starts;  // first vertices of the parts: per vertex range, then
  int32_t* parts;   // all of them
  int4* info;       // per vertex: row offset, |R|, first word of its bit matrix, rank
  int4* rinfo;      // per place in ord: row offset, |R|, rank, first rank of the part
  uint32_t* R32;    // R(u) at [off[u], off[u] + |R(u)|), later the pairs' values
  uint16_t* R16;    // the same, saturated, at row16 with headers
  int32_t* emap;    // per stored entry (u, x): its slot, or until wedge ~row16 of x if x ranks after u
  double* accw;     // per slot: sums of wedge (weighted)
  uint32_t* accu;   // (unweighted)
  uint32_t* bits;
  uint64_t bits_cap;
  int32_t* list_mid;  // vertices by class; ends of one array (orient), then reused
  int32_t* list_big;
  TriTask* task[2];
  int64_t task_cap;
  int32_t* list_wave;  // places in ord
  int32_t* list_s16;   // vertices with |R| in 1..16
  int32_t* list_s64;   // up to kRedWave
  int32_t* list_red[2];  // up to kRedWg, more
  // delivery
  int mode;
  const float* work32;
  float* out32;
  float* ws32;
  int accumulate;
};

// By a kernel of stage S: not this graph.
template <int S>
__device__ __forceinline__ void refuse(const TriArgs& a) {
  static_assert(S < kStReduce, "reduce refuses nothing");
  a.ctl->bad[S] = 1;
}

// Whether the stages before S left the graph to S.
template <int S>
__device__ __forceinline__ bool tri_go(const TriArgs& a) {
  int bad = 0;
#pragma unroll
  for (int i = 0; i < S; ++i) bad |= a.ctl->bad[i];
  return bad == 0;
}

// The same from wedge on, with the facts that must hold before it starts.
template <bool W, int S>
__device__ __forceinline__ bool tri_ready(const TriArgs& a) {
  static_assert(S >= kStWedge, "plan counts what this looks at");
  const TriCtl* c = a.ctl;
  if (!tri_go<S>(a) || 2ull * c->out_total.v != (unsigned long long)a.m || c->bits.v > a.bits_cap) return false;
  if constexpr (W) return exact_sums_fit_f64(ExactInfo{c->lsb.v, c->maxexp.v, 0, 0});
  return true;
}

// An entry (x, y) of the graph, the t-th of kSamples spread over it; false for x
// without entries (in a graph that is not symmetric). A neighbour's neighbour is as
// random an entry as any in a symmetric graph, and needs no search for its row.
__device__ __forceinline__ bool sample_entry(const TriArgs& a, int t, int32_t& x, int32_t& y, int& dx) {
  // one in each of kSamples equal runs of entries
  const int64_t k = min(a.m - 1, (t * a.m + (int64_t)((t * 0x9E3779B1u) >> 22) * a.m / 1024) / kSamples);
  x = a.ind[k];
  const int o = a.off[x];
  dx = a.off[x + 1] - o;
  if (dx <= 0) return false;
  y = a.ind[o + (int)((uint32_t)t * 0x85EBCA6Bu % (uint32_t)dx)];
  return true;
}

// Clears the control words and, before anything else is done for the graph, looks
// whether the engine would be the faster one. With len the mean of min(d_x, d_y, 512) over
// sampled entries and d the mean degree, it is where len is well above d (few hubs on
// most edges), or rows are long in any case. Owner / oriented engine, ms,
// weighted: RMAT len 85..230, d 6..54: 1.3 to 2.2 times as fast; Chung-Lu len
// 53..206, d 6..64: 1.4 to 2.2 times; uniform random graphs d = len = 16 1.44
// / 1.99, 37 0.99 / 1.39, 63 0.99 / 1.21, 76 1.77 / 1.78, 154 3.88 / 2.06;
// neighbours on a ring 24 1.56 / 2.50, 72 3.68 / 3.54, 196 3.62 / 2.15. A graph that
// is turned down here costs the launches that then do nothing, 25 to 50 us (uniform
// random, 4M entries weighted 422 us without the engine, 445 with; 576 when the degrees
// were counted and ranked first).
__global__ __launch_bounds__(kSamples) void k_tri_init(TriArgs a) {
  __shared__ int s_len[kSamples / kWave];
  int* p = reinterpret_cast<int*>(a.ctl);
  for (int i = threadIdx.x; i < (int)(sizeof(TriCtl) / sizeof(int)); i += kSamples) p[i] = 0;
  int len = 0;
  if (!a.always) {
    int32_t x, y;
    int dx;
    if (sample_entry(a, threadIdx.x, x, y, dx)) len = min(min(dx, a.off[y + 1] - a.off[y]), kSampleCap);
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) len += __shfl_xor(len, o);
    if (lane_id() == 0) s_len[threadIdx.x / kWave] = len;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    a.ctl->lsb.v = INT32_MAX;
    a.ctl->maxexp.v = INT32_MIN;
    a.ctl->wexp.v = INT32_MIN;
    if (!a.always) {
      int sum = 0;
      for (int i = 0; i < kSamples / kWave; ++i) sum += s_len[i];
      const float l = (float)sum / kSamples, d = (float)a.m / (float)a.n;
      if (l < 48.f || (l < 96.f && l < 1.5f * d)) refuse<kStLook>(a);
    }
  }
}

// Degree histogram over each workgroup's contiguous range of vertices, and
// the finest and the highest bit of the weights. The first kSamples / BLOCK
// workgroups look at one entry per thread instead, for its mirror, so
// that most graphs that are not symmetric are refused before the work of
// orient.
template <bool W, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_hist(TriArgs a) {
  __shared__ int h[kTriBuckets];
  constexpr int kLook = kSamples / BLOCK;
  if (!tri_go<kStCount>(a)) return;
  if (blockIdx.x < kLook) {
    int32_t x = 0, y = 0;
    int dx;
    const bool any = sample_entry(a, blockIdx.x * BLOCK + threadIdx.x, x, y, dx);
    if (any) {
      const int e = a.off[y + 1], at = lane_lower_bound(a.ind, a.off[y], e, x);
      if (at >= e || a.ind[at] != x) refuse<kStCount>(a);
    } else {
      refuse<kStCount>(a);
    }
    if constexpr (W) {
      float w = any ? a.vw[y] : 0.0f;
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) w += __shfl_xor(w, o);
      if (lane_id() == 0) unsafeAtomicAdd(&a.ctl->sampled_w.v, (double)w);
    }
    return;
  }
  const int ranges = gridDim.x - kLook, range = blockIdx.x - kLook;
  for (int i = threadIdx.x; i < kTriBuckets; i += BLOCK) h[i] = 0;
  __syncthreads();
  const int64_t per = ((int64_t)a.n + ranges - 1) / ranges;
  const int32_t r0 = (int32_t)min(per * range, (int64_t)a.n), r1 = (int32_t)min(per * (range + 1), (int64_t)a.n);
  int lsb = INT32_MAX, top = INT32_MIN;
  bool bad = false;
  for (int32_t u = r0 + threadIdx.x; u < r1; u += BLOCK) {
    const int d = a.off[u + 1] - a.off[u];
    atomicAdd(&h[deg_bucket(d)], 1);
    if constexpr (W) {
      const uint32_t b = __float_as_uint(a.vw[u]);
      const uint32_t ex = (b >> 23) & 0xFFu, man = b & 0x7FFFFFu;
      if (((b >> 31) && (b << 1)) || ex == 0xFFu) bad = true;  // negative or not finite (-0 is harmless)
      else if (ex != 0 || man != 0) {
        lsb = min(lsb, (ex ? (int)ex - 150 : -149) + (int)__builtin_ctz(ex ? (man | 0x800000u) : man));
        top = max(top, max((int)ex, 1) - 126);
      }
    }
  }
  if constexpr (W) {
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      lsb = min(lsb, __shfl_xor(lsb, o));
      top = max(top, __shfl_xor(top, o));
    }
    if (ballot(bad) && lane_id() == 0) refuse<kStCount>(a);
    if (lane_id() == 0 && lsb < *(volatile int*)&a.ctl->lsb.v) atomicMin(&a.ctl->lsb.v, lsb);
    if (lane_id() == 0 && top > *(volatile int*)&a.ctl->wexp.v) atomicMax(&a.ctl->wexp.v, top);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kTriBuckets; i += BLOCK)
    if (h[i]) atomicAdd(&a.ctl->hist[i], h[i]);
}

// Vertices of degree d in a group task of wedge.
__device__ __forceinline__ int group_rows(int d) { return min(kGroupRows, kWedgeB / d); }

// First rank of every bucket, largest degrees first; and whether the weights'
// sums may be exact.
__global__ __launch_bounds__(kTriBuckets) void k_tri_scan(TriArgs a) {
  __shared__ int part[kTriBuckets / kWave];
  __shared__ int s_top;
  if (!tri_go<kStCount>(a)) return;
  TriCtl* const c = a.ctl;
  const int b = kTriBuckets - 1 - threadIdx.x;
  if (b == 0) s_top = 0;
  __syncthreads();
  if (c->hist[b]) atomicMax(&s_top, b);
  __syncthreads();
  // a weight that alone is wider than fp64 sums can hold
  if (b == 0 && c->lsb.v != INT32_MAX && c->wexp.v - c->lsb.v > 53) refuse<kStCount>(a);
  if (b == 0 && !a.always) {
    // the longest row's weights, were they the sampled ones' mean: sums that
    // surely round are not found out after orient only
    const int top = s_top < 512 ? s_top : (16 + (s_top & 15)) << ((s_top - 512) / 16 + 5);
    const double sum = (double)top * c->sampled_w.v / kSamples;
    if (c->lsb.v != INT32_MAX && sum > 0.0 && !isinf(sum) && ilogb(sum) - c->lsb.v > 53) refuse<kStCount>(a);
  }
  const int v = c->hist[b];
  int incl = v;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int t = __shfl_up(incl, o);
    if (lane_id() >= o) incl += t;
  }
  if (lane_id() == kWave - 1) part[threadIdx.x / kWave] = incl;
  __syncthreads();
  int base = 0;
  for (int i = 0; i < (int)threadIdx.x / kWave; ++i) base += part[i];
  c->cur[b] = base + incl - v;
  // Group tasks of wedge. Buckets below kGroupMax hold one degree each, so a
  // group is group_rows(b) vertices of consecutive ranks and equal degree;
  // long rows of low rank go to the bitmap kernel instead.
  int ng = 0;
  if (b > 0 && b < kGroupMax) {
    const int first = b >= kWgMinDeg ? max(base + incl - v, a.grp_from) : base + incl - v;
    const int cnt = max(0, base + incl - first);
    c->grp_rank[b] = first;
    ng = (cnt + group_rows(b) - 1) / group_rows(b);
  }
  int gi = ng;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int t = __shfl_up(gi, o);
    if (lane_id() >= o) gi += t;
  }
  __syncthreads();
  if (lane_id() == kWave - 1) part[threadIdx.x / kWave] = gi;
  __syncthreads();
  int gbase = 0;
  for (int i = 0; i < (int)threadIdx.x / kWave; ++i) gbase += part[i];
  if (b < kGroupMax) c->grp_task[b] = gbase + gi - ng;
  if (b == 0) c->num_group.v = gbase + gi;
}

// Ranks: each workgroup counts its range per bucket, reserves the places with
// one atomic per bucket, then assigns. Also the rank-ordered copies, and the
// lists of the rows that orient takes by wave and by workgroup.
template <bool W, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_rank(TriArgs a) {
  __shared__ int h[kTriBuckets];
  __shared__ int base[kTriBuckets];
  __shared__ int s_cnt[2], s_base[2];
  if (!tri_go<kStRank>(a)) return;
  for (int i = threadIdx.x; i < kTriBuckets; i += BLOCK) h[i] = 0;
  if (threadIdx.x < 2) s_cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t per = ((int64_t)a.n + gridDim.x - 1) / gridDim.x;
  const int32_t r0 = (int32_t)min(per * blockIdx.x, (int64_t)a.n), r1 = (int32_t)min(per * (blockIdx.x + 1), (int64_t)a.n);
  for (int32_t u = r0 + threadIdx.x; u < r1; u += BLOCK) {
    const int d = a.off[u + 1] - a.off[u];
    atomicAdd(&h[deg_bucket(d)], 1);
    if (d > kTriRowWave) atomicAdd(&s_cnt[1], 1);
    else if (d > kWave) atomicAdd(&s_cnt[0], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kTriBuckets; i += BLOCK) {
    base[i] = h[i] ? atomicAdd(&a.ctl->cur[i], h[i]) : 0;
    h[i] = 0;
  }
  if (threadIdx.x == 0) {
    s_base[0] = s_cnt[0] ? atomicAdd(&a.ctl->num_mid.v, s_cnt[0]) : 0;
    s_base[1] = s_cnt[1] ? atomicAdd(&a.ctl->num_big.v, s_cnt[1]) : 0;
    s_cnt[0] = s_cnt[1] = 0;
  }
  __syncthreads();
  for (int32_t u = r0 + threadIdx.x; u < r1; u += BLOCK) {
    const int o = a.off[u], d = a.off[u + 1] - o;
    const int b = deg_bucket(d);
    const int r = base[b] + atomicAdd(&h[b], 1);
    a.ord[r] = u;
    a.dord[r] = d;
    if (!a.members) {
      const float w = W ? a.vw[u] : 0.0f;
      a.rw[u] = make_int4(r, __float_as_int(w), d > 0 ? (int)row16(o, u) : kNoRow, 0);
      if constexpr (W) a.wr[r] = w;
    }
    if (d > kTriRowWave) a.list_big[s_base[1] + atomicAdd(&s_cnt[1], 1)] = u;
    else if (d > kWave) a.list_mid[s_base[0] + atomicAdd(&s_cnt[0], 1)] = u;
  }
}

// Disjoint parts of a batch. A part begins at a vertex with neighbours that no
// row before it reaches past; vertices without neighbours belong to the part
// before them, or to the first one. Per contiguous range of vertices: the largest neighbour id ...
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_reach(TriArgs a) {
  __shared__ int s_max;
  if (!tri_go<kStRank>(a)) return;
  if (threadIdx.x == 0) s_max = -1;
  __syncthreads();
  const int64_t per = ((int64_t)a.n + gridDim.x - 1) / gridDim.x;
  const int32_t r0 = (int32_t)min(per * blockIdx.x, (int64_t)a.n), r1 = (int32_t)min(per * (blockIdx.x + 1), (int64_t)a.n);
  int m = -1;
  for (int32_t u = r0 + threadIdx.x; u < r1; u += BLOCK) {
    const int e = a.off[u + 1];
    if (e > a.off[u]) m = max(m, max(u, a.ind[e - 1]));
  }
  atomicMax(&s_max, m);
  __syncthreads();
  if (threadIdx.x == 0) a.ctl->reach[blockIdx.x] = s_max;
}

// ... then of all ranges before ...
__global__ __launch_bounds__(kTriParts) void k_tri_reach_scan(TriArgs a, int ranges) {
  __shared__ int s[2][kTriParts];
  if (!tri_go<kStRank>(a)) return;
  TriCtl* const c = a.ctl;
  const int t = threadIdx.x;
  s[0][t] = t < ranges ? c->reach[t] : -1;
  int b = 0;
  for (int o = 1; o < kTriParts; o <<= 1) {
    __syncthreads();
    s[b ^ 1][t] = t >= o ? max(s[b][t], s[b][t - o]) : s[b][t];
    b ^= 1;
  }
  __syncthreads();
  if (t < ranges) c->reach[t] = t > 0 ? s[b][t - 1] : -1;
}

// ... then the parts that begin in the range, in order.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_starts(TriArgs a) {
  constexpr int NW = BLOCK / kWave;
  __shared__ int s_m[NW], s_c[NW];
  if (!tri_go<kStRank>(a)) return;
  const int lane = lane_id(), w = threadIdx.x / kWave;
  const int64_t per = ((int64_t)a.n + gridDim.x - 1) / gridDim.x;
  const int32_t r0 = (int32_t)min(per * blockIdx.x, (int64_t)a.n), r1 = (int32_t)min(per * (blockIdx.x + 1), (int64_t)a.n);
  int before = a.ctl->reach[blockIdx.x], count = 0;
  for (int32_t b = r0; b < r1; b += BLOCK) {
    const int32_t u = b + threadIdx.x;
    int m = -1;
    if (u < r1) {
      const int e = a.off[u + 1];
      if (e > a.off[u]) m = max(u, a.ind[e - 1]);
    }
    int incl = m;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int t = __shfl_up(incl, o);
      if (lane >= o) incl = max(incl, t);
    }
    if (lane == kWave - 1) s_m[w] = incl;
    __syncthreads();
    int excl = __shfl_up(incl, 1);
    if (lane == 0) excl = -1;
    excl = max(excl, before);
    int all = before;
    for (int k = 0; k < NW; ++k) {
      if (k < w) excl = max(excl, s_m[k]);
      all = max(all, s_m[k]);
    }
    const bool start = m >= 0 && u > excl;
    const uint64_t sm = ballot(start);
    if (lane == 0) s_c[w] = popc64(sm);
    __syncthreads();
    int at = count + popc64(sm & ((1ull << lane) - 1)), tot = 0;
    for (int k = 0; k < NW; ++k) {
      if (k < w) at += s_c[k];
      tot += s_c[k];
    }
    if (start) a.starts[r0 + at] = u;
    count += tot;
    before = all;
    __syncthreads();
  }
  if (threadIdx.x == 0) a.ctl->nstart[blockIdx.x] = count;
}

// All parts in one list.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_parts(TriArgs a) {
  __shared__ int s_at, s_all;
  if (!tri_go<kStRank>(a)) return;
  if (threadIdx.x == 0) s_at = s_all = 0;
  __syncthreads();
  int at = 0, all = 0;
  for (int k = threadIdx.x; k < (int)gridDim.x; k += BLOCK) {
    const int c = a.ctl->nstart[k];
    all += c;
    if (k < (int)blockIdx.x) at += c;
  }
  atomicAdd(&s_at, at);
  atomicAdd(&s_all, all);
  __syncthreads();
  const int64_t per = ((int64_t)a.n + gridDim.x - 1) / gridDim.x;
  const int32_t r0 = (int32_t)min(per * blockIdx.x, (int64_t)a.n);
  for (int i = threadIdx.x; i < a.ctl->nstart[blockIdx.x]; i += BLOCK) a.parts[s_at + i] = a.starts[r0 + i];
  if (blockIdx.x == 0 && threadIdx.x == 0) a.ctl->num_part.v = s_all;
}

// Ranks of a part's vertices, [first vertex, ...): one workgroup sorts it by
// degree bucket. The vertex weights' finest bit is k_tri_hist's.
template <bool W>
__global__ __launch_bounds__(kTriBuckets) void k_tri_rank_parts(TriArgs a) {
  __shared__ int h[kTriBuckets], base[kTriBuckets];
  __shared__ int part[kTriBuckets / kWave];
  __shared__ int s_i;
  if (!tri_go<kStRank>(a)) return;
  const int tid = threadIdx.x, lane = lane_id();
  const int count = a.ctl->num_part.v;
  for (;;) {
    if (tid == 0) s_i = atomicAdd(&a.ctl->cur_part.v, 1);
    h[tid] = 0;
    __syncthreads();
    const int i = s_i;
    if (i >= count) return;
    // (every vertex has to be in a part: entries may name any of them)
    const int32_t first = a.parts[i], b0 = i > 0 ? first : 0, b1 = i + 1 < count ? a.parts[i + 1] : a.n;
    if (b1 - first > kPartMax) {
      if (tid == 0) refuse<kStRank>(a);
      return;
    }
    for (int32_t u0 = b0; u0 < b1; u0 += 4 * kTriBuckets) {
      int d[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int32_t u = min(u0 + t * kTriBuckets + tid, b1 - 1);
        d[t] = a.off[u + 1] - a.off[u];
      }
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (u0 + t * kTriBuckets + tid < b1) atomicAdd(&h[deg_bucket(d[t])], 1);
    }
    __syncthreads();
    const int b = kTriBuckets - 1 - tid;
    const int v = h[b];
    int incl = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int t = __shfl_up(incl, o);
      if (lane >= o) incl += t;
    }
    if (lane == kWave - 1) part[tid / kWave] = incl;
    __syncthreads();
    int before = 0;
    for (int k = 0; k < tid / kWave; ++k) before += part[k];
    base[b] = b0 + before + incl - v;
    // 16-bit ranks: every vertex with neighbours below kSat16
    if (b == 0 && before + incl - v > kSat16) refuse<kStRank>(a);
    __syncthreads();
    for (int32_t u0 = b0; u0 < b1; u0 += 4 * kTriBuckets) {
      int o[4], d[4];
      float w[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int32_t u = min(u0 + t * kTriBuckets + tid, b1 - 1);
        o[t] = a.off[u];
        d[t] = a.off[u + 1] - o[t];
        if constexpr (W) w[t] = a.vw[u];
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int32_t u = u0 + t * kTriBuckets + tid;
        if (u < b1) {
          const int r = atomicAdd(&base[deg_bucket(d[t])], 1);
          a.rw[u] = make_int4(r, __float_as_int(w[t]), d[t] > 0 ? (int)row16(o[t], u) : kNoRow, b0);
          a.vtx[r] = u;
          a.dr[r] = d[t];
          if constexpr (W) a.wr[r] = w[t];
        }
      }
    }
    __syncthreads();
  }
}

// Row sum of row u (rank ru) and the bound of all of them.
template <bool W>
__device__ __forceinline__ void put_row_sum(const TriArgs& a, int32_t ru, double s) {
  if constexpr (W) {
    a.sr[ru] = s;
    if (!(s >= 0.0) || isinf(s)) {
      refuse<kStOrient>(a);
    } else if (s > 0.0) {
      const int e = ilogb(s) + 1;
      if (e > *(volatile int*)&a.ctl->maxexp.v) atomicMax(&a.ctl->maxexp.v, e);
    }
  }
}

// Writes entry (rank r, row entry k) of row u at sorted position p; cb: the
// first rank of its part.
template <bool W>
__device__ __forceinline__ void put_out(const TriArgs& a, int32_t u, int o, int p, uint32_t r, int k, uint32_t cb) {
  const int e = o + p;
  a.R32[e] = r;
  a.R16[8 * ((size_t)row16(o, u) + kHead) + p] = (uint16_t)min(r - cb, (uint32_t)kSat16);
  a.emap[k] = e;
  if constexpr (W) a.accw[e] = 0.0;
  else a.accu[e] = 0u;
}

// Position p of n: where it is an eighth of the row, its rank goes to the
// header (rows of more than kPivotMin entries have these).
__device__ __forceinline__ void put_pivot(const TriArgs& a, int32_t u, int o, int n, int p, uint32_t r) {
  if (n <= kPivotMin) return;
  uint16_t* pv = a.R16 + 8 * ((size_t)row16(o, u) + 1);
#pragma unroll
  for (int k = 1; k <= 7; ++k)
    if (((n * k) >> 3) == p) pv[k - 1] = (uint16_t)min(r, (uint32_t)kSat16);
}

// Row u's facts (one lane).
__device__ __forceinline__ void put_info(const TriArgs& a, int32_t u, int o, int cnt, int wbits, int ru) {
  a.info[u] = make_int4(o, cnt, 0, ru);
  reinterpret_cast<int4*>(a.R16)[row16(o, u)] = make_int4(o, cnt, 0, wbits);
}

// Rows of at most 64 entries: groups of G lanes, one row each (16 lanes for
// rows of up to 16 entries). The position of an entry among the kept ones is
// the number of kept ranks below its own, counted over the group.
template <bool W, int G>
__device__ __forceinline__ void orient_group(const TriArgs& a, bool valid, int32_t u, int o, int d, int ru, float w,
                                             int cb) {
  const int gl = lane_id() & (G - 1), gb = lane_id() & ~(G - 1);
  bool in_row = valid && gl < d;
  int4 rw = make_int4(0, 0, 0, 0);
  int32_t x = 0;
  if (in_row) {
    x = a.ind[o + gl];
    rw = a.rw[x];
  }
  const int32_t before = __shfl_up(x, 1);
  // a self loop; a row out of order; a neighbour without entries of its own
  if (in_row && (x == u || (gl > 0 && before >= x) || rw.z == kNoRow)) refuse<kStOrient>(a);
  const bool keep = in_row && rw.x < ru;
  const uint64_t km = ballot(keep);
  // kept ranks below mine: a lane that keeps nothing offers no rank
  const int mine = keep ? rw.x : INT32_MAX;
  int pos = 0;
  const int dmax = G == kWave ? d : 16;
  for (int j = 0; j < dmax; ++j) {
    const int rj = G == kWave ? __builtin_amdgcn_readlane(mine, j) : __shfl(mine, gb + j);
    pos += rj < mine ? 1 : 0;
  }
  if (keep) put_out<W>(a, u, o, pos, (uint32_t)rw.x, o + gl, (uint32_t)cb);
  else if (in_row) a.emap[o + gl] = ~rw.z;
  const uint64_t gm = G == kWave ? ~0ull : ((1ull << G) - 1) << gb;
  const int cnt = popc64(km & gm);
  if constexpr (W) {
    double s = in_row ? (double)__int_as_float(rw.y) : 0.0;
#pragma unroll
    for (int t = 1; t < G; t <<= 1) s += __shfl_xor(s, t);
    if (valid && gl == 0) put_row_sum<W>(a, ru, s);
  }
  if (valid && gl == 0) put_info(a, u, o, cnt, __float_as_int(w), ru);
  if (keep) put_pivot(a, u, o, cnt, pos, (uint32_t)(rw.x - cb));
  if (valid && gl < 8) a.R16[8 * ((size_t)row16(o, u) + kHead) + cnt + gl] = (uint16_t)kSat16;
}

// (Eight waves per SIMD: RMAT-22 0.86 -> 0.76 ms.)
template <bool W, int BLOCK>
__global__ __launch_bounds__(BLOCK, 8) void k_tri_orient_small(TriArgs a, int rows) {
  if (!tri_go<kStOrient>(a)) return;
  const int lane = lane_id();
  const int nw = gridDim.x * (BLOCK / kWave);
  for (int64_t base = (int64_t)(blockIdx.x * (BLOCK / kWave) + threadIdx.x / kWave) * rows; base < a.n;
       base += (int64_t)nw * rows) {
    const int32_t u = (int32_t)base + lane;
    int o = 0, d = 0, ru = 0, cb = 0;
    float w = 0.0f;
    if (lane < rows && base + lane < a.n) {
      o = a.off[u];
      d = a.off[u + 1] - o;
      const int4 rw = a.rw[u];
      ru = rw.x;
      w = __int_as_float(rw.y);
      cb = rw.w;
    }
    uint64_t m16 = ballot(d > 0 && d <= 16), m64 = ballot(d > 16 && d <= kWave);
    while (m16) {
      int src = -1;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (m16) {
          const int b = __ffsll((unsigned long long)m16) - 1;
          if (lane / 16 == g) src = b;
          m16 &= m16 - 1;
        }
      }
      const int s = max(src, 0);
      orient_group<W, 16>(a, src >= 0, __shfl(u, s), __shfl(o, s), __shfl(d, s), __shfl(ru, s), __shfl(w, s),
                          __shfl(cb, s));
    }
    while (m64) {
      const int s = __ffsll((unsigned long long)m64) - 1;
      m64 &= m64 - 1;
      orient_group<W, kWave>(a, true, __builtin_amdgcn_readlane(u, s), __builtin_amdgcn_readlane(o, s),
                             __builtin_amdgcn_readlane(d, s), __builtin_amdgcn_readlane(ru, s), __shfl(w, s),
                             __builtin_amdgcn_readlane(cb, s));
    }
  }
}

// Rows of more entries: the kept ranks are compacted into LDS, then every
// kept entry counts the kept ranks below its own (LDS broadcasts, 16 bytes
// per read; quadratic, but the square of |R(u)| is what wedge then tests).
// One wave per row (T = 64 threads, up to kTriRowWave entries) or one
// workgroup per row.
template <bool W, int T, int CAP>
__device__ __forceinline__ void orient_row(const TriArgs& a, int32_t u, int tid, uint32_t* s_r, uint16_t* s_k, int* s_n,
                                           double* s_s) {
  const int o = a.off[u], d = a.off[u + 1] - o;
  const int4 me = a.rw[u];
  const int ru = me.x;
  const uint32_t cb = (uint32_t)me.w;
  const int lane = lane_id();
  if (tid == 0) {
    *s_n = 0;
    if constexpr (W && T > kWave) *s_s = 0.0;
  }
  if constexpr (T > kWave) __syncthreads();
  else lds_fence_wave();
  double sum = 0.0;
  int cnt = 0;  // T == 64: kept so far
  for (int b = 0; b < d; b += 4 * T) {
    int32_t x[4];
    int4 rw[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = a.ind[o + min(b + t * T + tid, d - 1)];
#pragma unroll
    for (int t = 0; t < 4; ++t) rw[t] = a.rw[x[t]];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int i = b + t * T + tid;
      const bool in_row = i < d;
      const bool keep = in_row && rw[t].x < ru;
      if (in_row && (x[t] == u || (i > 0 && a.ind[o + i - 1] >= x[t]) || rw[t].z == kNoRow)) refuse<kStOrient>(a);
      const uint64_t km = ballot(keep);
      int at = 0;
      if constexpr (T == kWave) {
        at = cnt + popc64(km & ((1ull << lane) - 1));
        cnt += popc64(km);
      } else {
        if (lane == 0 && km) at = atomicAdd(s_n, popc64(km));
        at = __builtin_amdgcn_readfirstlane(at) + popc64(km & ((1ull << lane) - 1));
      }
      if (keep) {
        if (at < CAP) {
          s_r[at] = (uint32_t)rw[t].x;
          if constexpr (T == kWave) s_k[at] = (uint16_t)i;
          else reinterpret_cast<int32_t*>(s_k)[at] = i;
        }
      } else if (in_row) {
        a.emap[o + i] = ~rw[t].z;
      }
      if constexpr (W) sum += in_row ? (double)__int_as_float(rw[t].y) : 0.0;
    }
  }
  if constexpr (W) {
#pragma unroll
    for (int t = 1; t < kWave; t <<= 1) sum += __shfl_xor(sum, t);
    if constexpr (T > kWave) {
      if (lane == 0) unsafeAtomicAdd(s_s, sum);
    }
  }
  if constexpr (T > kWave) {
    __syncthreads();
    cnt = *s_n;
    if constexpr (W) sum = *s_s;
  } else {
    lds_fence_wave();
  }
  if (tid == 0) {
    put_row_sum<W>(a, ru, sum);
    put_info(a, u, o, cnt, me.y, ru);
    if (cnt > CAP) refuse<kStOrient>(a);
  }
  const int c = min(cnt, CAP);
  if (tid < 8) a.R16[8 * ((size_t)row16(o, u) + kHead) + c + tid] = (uint16_t)kSat16;
  // pad to a multiple of four with a rank that counts for nobody
  for (int i = c + tid; i < ((c + 3) & ~3); i += T) s_r[i] = 0xFFFFFFFFu;
  if constexpr (T > kWave) __syncthreads();
  else lds_fence_wave();
  for (int i0 = 0; i0 < c; i0 += 2 * T) {
    const int ia = i0 + tid, ib = i0 + T + tid;
    const uint32_t ra = ia < c ? s_r[ia] : 0u, rb = ib < c ? s_r[ib] : 0u;
    int pa = 0, pb = 0;
    for (int j = 0; j < c; j += 4) {
      const uint4 q = *reinterpret_cast<const uint4*>(s_r + j);
      pa += (q.x < ra) + (q.y < ra) + (q.z < ra) + (q.w < ra);
      pb += (q.x < rb) + (q.y < rb) + (q.z < rb) + (q.w < rb);
    }
    const int ka = ia < c ? (T == kWave ? (int)s_k[ia] : reinterpret_cast<int32_t*>(s_k)[ia]) : 0;
    const int kb = ib < c ? (T == kWave ? (int)s_k[ib] : reinterpret_cast<int32_t*>(s_k)[ib]) : 0;
    if (ia < c) {
      put_out<W>(a, u, o, pa, ra, o + ka, cb);
      put_pivot(a, u, o, c, pa, ra - cb);
    }
    if (ib < c) {
      put_out<W>(a, u, o, pb, rb, o + kb, cb);
      put_pivot(a, u, o, c, pb, rb - cb);
    }
  }
  if constexpr (T > kWave) __syncthreads();
  else lds_fence_wave();
}

template <bool W, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_orient_mid(TriArgs a) {
  constexpr int NW = BLOCK / kWave;
  __shared__ __align__(16) uint32_t s_r[NW][kTriRowWave + 4];
  __shared__ uint16_t s_k[NW][kTriRowWave];
  __shared__ int s_n[NW];
  if (!tri_go<kStOrient>(a)) return;
  const int w = threadIdx.x / kWave;
  const int count = a.ctl->num_mid.v;
  for (int i = blockIdx.x * NW + w; i < count; i += gridDim.x * NW)
    orient_row<W, kWave, kTriRowWave>(a, a.list_mid[i], lane_id(), s_r[w], s_k[w], &s_n[w], nullptr);
}

// Lists here and below: a workgroup begins with the item of its own number and
// then asks for more, so that a short list costs no atomics (an empty one took
// reduce 10 us, and 5 without).
template <bool W, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_orient_big(TriArgs a) {
  __shared__ __align__(16) uint32_t s_r[kTriMaxOut + 4];
  __shared__ int32_t s_k[kTriMaxOut];
  __shared__ int s_n, s_i;
  __shared__ double s_s;
  if (!tri_go<kStOrient>(a)) return;
  const int count = a.ctl->num_big.v;
  for (int i = blockIdx.x; i < count;) {
    int next = 0;
    if (threadIdx.x == 0) next = gridDim.x + atomicAdd(&a.ctl->cur_big.v, 1);
    orient_row<W, BLOCK, kTriMaxOut>(a, a.list_big[i], threadIdx.x, s_r, reinterpret_cast<uint16_t*>(s_k), &s_n, &s_s);
    if (threadIdx.x == 0) s_i = next;
    __syncthreads();
    i = s_i;
  }
}

// In rank order: places in the bit matrix, wedge tasks, reduce lists. Each
// workgroup takes BLOCK ranks, scans its counts and reserves with one atomic
// per list; workgroups start in rank order, so the heavy tasks come first.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_plan(TriArgs a) {
  constexpr int NW = BLOCK / kWave;
  constexpr int NL = 7;  // tasks 16-bit, 32-bit, wave list, reduce lists by |R|
  __shared__ int s_w[NL][NW];
  __shared__ unsigned long long s_bw[NW], s_ow[NW];
  __shared__ int s_base[NL];
  __shared__ unsigned long long s_bbase;
  if (!tri_go<kStWedge>(a)) return;
  const int lane = lane_id(), wv = threadIdx.x / kWave;
  for (int64_t b0 = (int64_t)blockIdx.x * BLOCK; b0 < a.n; b0 += (int64_t)gridDim.x * BLOCK) {
    const int32_t at_ord = (int32_t)(b0 + threadIdx.x);
    int d = 0, dp = 0, o = 0, r = 0, lr = 0;  // lr: rank in the part
    int32_t u = 0;
    if (at_ord < a.n) {
      d = a.dord[at_ord];
      if (d > 0) {
        u = a.ord[at_ord];
        const int4 inf = a.info[u];
        const int cb = a.members ? a.rw[u].w : 0;
        o = inf.x;
        dp = inf.y;
        r = inf.w;
        lr = r - cb;
        a.rinfo[at_ord] = make_int4(o, dp, r, cb);
      }
    }
    const int din = d - dp;
    int c[NL] = {0, 0, 0, 0, 0, 0, 0};
    // v by a workgroup where its row is worth a bitmap: 16-bit ranks, or a
    // larger table for what the one-wave kernel's hash does not hold; short
    // rows are in the group tasks (k_tri_scan has the same rule)
    const int npiece = (d + kWedgeB - 1) / kWedgeB;
    const int kind = lr < kSat16 && dp <= kAccA ? 0 : 1;
    const bool grp = d < kGroupMax && (d < kWgMinDeg || at_ord >= a.grp_from);
    const bool wg = din > 0 && !grp && (kind == 0 || (dp > kWaveTab && dp <= kAccB && r <= 32 * kTabB));
    if (wg) c[kind] = npiece;
    else if (din > 0 && !grp) c[2] = 1;
    if (dp > 0) c[dp <= 16 ? 3 : dp <= kRedWave ? 4 : dp <= kRedWg ? 5 : 6] = 1;
    const unsigned long long words = tri_words(dp);
    int incl[NL];
    unsigned long long bi = words, oi = (unsigned long long)dp;
#pragma unroll
    for (int l = 0; l < NL; ++l) incl[l] = c[l];
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
#pragma unroll
      for (int l = 0; l < NL; ++l) {
        const int t = __shfl_up(incl[l], o);
        if (lane >= o) incl[l] += t;
      }
      const unsigned long long tb = __shfl_up(bi, o), to = __shfl_up(oi, o);
      if (lane >= o) {
        bi += tb;
        oi += to;
      }
    }
    if (lane == kWave - 1) {
#pragma unroll
      for (int l = 0; l < NL; ++l) s_w[l][wv] = incl[l];
      s_bw[wv] = bi;
      s_ow[wv] = oi;
    }
    __syncthreads();
    if (threadIdx.x < NL) {
      int t = 0;
      for (int k = 0; k < NW; ++k) {
        const int x = s_w[threadIdx.x][k];
        s_w[threadIdx.x][k] = t;
        t += x;
      }
      int* ctr[NL] = {&a.ctl->num_task[0].v, &a.ctl->num_task[1].v, &a.ctl->num_wave.v,
                      &a.ctl->num_s16.v, &a.ctl->num_s64.v, &a.ctl->num_red[0].v, &a.ctl->num_red[1].v};
      s_base[threadIdx.x] = t ? atomicAdd(ctr[threadIdx.x], t) : 0;
    } else if (threadIdx.x == NL) {
      unsigned long long t = 0, ot = 0;
      for (int k = 0; k < NW; ++k) {
        const unsigned long long x = s_bw[k];
        s_bw[k] = t;
        t += x;
        ot += s_ow[k];
      }
      s_bbase = t ? atomicAdd(&a.ctl->bits.v, t) : 0ull;
      if (ot) atomicAdd(&a.ctl->out_total.v, ot);
    }
    __syncthreads();
    int at[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) at[l] = s_base[l] + s_w[l][wv] + incl[l] - c[l];
    if (wg)
      for (int p = 0; p < npiece; ++p)
        if (at[kind] + p < a.task_cap) a.task[kind][at[kind] + p] = TriTask{kind == 0 ? lr : r, o, d, dp, p, (int32_t)row16(o, u), {0, 0}};
    if (c[2]) a.list_wave[at[2]] = at_ord;
    if (c[3]) a.list_s16[at[3]] = u;
    if (c[4]) a.list_s64[at[4]] = u;
    if (c[5]) a.list_red[0][at[5]] = u;
    if (c[6]) a.list_red[1][at[6]] = u;
    if (dp > 0) {
      const int z = (int)(uint32_t)(s_bbase + s_bw[wv] + bi - words);
      a.info[u].z = z;
      reinterpret_cast<int4*>(a.R16)[row16(o, u)].z = z;
    }
    __syncthreads();
  }
}

// Position of rank r in the sorted row R[0, n), or -1.
template <typename RT>
__device__ __forceinline__ int find_rank(const RT* __restrict__ R, int n, uint32_t r) {
  int lo = 0, len = n;
  while (len > 0) {
    const int half = len >> 1;
    if ((uint32_t)R[lo + half] < r) {
      lo += half + 1;
      len -= half + 1;
    } else {
      len = half;
    }
  }
  return lo < n && (uint32_t)R[lo] == r ? lo : -1;
}

// The same in 16-bit ranks (r < kSat16), the eighth of the row taken from the
// pivots in its header: the search then stays in about one cache line.
__device__ __forceinline__ int find_rank16(const uint16_t* __restrict__ R, int n, uint32_t r, const int4& pv) {
  if (n <= kPivotMin) return find_rank(R, n, r);
  const uint32_t w[4] = {(uint32_t)pv.x, (uint32_t)pv.y, (uint32_t)pv.z, (uint32_t)pv.w};
  int c = 0;
#pragma unroll
  for (int k = 0; k < 7; ++k) c += ((k & 1) ? w[k >> 1] >> 16 : w[k >> 1] & 0xFFFFu) <= r ? 1 : 0;
  const int lo = (n * c) >> 3, hi = (n * (c + 1)) >> 3;
  const int p = find_rank(R + lo, hi - lo, r);
  return p < 0 ? -1 : lo + p;
}

// Eight consecutive entries of a row.
template <typename RT>
struct Octet;
template <>
struct Octet<uint16_t> {
  uint32_t v[4];
  __device__ __forceinline__ void load(const uint16_t* p) {  // 16-byte aligned
    const uint4 x = *reinterpret_cast<const uint4*>(p);
    v[0] = x.x;
    v[1] = x.y;
    v[2] = x.z;
    v[3] = x.w;
  }
};
template <>
struct Octet<uint32_t> {
  uint32_t v[8];
  struct __attribute__((packed, aligned(4))) Raw {
    uint32_t v[4];
  };
  __device__ __forceinline__ void load(const uint32_t* p) {  // any alignment
    const Raw x = *reinterpret_cast<const Raw*>(p), y = *reinterpret_cast<const Raw*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[i] = x.v[i];
      v[4 + i] = y.v[i];
    }
  }
};

template <int CTRL>
__device__ __forceinline__ uint32_t or_dpp(uint32_t v) {
  return v | (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, false);
}

// Tests an octet against the bitmap; hits add w to the LDS sums and come back
// as a byte. A table word is 8 bytes: 32 bits and the byte offset of the sum
// before the one of its lowest bit. Shifting the word left so that the
// entry's own bit is the sign gives the test, and the count of the bits that
// stay is the entry's place: about 8 instructions per entry. 16-bit entries
// past the row's part are ranks of v and above, whose bits are 0; 32-bit ones
// (only nv are valid) read the guard word.
template <typename RT, typename AT>
__device__ __forceinline__ uint32_t probe_octet(const Octet<RT>& y, int nv, const unsigned char* tab, uint32_t guard,
                                                unsigned char* acc, AT w) {
  uint32_t byte = 0;
  // four entries at a time: eight would take the kernel's registers past eight
  // waves per SIMD
#pragma unroll
  for (int h = 1; h >= 0; --h) {
    uint2 t[4];
    uint32_t sh[4];
    if constexpr (sizeof(RT) == 2) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t d = y.v[2 * h + i];
        t[2 * i] = *reinterpret_cast<const uint2*>(tab + ((d >> 2) & 0x3FF8u));
        t[2 * i + 1] = *reinterpret_cast<const uint2*>(tab + ((d >> 18) & 0x3FF8u));
        sh[2 * i] = ~d;
        sh[2 * i + 1] = ~d >> 16;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t wi = 4 * h + i < nv ? min(y.v[4 * h + i] >> 5, guard) : guard;
        t[i] = *reinterpret_cast<const uint2*>(tab + 8u * wi);
        sh[i] = ~y.v[4 * h + i];
      }
    }
#pragma unroll
    for (int i = 3; i >= 0; --i) {
      t[i].x <<= sh[i] & 31u;
      byte = __builtin_amdgcn_alignbit(byte, t[i].x, 31);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if ((int32_t)t[i].x < 0) {
        AT* s = reinterpret_cast<AT*>(acc + ((uint32_t)__popc(t[i].x) * (uint32_t)sizeof(AT) + t[i].y));
        if constexpr (sizeof(AT) == 8) unsafeAtomicAdd(s, w);
        else atomicAdd(s, w);
      }
    }
  }
  return byte;
}

constexpr int kMapCap = 2048;  // words of a task looked at together

// Wedge, one workgroup per task (v, 512 entries of its row). The entries to
// test, rows of p ranks, are cut into words of 32; a map from word to (row,
// word of the row) deals the words to groups of four lanes, eight ranks each,
// so rows of all lengths fill the lanes (dealing rows to 8-lane and larger
// groups by length left half of them idle: RMAT-22 7.9 ms, this 6.1). What is
// left is spread over the lines touched (30 GB at 5 TB/s), the LDS (half of
// the time busy) and the chain of a task's steps.
template <bool W, typename RT, int TAB, int ACC>
__global__ __launch_bounds__(kWedgeB, (TAB <= kTabA ? 8 : 2)) void k_tri_wedge(TriArgs a) {
  constexpr int NW = kWedgeB / kWave;
  constexpr int KIND = sizeof(RT) == 2 ? 0 : 1;
  using AT = typename std::conditional<W, double, uint32_t>::type;
  __shared__ __align__(16) uint2 tab[TAB + (KIND == 0 ? 0 : 2)];
  __shared__ __align__(16) AT acc[ACC];
  __shared__ int4 s_item[kWedgeB];  // row (units of 8 entries, or entries), word of the bit matrix, weight, p
  __shared__ uint16_t s_map[kMapCap];  // item | word << 9
  __shared__ int s_wsum[NW];
  __shared__ int s_task;
  if (!tri_ready<W, kStWedge>(a)) return;
  const int tid = threadIdx.x, lane = lane_id(), w = tid / kWave;
  const int ntask = a.ctl->num_task[KIND].v;
  const unsigned char* const tabp = reinterpret_cast<const unsigned char*>(tab);
  unsigned char* const accp = reinterpret_cast<unsigned char*>(acc);
  // first entry of a row, from its place in s_item
  auto row_at = [&](uint32_t q) -> const RT* {
    if constexpr (KIND == 0) return a.R16 + 8 * (size_t)q;
    else return a.R32 + q;
  };
  // The next task's record and this thread's entry of it are loaded while a
  // task runs, and the task after that is reserved, so a task starts with the
  // headers of its entries.
  auto entry_of = [&](const TriTask& t, bool any) -> int {
    const int i = t.piece * kWedgeB + tid;
    return any && i < t.d ? a.emap[t.o + i] : 0;
  };
  int ti = blockIdx.x, ti1 = ti + gridDim.x;
  if (ti >= ntask) return;
  TriTask tk = a.task[KIND][ti];
  int e = entry_of(tk, true);
  for (;;) {
    const bool more = ti1 < ntask;
    const TriTask tk1 = a.task[KIND][more ? ti1 : ti];
    int ti2 = 0;
    if (tid == 0) ti2 = 2 * gridDim.x + atomicAdd(&a.ctl->cur_task[KIND].v, 1);
    const int32_t r = tk.r;
    const int d = tk.d, ov = tk.o, dpv = tk.dp;
    const uint32_t guard = KIND == 0 ? 0u : (uint32_t)(r + 31) >> 5;
    // 16-bit: the whole table, so that ranks of r and above find 0
    const int nclear = KIND == 0 ? TAB / 2 : (int)guard / 2 + 1;
    for (int i = tid; i < nclear; i += kWedgeB) reinterpret_cast<uint4*>(tab)[i] = make_uint4(0u, 0u, 0u, 0u);
    const RT* const Rv = row_at(KIND == 0 ? (uint32_t)(tk.row + kHead) : (uint32_t)ov);
    uint32_t y0 = 0, y0p = 0;
    if (tid < dpv) {
      y0 = (uint32_t)Rv[tid];
      y0p = tid > 0 ? (uint32_t)Rv[tid - 1] : 0u;
    }
    // the entries of v's row that are not in R(v): where v stands in R(x)
    int p = 0;
    {
      const int k = ov + tk.piece * kWedgeB + tid;
      if (e < 0) {
        const int4* const hd = reinterpret_cast<const int4*>(a.R16) + ~e;
        const int4 xi = hd[0];
        const uint32_t q = KIND == 0 ? (uint32_t)(~e + kHead) : (uint32_t)xi.x;
        if constexpr (KIND == 0) p = find_rank16(row_at(q), xi.y, (uint32_t)r, hd[1]);
        else p = find_rank(row_at(q), xi.y, (uint32_t)r);
        if (p < 0) {
          refuse<kStWedge>(a);  // (v, x) is stored, (x, v) is not
          p = 0;
        } else {
          a.emap[k] = xi.x + p;
          s_item[tid] = make_int4((int)q, (int)((uint32_t)xi.z + tri_words(p)), xi.w, p);
        }
      }
    }
    const int nw = (p + 31) >> 5;
    int incl = nw;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int t = __shfl_up(incl, o);
      if (lane >= o) incl += t;
    }
    if (lane == kWave - 1) s_wsum[w] = incl;
    __syncthreads();
    for (int j = tid; j < dpv; j += kWedgeB) {
      const uint32_t y = j < kWedgeB ? y0 : (uint32_t)Rv[j];
      const uint32_t yp = j < kWedgeB ? y0p : (uint32_t)Rv[j - 1];
      acc[j] = 0;
      atomicOr(&tab[y >> 5].x, 1u << (y & 31u));
      if (j == 0 || (yp >> 5) != (y >> 5)) tab[y >> 5].y = (uint32_t)((j - 1) * (int)sizeof(AT));
    }
    int wbase = incl - nw, total = 0;
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      const int x = s_wsum[k];
      wbase += k < w ? x : 0;
      total += x;
    }
    const int e1 = entry_of(tk1, more);
    for (int w0 = 0; w0 < total; w0 += kMapCap) {
      if (w0 > 0) __syncthreads();  // the words of the last round are done
      const int t1 = min(nw, w0 + kMapCap - wbase);
      for (int t = max(0, w0 - wbase); t < t1; ++t) s_map[wbase + t - w0] = (uint16_t)(tid | (t << 9));
      __syncthreads();
      const int end = min(total - w0, kMapCap);
      for (int j = w * (kWave / 4) + (lane >> 2); j < end; j += kWedgeB / 4) {
        const uint32_t me = s_map[j];
        const int4 it = s_item[me & 511u];
        const int t = (int)(me >> 9), at = 32 * t + 8 * (lane & 3);
        uint32_t byte = 0;
        if (at < it.w) {
          Octet<RT> y;
          y.load(row_at((uint32_t)it.x) + at);
          byte = probe_octet<RT, AT>(y, it.w - at, tabp, guard, accp, W ? (AT)__int_as_float(it.z) : (AT)1);
        }
        // four lanes' bytes make one word of the row
        uint32_t word = byte << ((lane & 3) * 8);
        word = or_dpp<0xB1>(word);
        word = or_dpp<0x4E>(word);
        if ((lane & 3) == 0) a.bits[(uint32_t)it.y + (uint32_t)t] = word;
      }
    }
    if (tid == 0) s_task = ti2;
    __syncthreads();
    // the pairs (v, w): alone on its row, or one of several pieces
    for (int j = tid; j < dpv; j += kWedgeB) {
      const AT s = acc[j];
      if constexpr (W) {
        if (d <= kWedgeB) a.accw[ov + j] = s;
        else if (s != 0.0) unsafeAtomicAdd(&a.accw[ov + j], s);
      } else {
        if (d <= kWedgeB) a.accu[ov + j] = s;
        else if (s != 0u) atomicAdd(&a.accu[ov + j], s);
      }
    }
    if (!more) return;
    ti = ti1;
    ti1 = s_task;
    tk = tk1;
    e = e1;
  }
}

// Wedge for short rows: group_rows(d) vertices v of degree d per task, a thread
// per entry of their rows. The R(v) of the group share one hash table in LDS
// (key: rank and place of v in the group; at most half full, linear probing).
// What a task costs is the chain of dependent reads from its first to its last
// step, which one wave per v paid for every v (RMAT-22 3.0 ms, Chung-Lu 2^20
// 1.0 ms; here 2.4 and 0.63, of which looking a task ahead is 0.6 and 0.17).
constexpr int kGroupSlots = 2 * kWedgeB;
constexpr int kGroupLb = 10;
static_assert(kGroupSlots == 1 << kGroupLb, "slots");

template <bool W>
__global__ __launch_bounds__(kWedgeB, 8) void k_tri_wedge_group(TriArgs a) {
  constexpr int NW = kWedgeB / kWave;
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  using AT = typename std::conditional<W, double, uint32_t>::type;
  __shared__ __align__(16) uint32_t s_key[kGroupSlots];
  __shared__ uint16_t s_slot[kGroupSlots];
  __shared__ AT acc[kWedgeB];
  __shared__ int4 s_item[kWedgeB];  // row, word of the bit matrix, weight, p | place of v << 16
  __shared__ uint16_t s_map[kMapCap];
  __shared__ int s_wsum[NW];
  __shared__ int s_task, s_d;
  __shared__ int s_gt[kGroupMax], s_gr[kGroupMax], s_ge[kGroupMax];  // per length: first task, first and end rank
  if (!tri_ready<W, kStWedge>(a)) return;
  const int tid = threadIdx.x, lane = lane_id(), w = tid / kWave;
  const int ntask = a.ctl->num_group.v;
  s_gt[tid] = a.ctl->grp_task[tid];
  s_gr[tid] = a.ctl->grp_rank[tid];
  s_ge[tid] = a.ctl->cur[tid];  // where the ranks of the next shorter length begin
  __syncthreads();
  // As the bitmap kernel, a task ahead: its length, then its rows, then this
  // thread's entry are looked up while the task before it runs. Lengths
  // descend with the tasks: a task's is the one whose tasks start at or before
  // it and whose next shorter length's start after it.
  auto find_length = [&](int t) {
    if (tid > 0 && s_gt[tid] <= t && t < s_gt[tid - 1]) s_d = tid;
  };
  struct Mine {
    int d, vl, i, nv;  // length, place of this thread's row, its entry of it, rows of the task
    int r0;            // place in ord of the task's first row
    int4 v;            // the row's rinfo
  };
  auto rows_of = [&](int t, int d) {
    Mine m;
    const int rows = group_rows(d);
    const int r0 = s_gr[d] + (t - s_gt[d]) * rows;
    m.d = d;
    m.nv = min(rows, s_ge[d] - r0);
    m.vl = tid / d;
    m.i = tid - m.vl * d;
    m.r0 = r0;
    m.v = m.vl < m.nv ? a.rinfo[r0 + m.vl] : make_int4(0, 0, 0, 0);
    return m;
  };
  int ti = blockIdx.x, ti1 = ti + gridDim.x;
  if (ti >= ntask) return;
  find_length(ti);
  __syncthreads();
  Mine me = rows_of(ti, s_d);
  int e = me.vl < me.nv ? a.emap[me.v.x + me.i] : 0;
  for (;;) {
    const bool more = ti1 < ntask;
    int ti2 = 0;
    if (tid == 0) ti2 = 2 * gridDim.x + atomicAdd(&a.ctl->cur_group.v, 1);
    for (int i = tid; i < kGroupSlots / 4; i += kWedgeB)
      reinterpret_cast<uint4*>(s_key)[i] = make_uint4(kNone, kNone, kNone, kNone);
    acc[tid] = 0;
    __syncthreads();  // (also: every thread has read s_d)
    if (more) find_length(ti1);
    // 16-bit ranks where every row of the task ranks below kSat16 in its part
    const bool use16 = a.members || me.r0 + me.nv <= kSat16;
    const uint32_t cb = use16 ? (uint32_t)me.v.w : 0u;
    const bool mine = me.vl < me.nv;
    const uint32_t r = (uint32_t)me.v.z - cb;
    int p = 0;
    if (mine) {
      const int ov = me.v.x, vl = me.vl;
      if (e >= 0) {
        const uint32_t y = a.R32[e] - cb;
        const uint32_t key = y | ((uint32_t)vl << 26);
        uint32_t q = hash_bucket((int32_t)(y ^ ((uint32_t)vl * 0x9E3B5u)), kGroupLb);
        while (atomicCAS(&s_key[q], kNone, key) != kNone) q = (q + 1) & (kGroupSlots - 1);  // at most half full: ends
        s_slot[q] = (uint16_t)(vl * me.d + (e - ov));
      } else {
        const int4* const hd = reinterpret_cast<const int4*>(a.R16) + ~e;
        const int4 xi = hd[0];
        if (use16) p = find_rank16(reinterpret_cast<const uint16_t*>(hd + kHead), xi.y, r, hd[1]);
        else p = find_rank(a.R32 + xi.x, xi.y, r);
        if (p < 0) {
          refuse<kStWedge>(a);  // (v, x) is stored, (x, v) is not
          p = 0;
        } else {
          a.emap[ov + me.i] = xi.x + p;
          s_item[tid] = make_int4(use16 ? ~e + kHead : xi.x, (int)((uint32_t)xi.z + tri_words(p)), xi.w, p | (vl << 16));
        }
      }
    }
    const int nw = (p + 31) >> 5;
    int incl = nw;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const int t = __shfl_up(incl, o);
      if (lane >= o) incl += t;
    }
    if (lane == kWave - 1) s_wsum[w] = incl;
    __syncthreads();
    int wbase = incl - nw, total = 0;
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      const int x = s_wsum[k];
      wbase += k < w ? x : 0;
      total += x;
    }
    Mine me1 = me;
    int e1 = 0;
    if (more) {
      me1 = rows_of(ti1, s_d);
      if (me1.vl < me1.nv) e1 = a.emap[me1.v.x + me1.i];
    }
    for (int w0 = 0; w0 < total; w0 += kMapCap) {
      if (w0 > 0) __syncthreads();
      const int t1 = min(nw, w0 + kMapCap - wbase);
      for (int t = max(0, w0 - wbase); t < t1; ++t) s_map[wbase + t - w0] = (uint16_t)(tid | (t << 9));
      __syncthreads();
      const int end = min(total - w0, kMapCap);
      for (int j = w * (kWave / 4) + (lane >> 2); j < end; j += kWedgeB / 4) {
        const uint32_t mp = s_map[j];
        const int4 it = s_item[mp & 511u];
        const int t = (int)(mp >> 9), at = 32 * t + 8 * (lane & 3), nvalid = (it.w & 0xFFFF) - at;
        uint32_t byte = 0;
        if (nvalid > 0) {
          const uint32_t vt = (uint32_t)it.w >> 16, mix = vt * 0x9E3B5u, tag = vt << 26;
          uint32_t y[8];
          if (use16) {
            Octet<uint16_t> o;
            o.load(a.R16 + 8 * (size_t)(uint32_t)it.x + at);
#pragma unroll
            for (int k = 0; k < 8; ++k) y[k] = (k & 1) ? o.v[k >> 1] >> 16 : o.v[k >> 1] & 0xFFFFu;
          } else {
            Octet<uint32_t> o;
            o.load(a.R32 + it.x + at);
#pragma unroll
            for (int k = 0; k < 8; ++k) y[k] = o.v[k];
          }
          const AT wu = W ? (AT)__int_as_float(it.z) : (AT)1;
#pragma unroll
          for (int h = 0; h < 8; h += 4) {
            uint32_t q[4], key[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              q[k] = hash_bucket((int32_t)(y[h + k] ^ mix), kGroupLb);
              key[k] = s_key[q[k]];
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              // an entry past the row's part looks like an empty slot
              const uint32_t want = h + k < nvalid ? y[h + k] | tag : kNone;
              while (key[k] != want && key[k] != kNone && want != kNone) {
                q[k] = (q[k] + 1) & (kGroupSlots - 1);
                key[k] = s_key[q[k]];
              }
              if (key[k] == want && want != kNone) {
                byte |= 1u << (h + k);
                AT* s = &acc[s_slot[q[k]]];
                if constexpr (W) unsafeAtomicAdd(s, wu);
                else atomicAdd(s, wu);
              }
            }
          }
        }
        uint32_t word = byte << ((lane & 3) * 8);
        word = or_dpp<0xB1>(word);
        word = or_dpp<0x4E>(word);
        if ((lane & 3) == 0) a.bits[(uint32_t)it.y + (uint32_t)t] = word;
      }
    }
    if (tid == 0) s_task = ti2;
    __syncthreads();
    if (mine && me.i < me.v.y) {
      AT* const gacc = W ? (AT*)a.accw : (AT*)a.accu;
      gacc[me.v.x + me.i] = acc[tid];
    }
    if (!more) return;
    ti = ti1;
    ti1 = s_task;
    me = me1;
    e = e1;
  }
}

// Wedge, one wave per v: long rows of ranks beyond the workgroup kernels' tables. R(v)
// is hashed in LDS (at most half full, linear probing); longer R(v) that the
// workgroup kernels cannot take are searched in memory. 64 entries of v's row
// at a time, their words dealt to groups of four lanes as above.
constexpr int kWaveSlots = 2 * kWaveTab;
constexpr int kWaveMap = 512;

template <bool W, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_wedge_wave(TriArgs a) {
  constexpr int NW = BLOCK / kWave;
  using AT = typename std::conditional<W, double, uint32_t>::type;
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  __shared__ uint32_t s_key[NW][kWaveSlots];
  __shared__ uint8_t s_pos[NW][kWaveSlots];
  __shared__ AT s_acc[NW][kWaveTab];
  __shared__ int4 s_item[NW][kWave];
  __shared__ uint16_t s_map[NW][kWaveMap];  // item | word << 6
  if (!tri_ready<W, kStWedge>(a)) return;
  const int lane = lane_id(), w = threadIdx.x / kWave;
  const int count = a.ctl->num_wave.v;
  AT* const gacc = W ? (AT*)a.accw : (AT*)a.accu;
  for (int li = blockIdx.x * NW + w; li < count; li += gridDim.x * NW) {
    const int place = a.list_wave[li];
    const int4 vi = a.rinfo[place];
    const int d = a.dord[place], ov = vi.x, dpv = vi.y, r = vi.z, lr = vi.z - vi.w;
    const bool lds = dpv <= kWaveTab;
    const int lb = max(ceil_log2(2 * dpv), 4);
    const uint32_t mask = (1u << lb) - 1u;
    if (lds) {
      for (int j = lane; j <= (int)mask; j += kWave) s_key[w][j] = kNone;
      lds_fence_wave();
      for (int j = lane; j < dpv; j += kWave) {
        const uint32_t y = a.R32[ov + j];
        s_acc[w][j] = 0;
        uint32_t q = hash_bucket((int32_t)y, lb);
        while (atomicCAS(&s_key[w][q], kNone, y) != kNone) q = (q + 1) & mask;  // at most half full: ends
        s_pos[w][q] = (uint8_t)j;
      }
    }
    for (int b = 0; b < d; b += kWave) {
      int p = 0;
      if (b + lane < d) {
        const int k = ov + b + lane;
        const int e = a.emap[k];
        if (e < 0) {
          const int4* const hd = reinterpret_cast<const int4*>(a.R16) + ~e;
          const int4 xi = hd[0];
          if (lr < kSat16)
            p = find_rank16(reinterpret_cast<const uint16_t*>(hd + kHead), xi.y, (uint32_t)lr, hd[1]);
          else
            p = find_rank(a.R32 + xi.x, xi.y, (uint32_t)r);
          if (p < 0) {
            refuse<kStWedge>(a);
            p = 0;
          } else {
            a.emap[k] = xi.x + p;
            s_item[w][lane] = make_int4(xi.x, (int)((uint32_t)xi.z + tri_words(p)), xi.w, p);
          }
        }
      }
      const int nw = (p + 31) >> 5;
      int incl = nw;
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const int t = __shfl_up(incl, o);
        if (lane >= o) incl += t;
      }
      const int total = __builtin_amdgcn_readlane(incl, kWave - 1), wbase = incl - nw;
      for (int w0 = 0; w0 < total; w0 += kWaveMap) {
        lds_fence_wave();
        const int t1 = min(nw, w0 + kWaveMap - wbase);
        for (int t = max(0, w0 - wbase); t < t1; ++t) s_map[w][wbase + t - w0] = (uint16_t)(lane | (t << 6));
        lds_fence_wave();
        const int end = min(total - w0, kWaveMap);
        for (int j = lane >> 2; j < end; j += kWave / 4) {
          const uint32_t e = s_map[w][j];
          const int4 it = s_item[w][e & 63u];
          const int t = (int)(e >> 6), at = 32 * t + 8 * (lane & 3);
          uint32_t byte = 0;
          if (at < it.w) {
            const AT wu = W ? (AT)__int_as_float(it.z) : (AT)1;
            Octet<uint32_t> y;
            y.load(a.R32 + it.x + at);
            if (lds) {
              uint32_t q[8], key[8];
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                q[i] = hash_bucket((int32_t)y.v[i], lb);
                key[i] = s_key[w][q[i]];
              }
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                const bool live = at + i < it.w;
                while (live && key[i] != y.v[i] && key[i] != kNone) {
                  q[i] = (q[i] + 1) & mask;
                  key[i] = s_key[w][q[i]];
                }
                if (live && key[i] == y.v[i]) {
                  byte |= 1u << i;
                  AT* s = &s_acc[w][s_pos[w][q[i]]];
                  if constexpr (W) unsafeAtomicAdd(s, wu);
                  else atomicAdd(s, wu);
                }
              }
            } else {
              for (int i = 0; i < 8 && at + i < it.w; ++i) {
                const int q = find_rank(a.R32 + ov, dpv, y.v[i]);
                if (q >= 0) {
                  byte |= 1u << i;
                  if constexpr (W) unsafeAtomicAdd(&gacc[ov + q], wu);
                  else atomicAdd(&gacc[ov + q], wu);
                }
              }
            }
          }
          uint32_t word = byte << ((lane & 3) * 8);
          word = or_dpp<0xB1>(word);
          word = or_dpp<0x4E>(word);
          if ((lane & 3) == 0) a.bits[(uint32_t)it.y + (uint32_t)t] = word;
        }
      }
      lds_fence_wave();
    }
    if (lds)
      for (int j = lane; j < dpv; j += kWave) gacc[ov + j] = s_acc[w][j];
    lds_fence_wave();
  }
}

// The value of slot e (row u of rank ru, neighbour rank rv): the quotient, or
// the intersection and the sum of the row sums for the kernel-level entry.
template <bool W>
__device__ __forceinline__ void put_value(const TriArgs& a, int e, int32_t u, int du, double su, uint32_t rv,
                                          double isum, uint32_t cnt) {
  if (a.mode == kModeIsF32) {
    const float add = W ? (float)isum : (float)cnt;
    const float ws = a.work32[u] + a.work32[a.vtx[rv]];
    // the slot's sum was read before: its place takes the pair
    if constexpr (W) reinterpret_cast<float2*>(a.accw)[e] = make_float2(add, ws);
    else {
      a.accu[e] = __float_as_uint(add);
      a.R32[e] = __float_as_uint(ws);
    }
    return;
  }
  float q;
  if constexpr (W) {
    const double ws = su + a.sr[rv];
    q = (float)(isum / (ws - isum));
  } else {
    const float fI = (float)cnt;
    q = fI / ((float)(du + a.dr[rv]) - fI);
  }
  a.R32[e] = __float_as_uint(q);
}

// Reduce for |R(u)| <= 16: four rows u per wave, lane p of a group holds row p
// of the matrix; the transpose comes from one ballot per column.
template <bool W>
__device__ __forceinline__ void reduce_16(const TriArgs& a, bool valid, int32_t u) {
  const int lane = lane_id(), gl = lane & 15, gb = lane & ~15;
  int4 inf = make_int4(0, 0, 0, 0);
  int4 me = make_int4(0, 0, 0, 0);
  if (valid) {
    inf = a.info[u];
    me = a.rw[u];
  }
  const int o = inf.x, dp = inf.y;
  const bool act = valid && gl < dp;
  uint32_t rv = 0, row = 0, cnt = 0;
  float wv = 0.0f;
  double sum = 0.0;
  if (act) {
    rv = a.R32[o + gl];
    if constexpr (W) {
      wv = a.wr[rv];
      sum = a.accw[o + gl];
    } else {
      cnt = a.accu[o + gl];
    }
    if (gl > 0) row = a.bits[(uint32_t)inf.z + tri_words(gl)];
  }
  int dmax = dp;
  dmax = max(dmax, __shfl_xor(dmax, 16));
  dmax = max(dmax, __shfl_xor(dmax, 32));
  dmax = __builtin_amdgcn_readfirstlane(dmax);
  uint32_t full = row;
  for (int c = 0; c < dmax; ++c) {
    const uint64_t col = ballot((row >> c) & 1u);
    if (gl == c) full |= (uint32_t)(col >> gb) & 0xFFFFu;
  }
  if constexpr (W) {
    for (int q = 0; q < dmax; ++q) {
      const float wq = __shfl(wv, gb + q);
      if ((full >> q) & 1u) sum += (double)wq;
    }
  } else {
    cnt += (uint32_t)__popc(full);
  }
  if (act) put_value<W>(a, o + gl, u, a.dr[me.x], W ? a.sr[me.x] : 0.0, rv, sum, cnt);
}

template <bool W, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_reduce_16(TriArgs a) {
  if (!tri_ready<W, kStReduce>(a)) return;
  const int gw = blockIdx.x * (BLOCK / kWave) + threadIdx.x / kWave, nw = gridDim.x * (BLOCK / kWave);
  const int n16 = a.ctl->num_s16.v;
  for (int i = gw * 4; i < n16; i += nw * 4) {
    const int j = i + lane_id() / 16;
    reduce_16<W>(a, j < n16, a.list_s16[min(j, n16 - 1)]);
  }
}

// Reduce for larger |R(u)|. I = M w for the symmetric 0/1 matrix M whose lower
// triangle is stored. A wave takes 64 rows P and runs over all 64-column
// blocks Q: the stored block (P, Q) for Q <= P and the transpose of the stored
// block (Q, P) for Q >= P. A block is held as 16-bit chunks, chunk h (columns
// 16h ..) of row 16g + r in lane 16h + r, register g. Bits are transposed
// inside 16 lanes by four butterfly steps (DPP), two registers packed in one,
// and register and lane group change places by the gfx950 row swaps: about 35
// instructions for 4096 bits.
//   Unweighted: the chunks' bit counts.
//   Weighted: matrix products of the bits, spread to bytes, with the weights
// as integers of 7-bit digits (weight = sum digit_n 2^(7n) 2^lsb, eight digits
// hold the 53 bits that tri_ready admits), int8 MFMA 16x16x64 with int32 sums,
// which are exact; each row's digit sums are put together in fp64, exactly.
// Both operands use the same order of k, so the product does not depend on it.
// (Adding the weights bit by bit in fp64 took 24 instructions per 64 bits:
// RMAT-22 9.8 ms for all of reduce, 3.9 with the products; Chung-Lu 2^20
// unweighted 0.61 and 0.36.)
struct Chunks {
  uint32_t x[2];  // registers g = 0, 1 and g = 2, 3, 16 bits each
};

__device__ __forceinline__ Chunks transpose_block(Chunks c) {
  const int r = lane_id() & 15;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint32_t x = c.x[i];
    auto step = [&](uint32_t t, int s, uint32_t low) {
      const bool up = (r & s) != 0;
      const uint32_t own = up ? ~low : low;  // columns this lane keeps
      const uint32_t rot = __builtin_amdgcn_alignbit(t, t, up ? s : 32 - s);
      x = (x & own) | (rot & ~own);
    };
    step((uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x128, 0xF, 0xF, false), 8, 0x00FF00FFu);  // row_ror:8
    int t = __builtin_amdgcn_update_dpp(0, (int)x, 0x104, 0xF, 0x5, false);                    // row_shl:4
    t = __builtin_amdgcn_update_dpp(t, (int)x, 0x114, 0xF, 0xA, false);                        // row_shr:4
    step((uint32_t)t, 4, 0x0F0F0F0Fu);
    step((uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, false), 2, 0x33333333u);
    step((uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, false), 1, 0x55555555u);
    c.x[i] = x;
  }
  const auto s32 = __builtin_amdgcn_permlane32_swap(c.x[0], c.x[1], false, false);
  const uint32_t sel = (lane_id() & 16) ? 0x07060302u : 0x05040100u;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto s16 = __builtin_amdgcn_permlane16_swap(s32[i], s32[i], false, false);
    c.x[i] = __builtin_amdgcn_perm(s16[1], s16[0], sel);
  }
  return c;
}

typedef int v4i __attribute__((ext_vector_type(4)));

// The 16 bits at `sh` of x as 16 bytes of 0 or 1.
__device__ __forceinline__ v4i spread16(uint32_t x, int sh) {
  v4i v;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t nib = __builtin_amdgcn_ubfe(x, sh + 4 * j, 4);
    v[j] = (int)((nib * 0x204081u) & 0x01010101u);
  }
  return v;
}

constexpr int kDigits = 8;      // 7-bit digits of a weight
constexpr int kRedRow = 64 + 4; // ints per digit of a wave's 64 row sums (padded)

// Digits of the weight of row entry k, to digit arrays in blocks of 16 entries
// (16 bytes per digit).
__device__ __forceinline__ void put_digits(unsigned char* dig, int k, float w, int lsb) {
  const uint32_t b = __float_as_uint(w);
  const int ex = (int)((b >> 23) & 0xFFu);
  const uint64_t full = ex ? (b & 0x7FFFFFu) | 0x800000u : b & 0x7FFFFFu;
  const int sh = (ex ? ex - 150 : -149) - lsb;
  uint64_t v = full == 0 ? 0ull : sh >= 0 ? full << sh : full >> -sh;  // (trailing zeros shifted out)
#pragma unroll
  for (int n = 0; n < kDigits; ++n) {
    dig[(k >> 4) * (16 * kDigits) + n * 16 + (k & 15)] = (unsigned char)(v & 127u);
    v >>= 7;
  }
}

// Rows [64 P, 64 P + 64) of u's product; returns the lane's row's result
// (lane = row), without the wedge part.
template <bool W>
__device__ __forceinline__ void reduce_rows(const TriArgs& a, uint32_t z, int dp, int P, const unsigned char* dig,
                                            int* stage, double unit, double& sum, uint32_t& cnt) {
  const int lane = lane_id(), r = lane & 15, h = lane >> 4;
  const int nb = (dp + 63) >> 6;
  const uint16_t* __restrict__ hw = reinterpret_cast<const uint16_t*>(a.bits);
  v4i acc[4];
  uint32_t c16[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int g = 0; g < 4; ++g) acc[g] = v4i{0, 0, 0, 0};
  auto use = [&](const Chunks& c, int Q) {
    if constexpr (W) {
      const v4i bq = *reinterpret_cast<const v4i*>(dig + (4 * Q + h) * (16 * kDigits) + (r & 7) * 16);
#pragma unroll
      for (int g = 0; g < 4; ++g)
        acc[g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(spread16(c.x[g >> 1], 16 * (g & 1)), bq, acc[g], 0, 0, 0);
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) c16[g] += (uint32_t)__popc(g & 1 ? c.x[g >> 1] >> 16 : c.x[g >> 1] & 0xFFFFu);
    }
  };
  // 16 columns from 16 * (4 C + h) of the rows 64 B + 16 g + r
  auto load = [&](int B, int C) {
    uint32_t v[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int p = 64 * B + 16 * g + r, c0 = 64 * C + 16 * h;
      v[g] = 0u;
      if (p < dp && c0 < p) v[g] = hw[2 * (size_t)(z + tri_words(p)) + (size_t)(4 * C + h)];
    }
    return Chunks{{v[0] | (v[1] << 16), v[2] | (v[3] << 16)}};
  };
  for (int Q = 0; Q <= P; ++Q) use(load(P, Q), Q);
  for (int Q = P; Q < nb; ++Q) use(transpose_block(load(Q, P)), Q);
  if constexpr (W) {
    // acc[g][i]: row 16 g + 4 h + i, digit r (r < 8)
    if (r < kDigits) {
#pragma unroll
      for (int g = 0; g < 4; ++g) *reinterpret_cast<v4i*>(stage + r * kRedRow + 16 * g + 4 * h) = acc[g];
    }
    lds_fence_wave();
    double t = 0.0;
#pragma unroll
    for (int n = kDigits - 1; n >= 0; --n) t = t * 128.0 + (double)stage[n * kRedRow + lane];
    sum = t * unit;
    lds_fence_wave();
  } else {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      c16[g] += __shfl_xor(c16[g], 16);
      c16[g] += __shfl_xor(c16[g], 32);
    }
    cnt = h == 0 ? c16[0] : h == 1 ? c16[1] : h == 2 ? c16[2] : c16[3];
  }
}

// All rows of u, by the T threads of a wave or workgroup.
template <bool W, int T>
__device__ __forceinline__ void reduce_vertex(const TriArgs& a, int32_t u, int tid, unsigned char* dig, int* stage) {
  constexpr int NW = T / kWave;
  const int lane = lane_id(), w = tid / kWave;
  const int4 inf = a.info[u];
  const int ru = a.rw[u].x;
  const int o = inf.x, dp = inf.y;
  const int nb = (dp + 63) >> 6;
  double unit = 1.0;
  if constexpr (W) {
    const int lsb = a.ctl->lsb.v == INT32_MAX ? 0 : a.ctl->lsb.v;
    unit = ldexp(1.0, lsb);
    for (int k = tid; k < nb * 64; k += T) put_digits(dig, k, k < dp ? a.wr[a.R32[o + k]] : 0.0f, lsb);
    if constexpr (T > kWave) __syncthreads();
    else lds_fence_wave();
  }
  const int du = a.dr[ru];
  const double su = W ? a.sr[ru] : 0.0;
  for (int P = w; P < nb; P += NW) {
    double sum = 0.0;
    uint32_t cnt = 0;
    reduce_rows<W>(a, (uint32_t)inf.z, dp, P, dig, stage, unit, sum, cnt);
    const int p = P * 64 + lane;
    if (p < dp) {
      const uint32_t rv = a.R32[o + p];
      if constexpr (W) sum += a.accw[o + p];
      else cnt += a.accu[o + p];
      put_value<W>(a, o + p, u, du, su, rv, sum, cnt);
    }
  }
  if constexpr (T > kWave) __syncthreads();
  else lds_fence_wave();
}

template <bool W, int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_tri_reduce_wave(TriArgs a) {
  constexpr int NW = BLOCK / kWave;
  __shared__ __align__(16) unsigned char dig[W ? NW : 1][W ? kRedWave * kDigits : 16];
  __shared__ __align__(16) int stage[W ? NW : 1][W ? kDigits * kRedRow : 4];
  if (!tri_ready<W, kStReduce>(a)) return;
  const int w = threadIdx.x / kWave;
  const int count = a.ctl->num_s64.v;
  for (int i = blockIdx.x * NW + w; i < count; i += gridDim.x * NW)
    reduce_vertex<W, kWave>(a, a.list_s64[i], lane_id(), dig[W ? w : 0], stage[W ? w : 0]);
}

template <bool W, int BLOCK, int CAP>
__global__ __launch_bounds__(BLOCK) void k_tri_reduce_wg(TriArgs a) {
  constexpr int NW = BLOCK / kWave;
  constexpr int L = CAP > kRedWg ? 1 : 0;
  __shared__ __align__(16) unsigned char dig[W ? CAP * kDigits : 16];
  __shared__ __align__(16) int stage[W ? NW : 1][W ? kDigits * kRedRow : 4];
  __shared__ int s_i;
  if (!tri_ready<W, kStReduce>(a)) return;
  const int count = a.ctl->num_red[L].v;
  for (int i = blockIdx.x; i < count;) {
    int next = 0;
    if (threadIdx.x == 0) next = gridDim.x + atomicAdd(&a.ctl->cur_red[L].v, 1);
    reduce_vertex<W, BLOCK>(a, a.list_red[L][i], threadIdx.x, dig, stage[W ? threadIdx.x / kWave : 0]);
    if (threadIdx.x == 0) s_i = next;
    __syncthreads();
    i = s_i;
  }
}

template <bool W>
__global__ __launch_bounds__(256) void k_tri_deliver(TriArgs a) {
  if (!tri_ready<W, kStReduce>(a)) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) a.ctl->done = 1;
  const int64_t nt = (int64_t)gridDim.x * blockDim.x;
  if (a.mode == kModeIsF32) {
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < a.m; k += nt) {
      const int e = a.emap[k];
      float2 x;
      if constexpr (W) x = reinterpret_cast<const float2*>(a.accw)[e];
      else x = make_float2(__uint_as_float(a.accu[e]), __uint_as_float(a.R32[e]));
      a.out32[k] = (a.accumulate ? a.out32[k] : 0.0f) + x.x;
      a.ws32[k] = x.y;
    }
    return;
  }
  // four entries per thread, a stride apart: their gathers are in flight together
  const int64_t quads = (a.m + 3) / 4;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < quads; i += nt) {
    int e[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) e[t] = i + t * quads < a.m ? a.emap[i + t * quads] : 0;
    uint32_t q[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) q[t] = a.R32[e[t]];
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (i + t * quads < a.m) a.out32[i + t * quads] = __uint_as_float(q[t]);
  }
}

size_t al256(size_t v) { return (v + 255) / 256 * 256; }

uint64_t bits_cap(int64_t m, int bits) { return std::min<uint64_t>((uint64_t)m * bits / 4, 0xFFFFFF00ull); }

int64_t tri_tasks(int32_t n, int64_t m) { return m / kWedgeB + std::min<int64_t>(n, m / kWgMinDeg) + 1; }

// Carves the workspace; with p == nullptr only measures it.
size_t carve(TriArgs& a, unsigned char* p, int32_t n, int64_t m, bool weighted, int bits) {
  size_t o = 0;
  auto take = [&](size_t bytes) {
    unsigned char* q = p ? p + o : nullptr;
    o += al256(bytes);
    return q;
  };
  const size_t nn = (size_t)std::max(n, 1), mm = (size_t)m;
  a.ctl = reinterpret_cast<TriCtl*>(take(sizeof(TriCtl)));
  a.rw = reinterpret_cast<int4*>(take(nn * sizeof(int4)));
  a.vtx = reinterpret_cast<int32_t*>(take(nn * 4));
  a.dr = reinterpret_cast<int32_t*>(take(nn * 4));
  a.wr = reinterpret_cast<float*>(weighted ? take(nn * 4) : nullptr);
  a.sr = reinterpret_cast<double*>(weighted ? take(nn * 8) : nullptr);
  a.info = reinterpret_cast<int4*>(take(nn * sizeof(int4)));
  a.rinfo = reinterpret_cast<int4*>(take(nn * sizeof(int4)));
  a.ord = reinterpret_cast<int32_t*>(take(nn * 4));
  a.dord = reinterpret_cast<int32_t*>(take(nn * 4));
  a.R32 = reinterpret_cast<uint32_t*>(take((mm + 16) * 4));
  a.R16 = reinterpret_cast<uint16_t*>(take((size_t)(row16_line(mm, nn) + 1) * 128));
  a.emap = reinterpret_cast<int32_t*>(take(mm * 4));
  unsigned char* acc = take(mm * (weighted ? 8 : 4));
  a.accw = weighted ? reinterpret_cast<double*>(acc) : nullptr;
  a.accu = weighted ? nullptr : reinterpret_cast<uint32_t*>(acc);
  a.bits_cap = bits_cap(m, bits);
  a.bits = reinterpret_cast<uint32_t*>(take((size_t)a.bits_cap * 4));
  a.list_mid = reinterpret_cast<int32_t*>(take(nn * 4));
  a.list_big = reinterpret_cast<int32_t*>(take(nn * 4));
  a.task_cap = tri_tasks(n, m);
  a.task[0] = reinterpret_cast<TriTask*>(take((size_t)a.task_cap * sizeof(TriTask)));
  a.task[1] = reinterpret_cast<TriTask*>(take((size_t)a.task_cap * sizeof(TriTask)));
  a.list_wave = reinterpret_cast<int32_t*>(take(nn * 4));
  a.list_s16 = reinterpret_cast<int32_t*>(take(nn * 4));
  a.starts = a.list_wave;  // (rank is done with them when plan runs)
  a.parts = a.list_s16;
  a.list_s64 = a.list_mid;  // orient is done with its lists when plan runs
  a.list_red[0] = a.list_big;
  a.list_red[1] = reinterpret_cast<int32_t*>(take((size_t)std::min<int64_t>(nn, m / kRedWg + 1) * 4));
  return o;
}

template <bool W>
hipError_t tri_launch(const TriArgs& a, hipStream_t s) {
  const int cus = device_cu_count();
  constexpr int PB = 256;
  auto grid = [&](int64_t items, int per, int cap) {
    return dim3((unsigned)std::max<int64_t>(1, std::min<int64_t>((items + per - 1) / per, (int64_t)cus * cap)));
  };
  {
    ProfScope ps("tri_rank", s);
    hipLaunchKernelGGL(k_tri_init, dim3(1), dim3(kSamples), 0, s, a);
    const dim3 g = grid(a.n, PB * 4, kTriParts / 256);
    static_assert(kTriParts % 256 == 0, "ranges");
    hipLaunchKernelGGL((k_tri_hist<W, PB>), dim3(g.x + kSamples / PB), dim3(PB), 0, s, a);
    hipLaunchKernelGGL(k_tri_scan, dim3(1), dim3(kTriBuckets), 0, s, a);
    hipLaunchKernelGGL((k_tri_rank<W, PB>), g, dim3(PB), 0, s, a);
    if (a.members) {
      const dim3 gp((unsigned)std::min<int64_t>(g.x, kTriParts));
      hipLaunchKernelGGL((k_tri_reach<PB>), gp, dim3(PB), 0, s, a);
      hipLaunchKernelGGL(k_tri_reach_scan, dim3(1), dim3(kTriParts), 0, s, a, (int)gp.x);
      hipLaunchKernelGGL((k_tri_starts<PB>), gp, dim3(PB), 0, s, a);
      hipLaunchKernelGGL((k_tri_parts<PB>), gp, dim3(PB), 0, s, a);
      hipLaunchKernelGGL((k_tri_rank_parts<W>), dim3(cus * 2), dim3(kTriBuckets), 0, s, a);
    }
  }
  {
    ProfScope ps("tri_orient", s);
    hipLaunchKernelGGL((k_tri_orient_big<W, 512>), dim3(cus * 4), dim3(512), 0, s, a);
    hipLaunchKernelGGL((k_tri_orient_mid<W, PB>), grid(std::min<int64_t>(a.n, a.m / kWave), PB / kWave, 32), dim3(PB), 0, s, a);
    // vertices per wave: a wave takes its rows one after another, so it is given
    // fewer where the graph has few (64 / 16: 200003 vertices 101 / 68 us, two
    // unions of 64 small graphs 387 / 293)
    int rows = kWave;
    while (rows > 16 && a.n < (int64_t)cus * 128 * rows) rows /= 2;
    hipLaunchKernelGGL((k_tri_orient_small<W, PB>), grid(a.n, PB / kWave * rows, 32), dim3(PB), 0, s, a, rows);
  }
  {
    ProfScope ps("tri_plan", s);
    hipLaunchKernelGGL((k_tri_plan<PB>), grid(a.n, PB, 64), dim3(PB), 0, s, a);
  }
  {
    ProfScope ps("tri_wedge", s);
    hipLaunchKernelGGL((k_tri_wedge<W, uint16_t, kTabA, kAccA>), dim3(cus * 4), dim3(kWedgeB), 0, s, a);
    hipLaunchKernelGGL((k_tri_wedge<W, uint32_t, kTabB, kAccB>), dim3(cus), dim3(kWedgeB), 0, s, a);
    hipLaunchKernelGGL((k_tri_wedge_group<W>), dim3(cus * 4), dim3(kWedgeB), 0, s, a);
    // (rows of kGroupMax entries and more at ranks past kSat16: not in smaller graphs,
    // but a batch's large |R| may be there by their ranks in the whole)
    if (a.members || a.m >= (int64_t)kGroupMax * kSat16)
      hipLaunchKernelGGL((k_tri_wedge_wave<W, PB>), grid(std::min<int64_t>(a.n, a.m / kGroupMax), PB / kWave, 16), dim3(PB), 0, s, a);
  }
  {
    ProfScope ps("tri_reduce", s);
    hipLaunchKernelGGL((k_tri_reduce_wg<W, PB, kTriMaxOut>), dim3(cus * (W ? 3 : 8)), dim3(PB), 0, s, a);
    hipLaunchKernelGGL((k_tri_reduce_wg<W, PB, kRedWg>), dim3(cus * 8), dim3(PB), 0, s, a);
    hipLaunchKernelGGL((k_tri_reduce_wave<W, PB>), grid(a.n, PB / kWave, 32), dim3(PB), 0, s, a);
    hipLaunchKernelGGL((k_tri_reduce_16<W, PB>), grid(a.n, 4 * PB / kWave, 32), dim3(PB), 0, s, a);
  }
  {
    ProfScope ps("tri_deliver", s);
    hipLaunchKernelGGL((k_tri_deliver<W>), grid(a.m, 1024, 32), dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

}  // namespace

size_t tri_workspace_bytes(int32_t n, int64_t m, bool weighted, int bits) {
  TriArgs a{};
  return carve(a, nullptr, n, m, weighted, bits);
}

hipError_t run_tri(int mode, const EngineArgs& e, bool always, void* ws, const int** done, hipStream_t s, int bits) {
  TriArgs a{};
  const bool weighted = e.vw != nullptr;
  carve(a, static_cast<unsigned char*>(ws), e.n, e.m, weighted, bits);
  a.n = e.n;
  a.m = e.m;
  a.off = e.off;
  a.ind = e.ind;
  a.vw = e.vw;
  a.mode = mode;
  a.work32 = e.work32;
  a.out32 = e.out32;
  a.ws32 = e.ws32;
  a.accumulate = e.accumulate;
  a.members = e.members;
  a.always = always;
  if (!a.members) {
    a.ord = a.vtx;
    a.dord = a.dr;
  }
  // (all parts' ranks are below kSat16)
  a.grp_from = a.members ? e.n : kSat16;
  *done = &a.ctl->done;
  return weighted ? tri_launch<true>(a, s) : tri_launch<false>(a, s);
}

}  // namespace jc
