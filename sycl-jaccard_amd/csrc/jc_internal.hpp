// Internal interfaces between the C ABI layer and the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace jc {

// Epilogue of an intersection: what is written for a pair (u, x).
enum Mode : int {
  kModeEcU = 0,   // EC unweighted: out = I / ((float)(du+dx) - I)
  kModeEcW = 1,   // EC weighted:   out = (float)(I / ((S[u]+S[x]) - I)), fp64
  kModeIsF32 = 2, // VC intersection, reference buffers: weight_i (+)= I, weight_s = work[u]+work[x]
  kModeIsF64 = 3, // VC intersection, fp64 internals: wi64 = I, ws64 = S[u]+S[x]
};

// Rows up to this degree are handled one wave per row; longer rows by a
// workgroup per task. Tasks cover at most kTaskSpan consecutive entries of a
// row (sized so item list, per-item state and a 128 KiB hash table fit the
// 160 KiB LDS of a CU, one 1024-thread workgroup per CU).
#ifndef JC_TASK_SPAN
#define JC_TASK_SPAN 896
#endif
constexpr int kSmallMax = 128;
constexpr int kTaskSpan = JC_TASK_SPAN;
// Graphs with fewer vertices than this use quotient hash tables (16-bit keys):
// every id is at most 2^24 - 2, so the padding key of a row's last pass
// (INT32_MAX, whose low 24 bits are 2^24 - 1) hashes like no id.
constexpr int32_t kQuotMaxN = 1 << 24;

// Range facts of the vertex weights of a weighted pass (launch_exact_info):
// every weight is a multiple of 2^min_lsb, every row sum is below 2^max_exp,
// bad != 0 if a weight is negative or not finite.
struct ExactInfo {
  int min_lsb;
  int max_exp;
  int bad;
  int pad;
};

// True when every weight sum of a pass is exact in plain fp64: all vertex
// weights non-negative multiples of 2^min_lsb and every row sum below
// 2^max_exp with max_exp - min_lsb <= 52, so every partial sum of a subset of
// a row fits 53 bits; double-double and plain fp64 then give the same bits.
// No non-zero weight (min_lsb unset) or no non-zero row sum (max_exp unset,
// so every weight that occurs in a row is 0) makes every sum 0: exact too.
// The difference is taken in 64 bits (the unset values are INT32_MAX and
// INT32_MIN).
__host__ __device__ inline bool exact_sums_fit_f64(const ExactInfo& e) {
  if (e.bad != 0) return false;
  if (e.min_lsb == INT32_MAX || e.max_exp == INT32_MIN) return true;
  return (int64_t)e.max_exp - (int64_t)e.min_lsb <= 52;
}

struct EngineArgs {
  int32_t n;
  int64_t m;
  const int32_t* off;
  const int32_t* ind;
  const float* vw;       // vertex weights (weighted modes), else nullptr
  const double* S64;     // fp64 row sums of vw (kModeEcW, kModeIsF64)
  const float* work32;   // fp32 row sums (kModeIsF32)
  float* out32;          // EC result, or weight_i (kModeIsF32)
  float* ws32;           // weight_s (kModeIsF32)
  double* wi64;          // kModeIsF64
  double* ws64;          // kModeIsF64
  int accumulate;        // kModeIsF32: add I to the prior weight_i contents
  // schedule (device memory)
  const int2* tasks;     // (row, piece) for rows with degree > kSmallMax, degree-descending buckets
  const int* num_tasks;
  int* task_counter;
  const int32_t* small_rows;  // rows with 1 <= degree <= small_max
  const int* num_small;
  // tuning (results do not depend on these)
  int small_max;              // degree bin threshold: one wave per row up to here (1..kSmallMax)
  int small_blocks_per_cu;    // grid of the one-wave-per-row kernel
  int wide_index;             // 1: rows are read with 64-bit addresses (set by the
                              // launcher when m * 4 does not fit 32-bit offsets)
  int bitmap_blocks_per_cu;   // workgroups per CU of the bitmap-task kernel (1 or 2)
  int hash_table;             // 1: 32-bit tables even where quotient tables apply
  int quot_max_disp;          // > 0: quotient keys move at most quot_max_disp - 1 buckets
  uint32_t bm_budget;         // bytes of the bitmap table region (set by the launcher)
  // Row segments (device memory, optional): when nseg > 0 only the rows of
  // the segments are computed. segs[i] = (first row, running row count before
  // segment i) for i < nseg, and segs[nseg] = (0, total rows); seg_rows and
  // seg_edges are the totals (rows and stored edges of all segments).
  const int2* segs;
  int nseg;
  int32_t seg_rows;
  int64_t seg_edges;
  // Weighted modes: optional range facts of vw and S64 (device memory); when
  // they show all sums are exact in fp64 the kernels add in plain fp64.
  ExactInfo* exact;
  // Parts of *exact that the schedule has yet to put together, or nfacts = 0.
  const ExactInfo* facts;
  int nfacts;
  // Hash-table tasks the quotient-table kernel had to abandon (device memory,
  // set by the launcher), and whether a launch is the 32-bit redo of them.
  int* redo;
  int* num_redo;
  int redo_pass;
  // Device flag, or nullptr: when it is not 0 the results are already there
  // (the oriented engine delivered them) and the pass does nothing.
  const int* skip;
  int members;  // the graph is a union of many small graphs (oriented engine)
  // The schedule counters at the head of the workspace are zero already
  // (launch_prepare over engine_counter_words() words of it).
  int counters_ready;
  // Capacity of the task array when every task is a bitmap task and the list
  // was written in one pass, longer rows from the front, the others from the
  // back (set by the launcher; 0: two counted lists).
  int32_t task_cap;
};
int engine_counter_words();

// Oriented engine (jc_tri.hip): kModeEcU / kModeEcW (out32 the result) and
// kModeIsF32. It delivers only where its conditions hold, which the device
// decides; *done then receives the address (in ws) of a flag that is set when
// the results were written, for EngineArgs::skip of the owner engine that
// must follow. ws holds tri_workspace_bytes(n, m, weighted) bytes. always: not
// only where the rows say that it is the faster engine.
constexpr int32_t kTriMaxN = 1 << 26;  // its hash keys hold 26-bit ranks
// Oriented engine (jc_tri.hip) before the owner engine: from tri_min_edges
// stored entries on, where no tuning is given or it names a batch (and then
// only if the device finds the rows skewed enough, see k_tri_init). Below,
// its two dozen dependent launches are most of its time. Owner and oriented
// engine, ms: weighted RMAT 1.5M entries 0.32 / 0.30, 2.8M 0.54 / 0.42, 4.0M
// 0.98 / 0.53, Chung-Lu 1.6M 0.29 / 0.32, 3.2M 0.49 / 0.44, 4.5M 1.09 / 0.52;
// unweighted RMAT 2.8M 0.37 / 0.36, 4.0M 0.53 / 0.47, 5.8M 0.78 / 0.61, 11.7M
// 1.63 / 1.19, Chung-Lu 3.2M 0.35 / 0.37, 4.2M 0.45 / 0.44, 6.4M 0.68 / 0.58,
// 12.8M 1.34 / 1.09, 25.6M 2.86 / 2.17. Above the crossing, for what a graph
// that the device turns down pays, 25 to 50 us (k_tri_init).
constexpr int32_t tri_min_edges(bool weighted) { return weighted ? 3 << 20 : 6 << 20; }
// (sum |R|^2 / 64 words of bit matrix are at least (m / 2)^2 / n / 64, above the
// engine's 4 m words from a mean row of 1024 entries on; a uniform random graph
// reaches them at 768)
constexpr bool tri_can(int32_t n, int64_t m) { return n <= kTriMaxN && m <= 768ll * n; }
// Where it is tried without being asked for. (Below a mean row of 2 entries its
// arrays over the vertices, 100 bytes of each, would be the most of it.)
constexpr bool tri_pays(int32_t n, int64_t m, bool weighted) {
  return m >= tri_min_edges(weighted) && m >= 2ll * n && tri_can(n, m);
}
constexpr int32_t kTriPart = 65536;  // vertices of a member (EngineArgs::members), at most
// bits: quarter words of bit matrix per stored entry; a graph that needs more is
// refused after orient. RMAT graphs need 1 (16 entries per vertex of 2^12) to 5.
constexpr int kTriBits = 16;
size_t tri_workspace_bytes(int32_t n, int64_t m, bool weighted, int bits = kTriBits);
hipError_t run_tri(int mode, const EngineArgs& base, bool always, void* ws, const int** done, hipStream_t s,
                   int bits = kTriBits);

// Workspace needed by an owner-engine pass over a graph with n vertices and m
// stored edges (task list, small-row list, counters). With row segments, n and
// m are the segments' totals.
size_t engine_workspace_bytes(int32_t n, int64_t m);

// Owner engine: every pair written once per stored direction. When
// check_sentinel is set the target array was pre-filled with the sentinel and
// a fix-up pass recomputes positions that no symmetric pair reached.
// ws must hold engine_workspace_bytes(n, m) bytes.
hipError_t run_engine(int mode, bool weighted, const EngineArgs& base, void* ws, bool fixup,
                      hipStream_t stream);

// Pair path: out per (first[i], second[i]); invalid ids give NaN. S: the row
// sums of vw, or nullptr (kModeEcW then sums the rows of each pair, as where *no_S,
// in device memory, is not 0).
hipError_t run_pairs(int mode, bool weighted, int32_t n, const int32_t* off, const int32_t* ind,
                     const float* vw, const float* work32, const double* S, int64_t np, const int32_t* first,
                     const int32_t* second, float* out32, float* ws32, int accumulate,
                     hipStream_t stream, const int* no_S = nullptr);
// *no_S (device memory) = whether the row sums of all of the graph are more work
// than those of the pairs' rows.
hipError_t launch_pairs_want(int32_t n, int64_t m, const int32_t* off, int64_t np, const int32_t* first,
                             const int32_t* second, int* no_S, hipStream_t stream);

// Fills *info (device memory) for vertex weights vw[n] and their row sums S[n].
hipError_t launch_exact_info(int32_t n, const float* vw, const double* S, ExactInfo* info, hipStream_t s,
                             const int* skip = nullptr);

// Records a failing HIP call for jc_last_hip_error(); returns the JC_ERR_* code.
int note_hip_error(hipError_t e);

// Workspace of one call (jc_mem.hip), for work on stream s from get() to
// release(), as if by hipMallocAsync and hipFreeAsync; most of it memory that the
// library keeps. kOptional: the caller can do without, and get() fails where a
// large one would have to be fresh memory. kOnce: a call that programs do not
// make over and over, for which less is kept.
struct CallBuf {
  enum Use { kNeeded, kOptional, kOnce };
  void* p = nullptr;
  CallBuf() = default;
  CallBuf(const CallBuf&) = delete;
  CallBuf& operator=(const CallBuf&) = delete;
  ~CallBuf() { release(); }
  hipError_t get(size_t bytes, hipStream_t stream, Use use = kNeeded);
  void release();

 private:
  hipStream_t s = nullptr;
  void* block = nullptr;  // the kept block, or nullptr
  int device = 0;
};

// Streaming kernels.
hipError_t launch_fill_f32(float* x, int64_t n, float v, hipStream_t s);
// (skip: as EngineArgs::skip)
hipError_t launch_fill_u32(uint32_t* x, int64_t n, uint32_t v, hipStream_t s, const int* skip = nullptr);
hipError_t launch_fill_u64(uint64_t* x, int64_t n, uint64_t v, hipStream_t s, const int* skip = nullptr);
// Row sums take a scratch area of rowsum_scratch_bytes(n) (long-row list),
// or nullptr to allocate one on the stream for the call.
size_t rowsum_scratch_bytes(int32_t n);
hipError_t launch_rowsum_f32(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* v,
                             float* work, void* scratch, hipStream_t s);
hipError_t launch_rowsum_f64(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* v,
                             double* S, void* scratch, hipStream_t s, const int* skip = nullptr);
hipError_t launch_vertex_weights(int32_t n, int64_t m, const int32_t* off, const float* edge_w, float* W,
                                 void* scratch, hipStream_t s);
// Row sums of graphs of n vertices and m stored edges are one launch, which can also
// fill *info (as launch_exact_info, into a started ExactInfo: launch_prepare), or, where
// *nfacts is not 0, leaves that many parts of it at scratch (EngineArgs::facts).
bool rowsum_one_launch(int32_t n, int64_t m);
hipError_t launch_rowsum_exact(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* v, double* S,
                               void* scratch, int* nfacts, ExactInfo* info, hipStream_t s,
                               const int* skip = nullptr);
// x[0, n) = v (x may be nullptr; skip: as EngineArgs::skip), zero[0, nzero) = 0, *info (may be nullptr) started.
hipError_t launch_prepare(uint32_t* x, int64_t n, uint32_t v, int* zero, int nzero, ExactInfo* info, hipStream_t s,
                          const int* skip = nullptr);
// Everything in one launch for graphs whose CSR fits the LDS (jc_tiny.hip):
// out as kModeEcU / kModeEcW. Any CSR, symmetric or not.
bool tiny_fits(int32_t n, int64_t m, bool weighted);
hipError_t run_tiny(int32_t n, int64_t m, const int32_t* off, const int32_t* ind, const float* vw, float* out,
                    hipStream_t s);
hipError_t launch_jw_f32(int64_t m, const float* wi, const float* ws, float* out, hipStream_t s);
hipError_t launch_jw_f64(int64_t m, const double* wi, const double* ws, float* out, hipStream_t s);
hipError_t launch_ec_scan(int32_t n, const int32_t* off, int32_t* dest, float* wj, hipStream_t s);
// bitmap table region of the workgroup kernel with one workgroup per CU:
// [0] unweighted, [1] weighted layout
void bitmap_table_bytes(int64_t out[2]);
// jc_degree_stats: 69 words (see k_degree_stats), zeroed by the caller
hipError_t launch_degree_stats(int32_t n, const int32_t* off, const int32_t* ind, unsigned long long* out,
                               hipStream_t s);
hipError_t launch_count_above(int64_t m, const float* x, float thresh, unsigned long long* cnt,
                              hipStream_t s);
hipError_t launch_validate(int32_t n, int64_t m, const int32_t* off, const int32_t* ind,
                           int* flags, hipStream_t s);

int device_cu_count();

}  // namespace jc
