// Graph ingest on the device: the preparation the reference driver does on
// the host with std::set (main.cpp:98-120, readMtxToCSR.cpp:116-208) --
// optional reverse edges, self loops dropped, repeated (src, dst) merged,
// columns sorted -- as a radix sort (hipCUB) of (src, dst) keys of as many
// bits as the ids take, then one counting and one compacting pass, which also
// writes the row offsets.
//
// All of it is bound by memory: each 8-bit digit of the key is a pass over
// keys and weights, so the keys hold 2 ceil(log2 n) bits and not 32 + that,
// in 32-bit words where these suffice. Flags, positions and source rows are
// formed again from the sorted keys where they are needed, not stored.
// Measured, 16M weighted draws symmetrized over 1000003 vertices: 5
// digits instead of 7, 2.66 -> 1.86 ms, of which the sort takes 1.46 (0.27 a
// digit, 768 MB each); keys 0.11, counting 0.08 and compacting 0.13 (8 keys per
// thread; 16 took 0.21), where flags, their scan and the offsets took 0.47.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <stdint.h>

#include <algorithm>

#include "../../include/jaccard_amd.h"
#include "jc_device.hpp"
#include "jc_internal.hpp"

namespace jc {
namespace {

constexpr int kTile = 4096;  // sorted keys of a workgroup of the compaction
constexpr int kTileB = 512;

// Bits of an id in a key.
int id_bits(int32_t n) {
  int b = 1;
  while (b < 31 && (1ll << b) < n) ++b;
  return b;
}

// The largest key, (n - 1, n - 1): a self loop, so no edge has it. Self loops
// and ids outside [0, n) get it, and are dropped.
template <typename Key>
__host__ __device__ __forceinline__ Key drop_key(int32_t n, int bits) {
  return n > 0 ? (Key)((Key)(n - 1) << bits | (Key)(n - 1)) : (Key)0;
}

// Keys (src, dst). Reverse edges follow the originals, so a stable sort keeps
// an original's weight for a repeated pair.
template <typename Key>
__global__ void k_make_keys(int32_t n, int bits, int64_t e, const int32_t* __restrict__ src,
                            const int32_t* __restrict__ dst, const float* __restrict__ w, int sym,
                            Key* __restrict__ keys, float* __restrict__ vals, int* bad) {
  const Key drop = drop_key<Key>(n, bits);
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < e; i += (int64_t)gridDim.x * blockDim.x) {
    const int32_t u = src[i], v = dst[i];
    const bool ok = u >= 0 && u < n && v >= 0 && v < n;
    if (!ok) atomicOr(bad, 1);
    const bool keep = ok && u != v;
    const float x = w ? w[i] : 1.0f;
    keys[i] = keep ? (Key)u << bits | (Key)v : drop;
    if (vals) vals[i] = x;
    if (sym) {
      keys[e + i] = keep ? (Key)v << bits | (Key)u : drop;
      if (vals) vals[e + i] = x;
    }
  }
}

// Sorted key i of a tile is a kept edge and differs from key i - 1.
template <typename Key>
__device__ __forceinline__ bool kept(const Key* __restrict__ keys, int64_t i, int64_t e2, Key drop, Key& k, Key& before) {
  k = drop;
  before = drop;
  if (i >= e2) return false;
  k = keys[i];
  if (i > 0) before = keys[i - 1];
  return k < drop && (i == 0 || before != k);
}

// Kept edges of every tile.
template <typename Key>
__global__ __launch_bounds__(kTileB) void k_count(int64_t e2, Key drop, const Key* __restrict__ keys,
                                                  int32_t* __restrict__ count) {
  __shared__ int part[kTileB / kWave];
  int c = 0;
#pragma unroll
  for (int j = 0; j < kTile / kTileB; ++j) {
    Key k, before;
    c += popc64(ballot(kept(keys, (int64_t)blockIdx.x * kTile + j * kTileB + threadIdx.x, e2, drop, k, before)));
  }
  if (lane_id() == 0) part[threadIdx.x / kWave] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int w = 0; w < kTileB / kWave; ++w) t += part[w];
    count[blockIdx.x] = t;
  }
}

// Counts of tiles -> kept edges before each, and their total.
__global__ __launch_bounds__(1024) void k_tile_scan(int tiles, int32_t* __restrict__ count, int32_t* total) {
  __shared__ int part[1024 / kWave];
  int carry = 0;
  for (int base = 0; base < tiles; base += 1024) {
    const int i = base + threadIdx.x;
    const int v = i < tiles ? count[i] : 0;
    int incl = v;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
      const int t = __shfl_up(incl, s);
      if (lane_id() >= s) incl += t;
    }
    if (lane_id() == kWave - 1) part[threadIdx.x / kWave] = incl;
    __syncthreads();
    int before = carry;
    for (int w = 0; w < 1024 / kWave; ++w) {
      if (w < (int)threadIdx.x / kWave) before += part[w];
      carry += part[w];
    }
    if (i < tiles) count[i] = before + incl - v;
    __syncthreads();
  }
  if (threadIdx.x == 0) *total = carry;
}

// The kept edges of a tile to their places; and offsets[r] = first kept edge
// of row r: the first key of a row writes the rows after the previous key's,
// the last edge (or the first dropped key) closes the rows up to n.
template <typename Key>
__global__ __launch_bounds__(kTileB) void k_compact(int32_t n, int bits, int64_t e2, Key drop,
                                                    const Key* __restrict__ keys, const float* __restrict__ vals,
                                                    const int32_t* __restrict__ tile, int64_t capacity,
                                                    int32_t* __restrict__ off, int32_t* __restrict__ ind,
                                                    float* __restrict__ wout) {
  constexpr int NJ = kTile / kTileB, NW = kTileB / kWave;
  static_assert(NJ * NW == kWave, "one count per lane");
  __shared__ int place[kWave];
  Key k[NJ], before[NJ];
  uint64_t mask[NJ];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t first = (int64_t)blockIdx.x * kTile + threadIdx.x;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    mask[j] = ballot(kept(keys, first + j * kTileB, e2, drop, k[j], before[j]));
    if (lane == 0) place[j * NW + wave] = popc64(mask[j]);
  }
  __syncthreads();
  if (wave == 0) {
    const int v = place[lane];
    int incl = v;
#pragma unroll
    for (int s = 1; s < kWave; s <<= 1) {
      const int t = __shfl_up(incl, s);
      if (lane >= s) incl += t;
    }
    place[lane] = tile[blockIdx.x] + incl - v;
  }
  __syncthreads();
  const Key low = ((Key)1 << bits) - 1;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int64_t i = first + j * kTileB;
    if (i >= e2) break;
    const int32_t p = place[j * NW + wave] + popc64(mask[j] & ((1ull << lane) - 1));
    const bool here = (mask[j] >> lane) & 1;
    const int32_t up = i > 0 ? (int32_t)(before[j] >> bits) : -1;
    const int32_t u = (int32_t)(k[j] >> bits);
    if (here) {
      for (int32_t r = up + 1; r <= u; ++r) off[r] = p;
      if (p < capacity) {  // (otherwise reported after the count is read)
        ind[p] = (int32_t)(k[j] & low);
        if (wout) wout[p] = vals[i];
      }
    }
    const bool last = k[j] < drop;
    if (last ? i == e2 - 1 : i == 0 || before[j] < drop)
      for (int32_t r = (last ? u : up) + 1; r <= n; ++r) off[r] = p + (here ? 1 : 0);
  }
}

int grid_of(int64_t items) {
  return (int)std::max<int64_t>(1, std::min<int64_t>((items + 255) / 256, (int64_t)device_cu_count() * 32));
}

// Everything from the draws on; *host: [0] an id out of range, [1] stored edges.
template <typename Key>
hipError_t ingest(int32_t n, int64_t num_edges, int64_t e2, const int32_t* src, const int32_t* dst, const float* edge_w,
                  int symmetrize, int32_t* offsets, int32_t* indices, float* weights_out, int64_t capacity,
                  int32_t* host, hipStream_t s) {
  const bool weighted = weights_out != nullptr;
  const int bits = id_bits(n);
  const int end_bit = std::min(2 * bits, (int)sizeof(Key) * 8);
  const int tiles = (int)((e2 + kTile - 1) / kTile);
  // device temporaries: keys x2, (weights x2), tile counts, counters, the sort's
  size_t sort_bytes = 0;
  hipError_t err;
  if (weighted)
    err = hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (Key*)nullptr, (Key*)nullptr, (float*)nullptr,
                                             (float*)nullptr, (int)e2, 0, end_bit, s);
  else
    err = hipcub::DeviceRadixSort::SortKeys(nullptr, sort_bytes, (Key*)nullptr, (Key*)nullptr, (int)e2, 0, end_bit, s);
  if (err != hipSuccess) return err;
  auto al = [](size_t v) { return (v + 255) / 256 * 256; };
  size_t o = 0;
  const size_t o_k0 = o; o += al(e2 * sizeof(Key));
  const size_t o_k1 = o; o += al(e2 * sizeof(Key));
  const size_t o_v0 = o; o += weighted ? al(e2 * 4) : 0;
  const size_t o_v1 = o; o += weighted ? al(e2 * 4) : 0;
  const size_t o_tl = o; o += al((size_t)tiles * 4);
  const size_t o_ct = o; o += al(2 * sizeof(int32_t));
  const size_t o_tmp = o; o += al(sort_bytes);
  CallBuf buf;
  if ((err = buf.get(o, s, CallBuf::kOnce)) != hipSuccess) return err;
  unsigned char* ws = static_cast<unsigned char*>(buf.p);
  Key* k0 = reinterpret_cast<Key*>(ws + o_k0);
  Key* k1 = reinterpret_cast<Key*>(ws + o_k1);
  float* v0 = weighted ? reinterpret_cast<float*>(ws + o_v0) : nullptr;
  float* v1 = weighted ? reinterpret_cast<float*>(ws + o_v1) : nullptr;
  int32_t* tile = reinterpret_cast<int32_t*>(ws + o_tl);
  int32_t* ctr = reinterpret_cast<int32_t*>(ws + o_ct);
  const Key drop = drop_key<Key>(n, bits);
  do {
    if ((err = launch_fill_u32(reinterpret_cast<uint32_t*>(ctr), 2, 0u, s)) != hipSuccess) break;
    hipLaunchKernelGGL((k_make_keys<Key>), dim3(grid_of(num_edges)), dim3(256), 0, s, n, bits, num_edges, src, dst,
                       edge_w, symmetrize, k0, v0, ctr);
    if ((err = hipGetLastError()) != hipSuccess) break;
    if (weighted) err = hipcub::DeviceRadixSort::SortPairs(ws + o_tmp, sort_bytes, k0, k1, v0, v1, (int)e2, 0, end_bit, s);
    else err = hipcub::DeviceRadixSort::SortKeys(ws + o_tmp, sort_bytes, k0, k1, (int)e2, 0, end_bit, s);
    if (err != hipSuccess) break;
    hipLaunchKernelGGL((k_count<Key>), dim3(tiles), dim3(kTileB), 0, s, e2, drop, k1, tile);
    hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(1024), 0, s, tiles, tile, ctr + 1);
    hipLaunchKernelGGL((k_compact<Key>), dim3(tiles), dim3(kTileB), 0, s, n, bits, e2, drop, k1, v1, tile, capacity,
                       offsets, indices, weights_out);
    if ((err = hipGetLastError()) != hipSuccess) break;
    if ((err = hipMemcpyAsync(host, ctr, 2 * sizeof(int32_t), hipMemcpyDeviceToHost, s)) != hipSuccess) break;
    err = hipStreamSynchronize(s);
  } while (false);
  return err;
}

}  // namespace
}  // namespace jc

extern "C" int jc_csr_from_edges(int32_t n, int64_t num_edges, const int32_t* src, const int32_t* dst,
                                 const float* edge_w, int symmetrize, int32_t* offsets, int32_t* indices,
                                 float* weights_out, int64_t capacity, int64_t* m_out, jc_stream_t stream) {
  if (n < 0 || num_edges < 0 || !offsets || !m_out || capacity < 0 || (num_edges > 0 && (!src || !dst)) ||
      (capacity > 0 && !indices))
    return JC_ERR_INVALID_ARG;
  const int64_t e2 = num_edges * (symmetrize ? 2 : 1);
  if (e2 >= INT32_MAX) return JC_ERR_INVALID_ARG;  // sort and scan index with int
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  int32_t host[2] = {0, 0};
  hipError_t err;
  if (num_edges == 0) {
    err = jc::launch_fill_u32(reinterpret_cast<uint32_t*>(offsets), (int64_t)n + 1, 0u, s);
    if (err == hipSuccess) err = hipStreamSynchronize(s);
  } else if (2 * jc::id_bits(n) <= 32) {
    err = jc::ingest<uint32_t>(n, num_edges, e2, src, dst, edge_w, symmetrize, offsets, indices, weights_out, capacity,
                               host, s);
  } else {
    err = jc::ingest<uint64_t>(n, num_edges, e2, src, dst, edge_w, symmetrize, offsets, indices, weights_out, capacity,
                               host, s);
  }
  if (err != hipSuccess) return jc::note_hip_error(err);
  *m_out = host[1];
  if (host[0]) return JC_ERR_INVALID_ARG;
  return host[1] > capacity ? JC_ERR_WORKSPACE : JC_OK;
}
