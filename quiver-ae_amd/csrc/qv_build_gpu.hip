// qv_build_gpu.hip -- index construction on the GPU.
//
// DiskANN's builder is absent from the reference checkout (deps/DiskANN is an
// empty submodule), so the 10M-100M point configurations are built here, on the
// device, in the same formats the reference reads.  Algorithms:
//   * PQ: data centred on the sample mean, M contiguous chunks, Lloyd k-means
//     with 256 centres per chunk (centre update in float64), then every point
//     encoded.
//   * Medoid: the point nearest to the mean of all points.
//   * Graph: Vamana with batched insertion (batch sizes double up to a cap).  For
//     each batch the persistent search kernel runs a beam search of width L for
//     every inserted point and records the expanded nodes; a workgroup per point then
//     applies RobustPrune(alpha, R) to expanded nodes plus current neighbours;
//     reverse edges are sorted by target (rocPRIM radix sort) and a wave per
//     target merges them, a workgroup pruning again when the list would exceed R.
// Every step is deterministic for a given seed.
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <type_traits>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <numeric>
#include <vector>

#include "qv_common.hpp"
#include "qv_device.hpp"
#include "qv_hip_util.hpp"
#include "qv_index_impl.hpp"
#include "qv_mixture.hpp"

using namespace qv;
using namespace qv::dev;

namespace {

struct GLayout {
  uint8_t* pages;
  int64_t n;
  int64_t npp;
  int64_t node_size;
  int64_t data_size;
  int32_t dim;
  int32_t R;
};

__device__ __forceinline__ uint8_t* node_rec(const GLayout& L, int64_t v) {
  const int64_t page = v / L.npp;
  return L.pages + page * 4096 + (v - page * L.npp) * L.node_size;
}

template <class T>
__global__ void gather_rows_f32(const T* __restrict__ base, int dim, const int32_t* __restrict__ ids,
                                int64_t count, float* __restrict__ out) {
  const int64_t total = count * dim;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = e / dim;
    const int j = (int)(e - r * dim);
    out[e] = (float)base[(int64_t)ids[r] * dim + j];
  }
}

// ---- PQ training and encoding ------------------------------------------------
//
// Lloyd's iterations run on the device from the sample's rows in place: nearest
// pivot per (row, chunk), a stable partition of the rows by pivot, and one wave
// per (chunk, pivot) that adds its rows.  The sums are float64 in ascending row
// order, as one thread on the host adds them, so the pivots do not depend on
// where they are computed.
// 15 iterations over 250,000 rows x 128 uint8 in 32 chunks: 0.45 ms of
// nearest-pivot search, 0.13 ms of partition and 0.23 ms of sums each, 13 ms in
// all; with the assignments copied to the host and added up there it was about
// 380 ms of a 576 ms build (now 230 ms).  100,003 x 96 float: 383 -> 240 ms.

constexpr int kPqSegment = 4096;  // rows one wave partitions

// Training sample: row i is (i * n) / ns.
__global__ void pq_rows_kernel(int64_t n, int64_t ns, int32_t* __restrict__ rows) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < ns) rows[i] = (int32_t)((i * n) / ns);
}

// Mean of the sample per dimension.  8-bit rows: whole-number sums, in any
// order; float rows: one float64 chain per dimension in row order, 32 rows'
// values in flight (a lane per dimension).
template <class T>
__global__ __launch_bounds__(64) void pq_mean_kernel(const T* __restrict__ base, int dim, const int32_t* __restrict__ rows,
                                                     int64_t ns, long long* __restrict__ sums, float* __restrict__ mean) {
  const int j = blockIdx.x * kWave + threadIdx.x;
  if (j >= dim) return;
  if constexpr (sizeof(T) == 1) {
    const int64_t per = (ns + gridDim.y - 1) / gridDim.y, r0 = blockIdx.y * per, r1 = min(ns, r0 + per);
    int s = 0;  // (under 2^23 rows of 8 bits)
#pragma unroll 8
    for (int64_t i = r0; i < r1; i++) s += (int)base[(int64_t)rows[i] * dim + j];
    atomicAdd(reinterpret_cast<unsigned long long*>(sums + j), (unsigned long long)(long long)s);
  } else {
    double s = 0.0;
    int64_t i = 0;
    for (; i + 32 <= ns; i += 32) {
      float v[32];
#pragma unroll
      for (int u = 0; u < 32; u++) v[u] = base[(int64_t)rows[i + u] * dim + j];
#pragma unroll
      for (int u = 0; u < 32; u++) s += (double)v[u];
    }
    for (; i < ns; i++) s += (double)base[(int64_t)rows[i] * dim + j];
    mean[j] = (float)(s / (double)ns);
  }
}

__global__ void pq_mean_final_kernel(const long long* __restrict__ sums, int dim, int64_t ns, float* __restrict__ mean) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < dim) mean[j] = (float)((double)sums[j] / (double)ns);
}

// Sample row a pivot starts from, or restarts from when no row is nearest to it.
__device__ __forceinline__ int64_t pq_pick(uint64_t seed, uint64_t stream, uint64_t counter, int64_t ns) {
  return (int64_t)(rng_u64(seed, stream, counter) % (uint64_t)ns);
}

template <class T>
__global__ void pq_first_kernel(const T* __restrict__ base, int dim, const int32_t* __restrict__ rows, int64_t ns,
                                const float* __restrict__ centroid, const int32_t* __restrict__ chunk_off, int M,
                                uint64_t seed, float* __restrict__ pivots) {
  const int c = threadIdx.x, m = blockIdx.x;
  const int64_t row = rows[pq_pick(seed, 12 + (uint64_t)m, (uint64_t)c, ns)];
  for (int j = chunk_off[m]; j < chunk_off[m + 1]; j++) pivots[c * dim + j] = (float)base[row * dim + j] - centroid[j];
}

// Nearest pivot of chunk blockIdx.y for rows[i] (row i when rows is null), to
// out[chunk][i]: four rows per thread against each pivot of the chunk, read
// from LDS by every lane at once.  W is the chunk width rounded up: the missing
// dimensions are zero on both sides and add nothing to the distance's chain.
// (VALU-bound: 2 W + 3 instructions per row and pivot.  262,144 rows x 32
// chunks of 4: 0.6 ms of issue at one wave per 4 cycles.)
template <class T, int W>
__global__ __launch_bounds__(256) void pq_assign_kernel(const T* __restrict__ base, int dim,
                                                        const int32_t* __restrict__ rows, int64_t nrows,
                                                        const float* __restrict__ centroid,
                                                        const int32_t* __restrict__ chunk_off,
                                                        const float* __restrict__ pivots, uint8_t* __restrict__ out) {
  constexpr int kPer = 4;
  __shared__ __align__(16) float cen[kPivots * W];
  const int m = blockIdx.y, o = chunk_off[m], w = chunk_off[m + 1] - o;
  for (int i = threadIdx.x; i < kPivots * W; i += 256) {
    const int c = i / W, j = i % W;
    cen[i] = j < w ? pivots[c * dim + o + j] : 0.f;
  }
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.x * (256 * kPer) + threadIdx.x;
  float x[kPer][W], best[kPer];
  int at[kPer];
#pragma unroll
  for (int k = 0; k < kPer; k++) {
    const int64_t r = min(r0 + 256 * k, nrows - 1);
    const int64_t row = rows ? (int64_t)rows[r] : r;
#pragma unroll
    for (int j = 0; j < W; j++) x[k][j] = j < w ? (float)base[row * dim + o + j] - centroid[o + j] : 0.f;
    best[k] = __int_as_float(0x7f800000);
    at[k] = 0;
  }
#pragma unroll 4
  for (int c = 0; c < kPivots; c++) {
    float p[W];
#pragma unroll
    for (int j = 0; j < W; j++) p[j] = cen[c * W + j];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < W; j++) {
        const float d = x[k][j] - p[j];
        s = __fmaf_rn(d, d, s);
      }
      if (s < best[k]) {
        best[k] = s;
        at[k] = c;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < kPer; k++)
    if (r0 + 256 * k < nrows) out[(int64_t)m * nrows + r0 + 256 * k] = (uint8_t)at[k];
}

// Chunk-major codes [M][n] to rows [n][M].
__global__ __launch_bounds__(256) void pq_rows_of_codes_kernel(const uint8_t* __restrict__ planes, int64_t n, int M,
                                                               uint8_t* __restrict__ codes) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= n) return;
  int m = 0;
  for (; m + 4 <= M && M % 4 == 0; m += 4) {
    uint32_t v = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) v |= (uint32_t)planes[(int64_t)(m + e) * n + r] << (8 * e);
    *reinterpret_cast<uint32_t*>(codes + r * M + m) = v;
  }
  for (; m < M; m++) codes[r * M + m] = planes[(int64_t)m * n + r];
}

// Rows per pivot of one segment (blockIdx.x) of one chunk (blockIdx.y), to
// counts[chunk][pivot][segment].
__global__ __launch_bounds__(64) void pq_count_kernel(const uint8_t* __restrict__ assign, int64_t ns,
                                                      int32_t* __restrict__ counts) {
  __shared__ int32_t hist[kPivots];
  const int lane = lane_id();
  for (int i = lane; i < kPivots; i += kWave) hist[i] = 0;
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.x * kPqSegment, r1 = min(ns, r0 + kPqSegment);
  const uint8_t* const a = assign + (int64_t)blockIdx.y * ns;
#pragma unroll 4
  for (int64_t r = r0 + lane; r < r1; r += kWave) atomicAdd(&hist[a[r]], 1);
  __syncthreads();
  for (int c = lane; c < kPivots; c += kWave) counts[((int64_t)blockIdx.y * kPivots + c) * gridDim.x + blockIdx.x] = hist[c];
}

// counts to each (pivot, segment)'s first place in the chunk's list of rows,
// and each pivot's range: first[chunk][257].
__global__ __launch_bounds__(256) void pq_places_kernel(int32_t* __restrict__ counts, int segments,
                                                        int32_t* __restrict__ first) {
  __shared__ int32_t total[kPivots];
  const int c = threadIdx.x;
  int32_t* const mine = counts + ((int64_t)blockIdx.x * kPivots + c) * segments;
  int32_t sum = 0;
  for (int s = 0; s < segments; s++) sum += mine[s];
  total[c] = sum;
  __syncthreads();
  for (int off = 1; off < kPivots; off <<= 1) {
    const int32_t add = c >= off ? total[c - off] : 0;
    __syncthreads();
    total[c] += add;
    __syncthreads();
  }
  int32_t at = total[c] - sum;
  first[blockIdx.x * (kPivots + 1) + c] = at;
  if (c == kPivots - 1) first[blockIdx.x * (kPivots + 1) + kPivots] = total[c];
  for (int s = 0; s < segments; s++) {
    const int32_t v = mine[s];
    mine[s] = at;
    at += v;
  }
}

// The rows of one segment to their pivots' lists, in row order: one wave, 64
// rows at a time, a row's place being its pivot's next one plus its rank among
// the wave's rows of that pivot.
__global__ __launch_bounds__(64) void pq_partition_kernel(const uint8_t* __restrict__ assign, int64_t ns,
                                                          const int32_t* __restrict__ places,
                                                          int32_t* __restrict__ members) {
  __shared__ int32_t next[kPivots];
  const int lane = lane_id();
  for (int c = lane; c < kPivots; c += kWave)
    next[c] = places[((int64_t)blockIdx.y * kPivots + c) * gridDim.x + blockIdx.x];
  __syncthreads();
  const int64_t r0 = (int64_t)blockIdx.x * kPqSegment, r1 = min(ns, r0 + kPqSegment);
  const uint8_t* const a = assign + (int64_t)blockIdx.y * ns;
  int32_t* const out = members + (int64_t)blockIdx.y * ns;
  for (int64_t rb = r0; rb < r1; rb += kWave) {
    const int64_t r = rb + lane;
    const bool ok = r < r1;
    const int c = ok ? (int)a[r] : 0;
    uint64_t same = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 8; b++) {
      const uint64_t one = __ballot((c >> b) & 1);
      same &= (c >> b) & 1 ? one : ~one;
    }
    const int rank = (int)__popcll(same & ((1ull << lane) - 1));
    const int at = next[c];
    __syncthreads();
    if (ok) {
      out[at + rank] = (int32_t)r;
      if (rank == 0) next[c] = at + (int)__popcll(same);
    }
    __syncthreads();
  }
}

// New pivot (chunk blockIdx.y, number blockIdx.x): the mean of its rows, less
// the centroid, added in row order: 64 rows' values at a time in LDS, a lane
// per dimension adding them; a pivot without rows restarts from a sample row.
template <class T>
__global__ __launch_bounds__(64) void pq_update_kernel(const T* __restrict__ base, int dim,
                                                       const int32_t* __restrict__ rows, int64_t ns,
                                                       const float* __restrict__ centroid,
                                                       const int32_t* __restrict__ chunk_off,
                                                       const int32_t* __restrict__ first,
                                                       const int32_t* __restrict__ members, uint64_t seed, int it,
                                                       float* __restrict__ pivots) {
  __shared__ double val[16 * (kWave + 1)];  // [dimension][row], rows of 65
  const int lane = lane_id(), c = blockIdx.x, m = blockIdx.y;
  const int o = chunk_off[m], w = chunk_off[m + 1] - o;
  const int32_t b = first[m * (kPivots + 1) + c], e = first[m * (kPivots + 1) + c + 1];
  if (b == e) {
    const int64_t row = rows[pq_pick(seed, 400 + (uint64_t)m, (uint64_t)(it * 256 + c), ns)];
    if (lane < w) pivots[c * dim + o + lane] = (float)base[row * dim + o + lane] - centroid[o + lane];
    return;
  }
  const int32_t* const list = members + (int64_t)m * ns;
  double sum = 0.0;
  // the next 64 rows' numbers are in flight while these are added
  int64_t row = rows[list[min(b + lane, e - 1)]];
  for (int32_t i = b; i < e; i += kWave) {
    const int64_t cur = row;
    const int here = min((int)(e - i), kWave);
    row = rows[list[min(i + kWave + lane, e - 1)]];
    for (int j = 0; j < w; j++) val[j * (kWave + 1) + lane] = (double)(float)base[cur * dim + o + j] - (double)centroid[o + j];
    __syncthreads();
    if (lane < w) {
      const double* const v = val + lane * (kWave + 1);
      int k = 0;
      for (; k + 16 <= here; k += 16) {
        double t[16];
#pragma unroll
        for (int u = 0; u < 16; u++) t[u] = v[k + u];
#pragma unroll
        for (int u = 0; u < 16; u++) sum += t[u];
      }
      for (; k < here; k++) sum += v[k];
    }
    __syncthreads();
  }
  if (lane < w) pivots[c * dim + o + lane] = (float)(sum / (double)(e - b));
}

template <class T>
__global__ void mean_partial_kernel(const T* __restrict__ base, int64_t n, int dim, int64_t rows_per_block,
                                    double* __restrict__ partial) {
  const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
  const int64_t r1 = min(n, r0 + rows_per_block);
  for (int j = threadIdx.x; j < dim; j += blockDim.x) {
    // in row order, 16 rows' values in flight
    double s = 0.0;
    int64_t r = r0;
    for (; r + 16 <= r1; r += 16) {
      T v[16];
#pragma unroll
      for (int u = 0; u < 16; u++) v[u] = base[(r + u) * dim + j];
#pragma unroll
      for (int u = 0; u < 16; u++) s += (double)v[u];
    }
    for (; r < r1; r++) s += (double)base[r * dim + j];
    partial[(int64_t)blockIdx.x * dim + j] = s;
  }
}

template <class T>
__global__ void nearest_kernel(const T* __restrict__ base, int64_t n, int dim, const float* __restrict__ target,
                               unsigned long long* __restrict__ best) {
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
    float s = 0.f;
    for (int j = 0; j < dim; j++) {
      const float d = (float)base[r * dim + j] - target[j];
      s = __fmaf_rn(d, d, s);
    }
    atomicMin(best, ((unsigned long long)__float_as_uint(s) << 32) | (unsigned long long)r);
  }
}

// Node records: vector bytes, degree 0.
template <class T>
__global__ void init_pages_kernel(GLayout L, const T* __restrict__ base) {
  const int64_t ds4 = L.data_size / 4;
  const int64_t total = L.n * (ds4 + 1);
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t v = e / (ds4 + 1);
    const int64_t w = e - v * (ds4 + 1);
    uint32_t* rec = reinterpret_cast<uint32_t*>(node_rec(L, v));
    rec[w] = w < ds4 ? reinterpret_cast<const uint32_t*>(base + v * L.dim)[w] : 0u;
  }
}

// ---- RobustPrune -----------------------------------------------------------

constexpr int kMaxCand = 512;        // candidates before dedupe
constexpr int kPruneThreads = 256;   // one candidate each after it

template <class T>
__device__ __forceinline__ int32_t vec_norm(const uint32_t* a, int ds4) {
  if constexpr (sizeof(T) == 4) {
    return 0;
  } else if constexpr (std::is_signed<T>::value) {
    int32_t acc = 0;
    for (int w = 0; w < ds4; w++) acc = __builtin_amdgcn_sdot4((int)a[w], (int)a[w], acc, false);
    return acc;
  } else {
    uint32_t acc = 0;
    for (int w = 0; w < ds4; w++) acc = __builtin_amdgcn_udot4(a[w], a[w], acc, false);
    return (int32_t)acc;
  }
}

struct PruneArgs {
  GLayout L;
  int mode;                  // 0: forward (search record), 1: reverse (marked segments), 2: flush
  const int32_t* centers;    // modes 0 and 2: node ids
  int64_t num_centers;
  const int32_t* rec_ids;    // forward: [num_centers][rec_cap]
  const int32_t* hops;       // forward: [num_centers]
  int rec_cap;
  const uint64_t* pairs;     // reverse: sorted (target << 32 | source)
  const int32_t* heads;      // reverse: segment starts
  const int32_t* marks;      // reverse: indexes into heads of the segments to prune
  int64_t num_pairs;
  uint32_t* pend;            // [n][P] pending reverse edges (the slack beyond R)
  int32_t* pcnt;             // [n] pending count
  int P;
  float alpha;
  int cmax;                  // candidate capacity after dedupe
  int stride;                // LDS row stride in dwords: a multiple of 4, stride / 4 odd, >= the row
  int G;                     // lanes that fetch one row together (power of two, >= 4)
};

// LDS of one prune: keys [cmax] u64, norms [cmax] i32, the centre row and cmax
// candidate rows at `stride` dwords (16-byte aligned), the output list, then the
// greedy loop's masks and the compaction's counts.  The candidate rows double
// as the fetch phase's (id, distance) table and the sorted keys.  rule: the
// bytes that decide cmax (build_gpu_t).
struct PruneLds {
  int norms_off, cvec_off, vecs_off, outl_off, masks_off, rule, total;
};
__host__ __device__ inline PruneLds prune_lds_plan(int cmax, int stride, int R) {
  PruneLds p;
  p.norms_off = 8 * cmax;
  p.cvec_off = (12 * cmax + 15) & ~15;
  p.vecs_off = p.cvec_off + 4 * stride;
  const int rows = 4 * cmax * stride;
  p.rule = p.vecs_off + (rows > 8 * kMaxCand ? rows : 8 * kMaxCand) + 4 * R;
  p.outl_off = p.vecs_off + (rows > 16 * kMaxCand ? rows : 16 * kMaxCand);
  p.masks_off = (p.outl_off + 4 * R + 7) & ~7;
  p.total = p.masks_off + 2 * (kPruneThreads / kWave) * (8 + 4);
  return p;
}

// Partial squared distance between the centre words c and row words x (8-bit
// data: x.x - 2 c.x, the centre's norm added once per row; float: (c - x)^2).
template <class T>
struct RowAcc {
  using type = typename std::conditional<sizeof(T) == 4, float, int32_t>::type;
  __device__ static __forceinline__ type add(type acc, uint32_t c, uint32_t x) {
    if constexpr (sizeof(T) == 4) {
      const float d = __uint_as_float(c) - __uint_as_float(x);
      return __fmaf_rn(d, d, acc);
    } else if constexpr (std::is_signed<T>::value) {
      return acc + __builtin_amdgcn_sdot4((int)x, (int)x, 0, false) - 2 * __builtin_amdgcn_sdot4((int)c, (int)x, 0, false);
    } else {
      return acc + (int32_t)__builtin_amdgcn_udot4(x, x, 0u, false) -
             2 * (int32_t)__builtin_amdgcn_udot4(c, x, 0u, false);
    }
  }
  __device__ static __forceinline__ type norm_add(type acc, uint32_t x) {
    if constexpr (sizeof(T) == 4) return acc;
    else if constexpr (std::is_signed<T>::value) return acc + __builtin_amdgcn_sdot4((int)x, (int)x, 0, false);
    else return acc + (int32_t)__builtin_amdgcn_udot4(x, x, 0u, false);
  }
};

template <class V>
__device__ __forceinline__ V group_sum(V v, int G) {
  for (int off = G >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// Squared distance of LDS row a (q4 pieces of 16 bytes, the same for every
// lane) and this lane's row, held in registers when KR pieces hold it (b), else
// in LDS (bl).  Words past the row are zero in both.  Float: the dimension
// order of a sequential loop; 8-bit data: exact integers from the dot product
// and the norms.
template <class T, int KR>
__device__ __forceinline__ float row_dist(const uint32_t* a, const uint4 (&b)[KR > 0 ? KR : 1], const uint32_t* bl,
                                          int q4, int32_t na, int32_t nb) {
  const uint4* a4 = reinterpret_cast<const uint4*>(a);
  const uint4* b4 = reinterpret_cast<const uint4*>(bl);
  float s = 0.f;
  int32_t acc = 0;
  auto add = [&](const uint4& x, const uint4& y) {
    if constexpr (sizeof(T) == 4) {
      float d = __uint_as_float(x.x) - __uint_as_float(y.x);
      s = __fmaf_rn(d, d, s);
      d = __uint_as_float(x.y) - __uint_as_float(y.y);
      s = __fmaf_rn(d, d, s);
      d = __uint_as_float(x.z) - __uint_as_float(y.z);
      s = __fmaf_rn(d, d, s);
      d = __uint_as_float(x.w) - __uint_as_float(y.w);
      s = __fmaf_rn(d, d, s);
    } else if constexpr (std::is_signed<T>::value) {
      acc = __builtin_amdgcn_sdot4((int)x.x, (int)y.x, acc, false);
      acc = __builtin_amdgcn_sdot4((int)x.y, (int)y.y, acc, false);
      acc = __builtin_amdgcn_sdot4((int)x.z, (int)y.z, acc, false);
      acc = __builtin_amdgcn_sdot4((int)x.w, (int)y.w, acc, false);
    } else {
      acc = (int32_t)__builtin_amdgcn_udot4(x.x, y.x, (uint32_t)acc, false);
      acc = (int32_t)__builtin_amdgcn_udot4(x.y, y.y, (uint32_t)acc, false);
      acc = (int32_t)__builtin_amdgcn_udot4(x.z, y.z, (uint32_t)acc, false);
      acc = (int32_t)__builtin_amdgcn_udot4(x.w, y.w, (uint32_t)acc, false);
    }
  };
  if constexpr (KR > 0) {
#pragma unroll
    for (int q = 0; q < KR; q++)
      if (q < q4) add(a4[q], b[q]);
  } else {
    for (int q = 0; q < q4; q++) add(a4[q], b4[q]);
  }
  if constexpr (sizeof(T) == 4) return s;
  // (64-bit: rows of more than 32,768 bytes do not exist, sums of 8-bit squares fit 32)
  else return (float)((int64_t)na + (int64_t)nb - 2 * (int64_t)acc);
}

// One workgroup of four waves per centre: forward prunes (mode 0: the nodes
// expanded by the centre's build search, then its current list and pending
// edges), reverse prunes of marked segments (mode 1: current list, pending
// edges, then the segment's incoming sources) and the flush of pending edges
// (mode 2: list and pending).  Per centre: exact distances to the candidates
// (candidate i -> node id, or -1 to skip), sort by (distance, id), dedupe, then
// the list is the candidates themselves when they fit in R, else
// RobustPrune(alpha, R) over them.  The centre's pending edges are cleared: they
// are among the candidates.
//   * Candidate rows are fetched cooperatively: G lanes per row, lane p of a row
//     reading words p, p + G, ... (a contiguous G-word run per load
//     instruction), 64 / G rows per instruction and two instructions' rows in
//     flight per wave.
//   * Sorted by rank: a thread counts the keys below its own; equal keys are
//     one node listed twice and share a place, whose gap the compaction closes.
//   * A thread owns a candidate (cmax <= 256), its row in registers where KR
//     16-byte pieces hold it: an accepted row is read from LDS by every lane at
//     once, so a step of the greedy loop is one row of arithmetic and a barrier.
// What bounds it: the candidate rows in LDS (37 KB of 128-byte rows, 74 KB of
// 96 floats) allow four or two centres per CU, which with one wave per centre
// left the SIMDs at one or half a wave each, waiting on LDS and on each row's
// chain.  All prunes of a build of 250,000 x 128 uint8 (R = 64, L = 100): 84 ms
// with one wave per centre, 40 ms; 100,003 x 96 float: 150 and 63 ms.
template <class T, int KR>
__global__ __launch_bounds__(kPruneThreads) void prune_kernel(PruneArgs a) {
  using Acc = RowAcc<T>;
  using AccT = typename Acc::type;
  extern __shared__ __align__(16) char smem[];
  const GLayout& L = a.L;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  constexpr int kWaves = kPruneThreads / kWave;
  const int ds4 = (int)(L.data_size / 4);
  const PruneLds pl = prune_lds_plan(a.cmax, a.stride, L.R);
  uint64_t* const keys = reinterpret_cast<uint64_t*>(smem);
  int32_t* const norms = reinterpret_cast<int32_t*>(smem + pl.norms_off);
  uint32_t* const cvec = reinterpret_cast<uint32_t*>(smem + pl.cvec_off);
  uint32_t* const vecs = reinterpret_cast<uint32_t*>(smem + pl.vecs_off);
  uint32_t* const outl = reinterpret_cast<uint32_t*>(smem + pl.outl_off);
  uint64_t* const masks = reinterpret_cast<uint64_t*>(smem + pl.masks_off);  // [2][kWaves]
  int32_t* const counts = reinterpret_cast<int32_t*>(masks + 2 * kWaves);    // [2 * kWaves]
  // before the rows are staged, their place holds the fetch table and the sorted keys
  uint32_t* const cand_id = vecs;             // [kMaxCand] ids (~0u: none)
  uint32_t* const cand_d = vecs + kMaxCand;   // [kMaxCand] distance bits (~0u: none)
  uint64_t* const sorted = reinterpret_cast<uint64_t*>(vecs + 2 * kMaxCand);  // [kMaxCand]
  const int S = a.stride;
  const int w4 = (ds4 + 3) & ~3;  // row words row_dist reads (zero past ds4)
  const int G = a.G, rpr = kWave / G, p = lane & (G - 1), sub = lane / G;
  const int kk = (ds4 + G - 1) / G;  // words per lane per row
  for (int64_t ci = blockIdx.x; ci < a.num_centers; ci += gridDim.x) {
    int64_t center;
    int64_t seg_begin = 0, seg_end = 0;
    if (a.mode != 1) {
      center = a.centers[ci];
    } else {
      seg_begin = a.heads[a.marks[ci]];
      center = (int64_t)(a.pairs[seg_begin] >> 32);
      // pairs are sorted by target, so the segment is the run of pairs whose
      // target matches: advance by whole waves, then to the first miss
      seg_end = seg_begin;
      while (true) {
        const int64_t q = seg_end + lane;
        const bool same = q < a.num_pairs && (int64_t)(a.pairs[q] >> 32) == center;
        const uint64_t mk = __ballot(same);
        if (mk == ~0ull) {
          seg_end += kWave;
          continue;
        }
        seg_end += __ffsll((long long)~mk) - 1;
        break;
      }
    }
    uint32_t* const crec = reinterpret_cast<uint32_t*>(node_rec(L, center));
    uint32_t* const cnb = crec + ds4;
    for (int w = tid; w < a.stride; w += kPruneThreads) cvec[w] = w < ds4 ? crec[w] : 0u;
    const int cdeg = (int)cnb[0];
    const int pc = a.pcnt[center];
    const uint32_t* const pend = a.pend + center * a.P;
    // candidate i: [lead candidates][current list][pending][trailing sources]
    int lead = 0, tail = 0;
    if (a.mode == 0) lead = min(a.hops[ci], a.rec_cap);
    if (a.mode == 1) tail = (int)min<int64_t>(seg_end - seg_begin, kMaxCand - L.R - a.P);
    const int C0 = min(lead + cdeg + pc + tail, kMaxCand);
    auto cand = [&](int i) -> int64_t {
      int64_t id;
      if (i < lead) id = (int64_t)a.rec_ids[ci * a.rec_cap + i];
      else if (i < lead + cdeg) id = (int64_t)cnb[1 + (i - lead)];
      else if (i < lead + cdeg + pc) id = (int64_t)pend[i - lead - cdeg];
      else id = (int64_t)(uint32_t)a.pairs[seg_begin + (i - lead - cdeg - pc)];
      return id == center ? -1 : id;
    };
    __syncthreads();
    const int32_t cnorm = vec_norm<T>(cvec, ds4);

    // ---- distances centre -> candidates, rows fetched by groups of G lanes
    for (int r0 = wave * 2 * rpr; r0 < C0; r0 += kWaves * 2 * rpr) {
      const int i0 = r0 + sub, i1 = r0 + rpr + sub;
      const int64_t id0 = i0 < C0 ? cand(i0) : -1;
      const int64_t id1 = i1 < C0 ? cand(i1) : -1;
      const uint32_t* x0 = reinterpret_cast<const uint32_t*>(node_rec(L, id0 >= 0 ? id0 : center));
      const uint32_t* x1 = reinterpret_cast<const uint32_t*>(node_rec(L, id1 >= 0 ? id1 : center));
      AccT s0 = 0, s1 = 0;
      for (int k0 = 0; k0 < kk; k0 += 4) {
        uint32_t v0[4], v1[4], cw[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const int w = p + G * (k0 + t);
          const bool ok = k0 + t < kk && w < ds4;
          v0[t] = ok ? x0[w] : 0u;
          v1[t] = ok ? x1[w] : 0u;
          cw[t] = ok ? cvec[w] : 0u;
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
          s0 = Acc::add(s0, cw[t], v0[t]);
          s1 = Acc::add(s1, cw[t], v1[t]);
        }
      }
      s0 = group_sum(s0, G);
      s1 = group_sum(s1, G);
      if (p == 0) {
        float d0, d1;
        if constexpr (sizeof(T) == 4) {
          d0 = s0;
          d1 = s1;
        } else {
          d0 = (float)(cnorm + s0);
          d1 = (float)(cnorm + s1);
        }
        if (i0 < C0) {
          cand_id[i0] = id0 >= 0 ? (uint32_t)id0 : ~0u;
          cand_d[i0] = id0 >= 0 ? __float_as_uint(d0) : ~0u;
        }
        if (i1 < C0) {
          cand_id[i1] = id1 >= 0 ? (uint32_t)id1 : ~0u;
          cand_d[i1] = id1 >= 0 ? __float_as_uint(d1) : ~0u;
        }
      }
    }
    // (the rank loop reads the table four keys at a time)
    if (tid < 4 && C0 + tid < kMaxCand && C0 + tid < ((C0 + 3) & ~3)) cand_id[C0 + tid] = cand_d[C0 + tid] = ~0u;
    for (int i = tid; i < C0; i += kPruneThreads) sorted[i] = kPadKey;
    __syncthreads();
    for (int i = tid; i < C0; i += kPruneThreads) {
      const uint64_t key = ((uint64_t)cand_d[i] << 32) | cand_id[i];
      int rank = 0;
      for (int k = 0; k < C0; k += 4) {
        const uint4 kd = *reinterpret_cast<const uint4*>(cand_d + k);
        const uint4 ki = *reinterpret_cast<const uint4*>(cand_id + k);
        rank += (((uint64_t)kd.x << 32) | ki.x) < key ? 1 : 0;
        rank += (((uint64_t)kd.y << 32) | ki.y) < key ? 1 : 0;
        rank += (((uint64_t)kd.z << 32) | ki.z) < key ? 1 : 0;
        rank += (((uint64_t)kd.w << 32) | ki.w) < key ? 1 : 0;
      }
      if (key != kPadKey) sorted[rank] = key;
    }
    __syncthreads();
    // compact: places 0..255 by the four waves, then 256..511
    uint64_t kept[2];
    uint64_t in[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int i = s * kPruneThreads + tid;
      in[s] = i < C0 ? sorted[i] : kPadKey;
      kept[s] = __ballot(in[s] != kPadKey);
      if (lane == 0) counts[s * kWaves + wave] = (int)__popcll(kept[s]);
    }
    __syncthreads();
    int C = 0;
#pragma unroll
    for (int s = 0; s < 2; s++) {
      for (int w = 0; w < kWaves; w++) {
        if (w == wave && in[s] != kPadKey) {
          const int pos = C + (int)__popcll(kept[s] & ((1ull << lane) - 1));
          if (pos < a.cmax) keys[pos] = in[s];
        }
        C += counts[s * kWaves + w];
      }
    }
    C = min(C, a.cmax);
    __syncthreads();  // the table and the sorted keys are overwritten by the rows below

    int out_n = 0;
    if (C <= L.R) {
      for (int i = tid; i < C; i += kPruneThreads) cnb[1 + i] = (uint32_t)keys[i];
      out_n = C;
    } else {
      // stage the candidate rows (and their norms) in LDS, fetched as above
      for (int r0 = wave * 2 * rpr; r0 < C; r0 += kWaves * 2 * rpr) {
        const int i0 = r0 + sub, i1 = r0 + rpr + sub;
        const int64_t id0 = i0 < C ? (int64_t)(uint32_t)keys[i0] : center;
        const int64_t id1 = i1 < C ? (int64_t)(uint32_t)keys[i1] : center;
        const uint32_t* x0 = reinterpret_cast<const uint32_t*>(node_rec(L, id0));
        const uint32_t* x1 = reinterpret_cast<const uint32_t*>(node_rec(L, id1));
        AccT n0 = 0, n1 = 0;
        for (int k0 = 0; k0 < kk; k0 += 4) {
          uint32_t v0[4], v1[4];
#pragma unroll
          for (int t = 0; t < 4; t++) {
            const int w = p + G * (k0 + t);
            const bool ok = k0 + t < kk && w < ds4;
            v0[t] = ok ? x0[w] : 0u;
            v1[t] = ok ? x1[w] : 0u;
          }
#pragma unroll
          for (int t = 0; t < 4; t++) {
            const int w = p + G * (k0 + t);
            if (k0 + t < kk && w < w4) {
              if (i0 < C) vecs[i0 * S + w] = v0[t];
              if (i1 < C) vecs[i1 * S + w] = v1[t];
            }
            n0 = Acc::norm_add(n0, v0[t]);
            n1 = Acc::norm_add(n1, v1[t]);
          }
        }
        if constexpr (sizeof(T) != 4) {
          n0 = group_sum(n0, G);
          n1 = group_sum(n1, G);
          if (p == 0) {
            if (i0 < C) norms[i0] = n0;
            if (i1 < C) norms[i1] = n1;
          }
        }
      }
      __syncthreads();
      const int q4 = w4 / 4;
      bool alive = tid < C;
      const int j = alive ? tid : 0;
      const float dpj = __uint_as_float((uint32_t)(keys[j] >> 32));
      const int32_t nj = sizeof(T) == 4 ? 0 : norms[j];
      uint4 row[KR > 0 ? KR : 1];
      if constexpr (KR > 0) {
#pragma unroll
        for (int q = 0; q < KR; q++)
          if (q < q4) row[q] = reinterpret_cast<const uint4*>(vecs + j * S)[q];
      }
      int i = 0;  // the first candidate is always taken
      for (int buf = 0;; buf ^= 1) {
        if (tid == 0) outl[out_n] = (uint32_t)keys[i];
        out_n++;
        if (out_n == L.R) break;
        alive = alive && tid > i;
        if (alive) {
          const float dij =
              row_dist<T, KR>(vecs + i * S, row, vecs + j * S, q4, sizeof(T) == 4 ? 0 : norms[i], nj);
          if (a.alpha * dij <= dpj) alive = false;
        }
        const uint64_t m = __ballot(alive);
        if (lane == 0) masks[buf * kWaves + wave] = m;
        __syncthreads();
        i = -1;
#pragma unroll
        for (int w = kWaves - 1; w >= 0; w--) {
          const uint64_t mw = masks[buf * kWaves + w];
          if (mw) i = w * kWave + __ffsll((long long)mw) - 1;
        }
        if (i < 0) break;
      }
      __syncthreads();
      for (int t = tid; t < out_n; t += kPruneThreads) cnb[1 + t] = outl[t];
    }
    if (tid == 0) {
      cnb[0] = (uint32_t)out_n;
      a.pcnt[center] = 0;
    }
    __syncthreads();
  }
}

// Reverse edges of a batch, one wave per target (a run of sorted pairs):
// sources already among the target's list or pending edges are dropped; the
// rest are appended to the list while it has room, then to the pending edges
// (up to P, DiskANN's graph slack: a list may hold 1.3 R before it is pruned);
// a target whose new edges fit neither is marked for a reverse prune.
__global__ __launch_bounds__(64) void reverse_insert_kernel(GLayout L, const uint64_t* __restrict__ pairs,
                                                            const int32_t* __restrict__ heads, int64_t nheads,
                                                            int64_t npairs, uint32_t* __restrict__ pend,
                                                            int32_t* __restrict__ pcnt, int P,
                                                            int32_t* __restrict__ marks,
                                                            unsigned int* __restrict__ nmarks) {
  const int lane = lane_id();
  for (int64_t hi = blockIdx.x; hi < nheads; hi += gridDim.x) {
    const int64_t b = heads[hi];
    const uint32_t t = (uint32_t)(pairs[b] >> 32);
    uint32_t* nb = reinterpret_cast<uint32_t*>(node_rec(L, t) + L.data_size);
    const int cdeg = (int)nb[0];
    const int pc = pcnt[t];
    // the list, two slots per lane (R <= 128), and the pending edges (P <= 64)
    const uint32_t mine0 = lane < cdeg ? nb[1 + lane] : ~0u;
    const uint32_t mine1 = lane + kWave < cdeg ? nb[1 + kWave + lane] : ~0u;
    const uint32_t pmine = lane < pc ? pend[(int64_t)t * P + lane] : ~0u;
    const int c0 = min(cdeg, kWave);
    // new sources, counted over the whole run, 64 pairs at a time
    auto fresh = [&](int64_t q, uint32_t& src) -> bool {
      if (q >= npairs || (uint32_t)(pairs[q] >> 32) != t) return false;
      src = (uint32_t)pairs[q];
      bool dup = false;
      for (int k = 0; k < c0; k++) dup |= src == (uint32_t)__builtin_amdgcn_readlane((int)mine0, k);
      for (int k = kWave; k < cdeg; k++) dup |= src == (uint32_t)__builtin_amdgcn_readlane((int)mine1, k - kWave);
      for (int k = 0; k < pc; k++) dup |= src == (uint32_t)__builtin_amdgcn_readlane((int)pmine, k);
      return !dup;
    };
    int u = 0;
    int64_t q0 = b;
    while (true) {
      uint32_t src = 0;
      const bool in_run = q0 + lane < npairs && (uint32_t)(pairs[q0 + lane] >> 32) == t;
      const bool f = in_run && fresh(q0 + lane, src);
      u += __popcll(__ballot(f));
      if (__ballot(in_run) != ~0ull) break;
      q0 += kWave;
    }
    const int room = L.R - cdeg;
    if (u > room + (P - pc)) {
      if (lane == 0) marks[atomicAdd(nmarks, 1u)] = (int32_t)hi;
      continue;
    }
    if (u == 0) continue;
    int placed = 0;
    q0 = b;
    while (true) {
      uint32_t src = 0;
      const bool in_run = q0 + lane < npairs && (uint32_t)(pairs[q0 + lane] >> 32) == t;
      const bool f = in_run && fresh(q0 + lane, src);
      const uint64_t fm = __ballot(f);
      if (f) {
        const int r = placed + __popcll(fm & ((lane == 0) ? 0ull : (~0ull >> (64 - lane))));
        if (r < room) nb[1 + cdeg + r] = src;
        else pend[(int64_t)t * P + pc + (r - room)] = src;
      }
      placed += __popcll(fm);
      if (__ballot(in_run) != ~0ull) break;
      q0 += kWave;
    }
    if (lane == 0) {
      const int to_list = min(u, room);
      nb[0] = (uint32_t)(cdeg + to_list);
      pcnt[t] = pc + (u - to_list);
    }
  }
}

// Nodes with pending edges, for the flush at the end of a pass.
__global__ void pending_nodes_kernel(const int32_t* __restrict__ pcnt, int64_t n, int32_t* __restrict__ out,
                                     unsigned int* __restrict__ count) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x)
    if (pcnt[v] > 0) out[atomicAdd(count, 1u)] = (int32_t)v;
}

// Reverse-edge pairs (target << 32 | source) of every new list of the batch.
__global__ void emit_pairs_kernel(GLayout L, const int32_t* __restrict__ centers, int64_t nc,
                                  uint64_t* __restrict__ pairs, unsigned long long* __restrict__ count) {
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nc * L.R;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t ci = e / L.R;
    const int j = (int)(e - ci * L.R);
    const int64_t p = centers[ci];
    const uint32_t* nb = reinterpret_cast<const uint32_t*>(node_rec(L, p) + L.data_size);
    uint64_t key = kPadKey;
    if (j < (int)nb[0]) {
      key = ((uint64_t)nb[1 + j] << 32) | (uint64_t)(uint32_t)p;
      atomicAdd(count, 1ull);
    }
    pairs[e] = key;
  }
}

__global__ void heads_kernel(const uint64_t* __restrict__ pairs, int64_t n, int32_t* __restrict__ heads,
                             unsigned int* __restrict__ nheads) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    if (i == 0 || (pairs[i] >> 32) != (pairs[i - 1] >> 32)) heads[atomicAdd(nheads, 1u)] = (int32_t)i;
  }
}

int grid_of(int64_t work, int block) {
  return (int)std::max<int64_t>(1, std::min<int64_t>((work + block - 1) / block, 1 << 20));
}

// ---- host driver ------------------------------------------------------------

struct DevBuf {
  void* p = nullptr;
  ~DevBuf() {
    if (p) (void)hipFree(p);
  }
  template <class U>
  U* as() const {
    return static_cast<U*>(p);
  }
};

// Launches pq_assign_kernel for the widest chunk's width.
template <class T>
void pq_assign(const T* d_base, int dim, const int32_t* d_rows, int64_t nrows, const float* d_cent,
               const int32_t* d_off, int M, int maxw, const float* d_piv, uint8_t* d_out, hipStream_t st) {
  const dim3 grid((unsigned)((nrows + 1023) / 1024), (unsigned)M);
#define QV_ASSIGN(W)                                                                                              \
  hipLaunchKernelGGL((pq_assign_kernel<T, W>), grid, dim3(256), 0, st, d_base, dim, d_rows, nrows, d_cent, d_off, \
                     d_piv, d_out)
  if (maxw <= 2) QV_ASSIGN(2);
  else if (maxw <= 4) QV_ASSIGN(4);
  else if (maxw <= 8) QV_ASSIGN(8);
  else QV_ASSIGN(16);
#undef QV_ASSIGN
  HIP_OK(hipGetLastError());
}

// PQ tables (t, without the codes) and the codes of all n rows, which stay on
// the device: d_codes [n][M].
template <class T>
void train_pq_gpu(const T* d_base, int64_t n, int dim, const qv_build_params& prm, PQTables& t, uint8_t* d_codes,
                  hipStream_t st) {
  const int M = prm.num_chunks;
  t.dim = dim;
  t.num_chunks = M;
  t.num_pts = n;
  t.chunk_offsets.resize((size_t)M + 1);
  for (int i = 0; i <= M; i++) t.chunk_offsets[(size_t)i] = (int32_t)(((int64_t)i * dim) / M);
  for (int i = 0; i < M; i++)
    if (t.chunk_offsets[(size_t)i + 1] - t.chunk_offsets[(size_t)i] > 16)
      fail(QV_EUNSUPPORTED, "PQ chunks wider than 16 dimensions");
  t.chunk_id.assign((size_t)dim, 0);
  for (int i = 0; i < M; i++)
    for (int j = t.chunk_offsets[(size_t)i]; j < t.chunk_offsets[(size_t)i + 1]; j++) t.chunk_id[(size_t)j] = i;
  const int maxw = (dim + M - 1) / M;

  const int64_t ns = std::min<int64_t>(n, prm.pq_train_max > 0 ? prm.pq_train_max : 262144);
  const int segments = (int)((ns + kPqSegment - 1) / kPqSegment);
  DevBuf rows, off, cent, piv, sums, assign, counts, first, members, planes;
  HIP_OK(hipMalloc(&rows.p, sizeof(int32_t) * (size_t)ns));
  HIP_OK(hipMalloc(&off.p, sizeof(int32_t) * (size_t)(M + 1)));
  HIP_OK(hipMalloc(&cent.p, sizeof(float) * (size_t)dim));
  HIP_OK(hipMalloc(&piv.p, sizeof(float) * (size_t)kNumPivots * dim));
  HIP_OK(hipMalloc(&sums.p, sizeof(long long) * (size_t)dim));
  HIP_OK(hipMalloc(&assign.p, (size_t)ns * M));
  HIP_OK(hipMalloc(&counts.p, sizeof(int32_t) * (size_t)M * kNumPivots * segments));
  HIP_OK(hipMalloc(&first.p, sizeof(int32_t) * (size_t)M * (kNumPivots + 1)));
  HIP_OK(hipMalloc(&members.p, sizeof(int32_t) * (size_t)ns * M));
  HIP_OK(hipMalloc(&planes.p, (size_t)n * M));
  int32_t* const d_rows = rows.as<int32_t>();
  const int32_t* const d_off = off.as<int32_t>();
  float *const d_cent = cent.as<float>(), *const d_piv = piv.as<float>();
  HIP_OK(hipMemcpyAsync(off.p, t.chunk_offsets.data(), sizeof(int32_t) * (size_t)(M + 1), hipMemcpyHostToDevice, st));
  HIP_OK(hipMemsetAsync(sums.p, 0, sizeof(long long) * (size_t)dim, st));
  hipLaunchKernelGGL(pq_rows_kernel, dim3((unsigned)((ns + 255) / 256)), dim3(256), 0, st, n, ns, d_rows);
  HIP_OK(hipGetLastError());
  const unsigned dim_blocks = (unsigned)((dim + kWave - 1) / kWave);
  hipLaunchKernelGGL(pq_mean_kernel<T>, dim3(dim_blocks, sizeof(T) == 1 ? 256 : 1), dim3(64), 0, st, d_base, dim, d_rows,
                     ns, sums.as<long long>(), d_cent);
  HIP_OK(hipGetLastError());
  if (sizeof(T) == 1) {
    hipLaunchKernelGGL(pq_mean_final_kernel, dim3(dim_blocks), dim3(64), 0, st, sums.as<long long>(), dim, ns, d_cent);
    HIP_OK(hipGetLastError());
  }
  hipLaunchKernelGGL(pq_first_kernel<T>, dim3((unsigned)M), dim3(kNumPivots), 0, st, d_base, dim, d_rows, ns, d_cent,
                     d_off, M, prm.seed, d_piv);
  HIP_OK(hipGetLastError());
  for (int it = 0; it < std::max(1, prm.kmeans_iters); it++) {
    pq_assign<T>(d_base, dim, d_rows, ns, d_cent, d_off, M, maxw, d_piv, assign.as<uint8_t>(), st);
    const dim3 seg((unsigned)segments, (unsigned)M);
    hipLaunchKernelGGL(pq_count_kernel, seg, dim3(64), 0, st, assign.as<uint8_t>(), ns, counts.as<int32_t>());
    HIP_OK(hipGetLastError());
    hipLaunchKernelGGL(pq_places_kernel, dim3((unsigned)M), dim3(kNumPivots), 0, st, counts.as<int32_t>(), segments,
                       first.as<int32_t>());
    HIP_OK(hipGetLastError());
    hipLaunchKernelGGL(pq_partition_kernel, seg, dim3(64), 0, st, assign.as<uint8_t>(), ns, counts.as<int32_t>(),
                       members.as<int32_t>());
    HIP_OK(hipGetLastError());
    hipLaunchKernelGGL(pq_update_kernel<T>, dim3(kNumPivots, (unsigned)M), dim3(64), 0, st, d_base, dim, d_rows, ns,
                       d_cent, d_off, first.as<int32_t>(), members.as<int32_t>(), prm.seed, it, d_piv);
    HIP_OK(hipGetLastError());
  }
  pq_assign<T>(d_base, dim, nullptr, n, d_cent, d_off, M, maxw, d_piv, planes.as<uint8_t>(), st);
  hipLaunchKernelGGL(pq_rows_of_codes_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, planes.as<uint8_t>(),
                     n, M, d_codes);
  HIP_OK(hipGetLastError());
  t.centroid.resize((size_t)dim);
  t.pivots.resize((size_t)kNumPivots * dim);
  HIP_OK(hipMemcpyAsync(t.centroid.data(), d_cent, sizeof(float) * (size_t)dim, hipMemcpyDeviceToHost, st));
  HIP_OK(hipMemcpyAsync(t.pivots.data(), d_piv, sizeof(float) * t.pivots.size(), hipMemcpyDeviceToHost, st));
  HIP_OK(hipStreamSynchronize(st));
  t.pivots_t.assign((size_t)dim * kNumPivots, 0.f);
  for (int c = 0; c < kNumPivots; c++)
    for (int j = 0; j < dim; j++) t.pivots_t[(size_t)j * kNumPivots + c] = t.pivots[(size_t)c * dim + j];
}

template <class T>
int64_t medoid_gpu(const T* d_base, int64_t n, int dim, hipStream_t st) {
  const int64_t rpb = 4096;
  const int64_t nblk = (n + rpb - 1) / rpb;
  double* d_part = nullptr;
  HIP_OK(hipMalloc(&d_part, sizeof(double) * (size_t)(nblk * dim)));
  hipLaunchKernelGGL(mean_partial_kernel<T>, dim3((unsigned)nblk), dim3(128), 0, st, d_base, n, dim, rpb, d_part);
  HIP_OK(hipGetLastError());
  std::vector<double> part((size_t)(nblk * dim));
  HIP_OK(hipMemcpyAsync(part.data(), d_part, sizeof(double) * part.size(), hipMemcpyDeviceToHost, st));
  HIP_OK(hipStreamSynchronize(st));
  hipFree(d_part);
  std::vector<float> mean((size_t)dim);
  for (int j = 0; j < dim; j++) {
    double s = 0.0;
    for (int64_t b = 0; b < nblk; b++) s += part[(size_t)(b * dim + j)];
    mean[(size_t)j] = (float)(s / (double)n);
  }
  float* d_mean = nullptr;
  unsigned long long* d_best = nullptr;
  HIP_OK(hipMalloc(&d_mean, sizeof(float) * (size_t)dim));
  HIP_OK(hipMalloc(&d_best, sizeof(unsigned long long)));
  HIP_OK(hipMemcpy(d_mean, mean.data(), sizeof(float) * (size_t)dim, hipMemcpyHostToDevice));
  HIP_OK(hipMemsetAsync(d_best, 0xff, sizeof(unsigned long long), st));
  hipLaunchKernelGGL(nearest_kernel<T>, dim3((unsigned)grid_of(n, 256)), dim3(256), 0, st, d_base, n, dim, d_mean,
                     d_best);
  HIP_OK(hipGetLastError());
  unsigned long long best = 0;
  HIP_OK(hipMemcpyAsync(&best, d_best, sizeof(best), hipMemcpyDeviceToHost, st));
  HIP_OK(hipStreamSynchronize(st));
  hipFree(d_mean);
  hipFree(d_best);
  return (int64_t)(best & 0xffffffffull);
}

template <class T>
qv_index* build_gpu_t(const T* d_base, int dtype, int64_t n, int dim, const qv_build_params& prm, int device) {
  hipStream_t st;
  HIP_OK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  std::unique_ptr<std::remove_pointer<hipStream_t>::type, void (*)(hipStream_t)> sg(
      st, [](hipStream_t s) { (void)hipStreamDestroy(s); });
  const auto t_start = std::chrono::steady_clock::now();

  if (prm.num_chunks <= 0 || prm.num_chunks > dim) fail(QV_EINVAL, "num_chunks must be in [1, dim]");
  PQTables pq;
  DevBuf pages, codes;
  HIP_OK(hipMalloc(&codes.p, std::max<size_t>((size_t)n * prm.num_chunks, 64)));
  train_pq_gpu<T>(d_base, n, dim, prm, pq, codes.as<uint8_t>(), st);
  const int64_t medoid = medoid_gpu<T>(d_base, n, dim, st);

  Layout lay;
  lay.data_type = dtype;
  lay.num_data = n;
  lay.num_dims = dim;
  lay.max_m0 = prm.R;
  lay.enter_point = medoid;
  lay.data_size = (int64_t)dim * (int64_t)sizeof(T);
  lay.node_size = lay.data_size + 4 + 4ll * prm.R;
  if (lay.node_size > kPageSize) fail(QV_EINVAL, "node record exceeds one 4 KB page");
  if (lay.data_size % 4) fail(QV_EUNSUPPORTED, "vector bytes must be a multiple of 4");
  lay.nodes_per_page = kPageSize / lay.node_size;
  lay.num_pages = (n + lay.nodes_per_page - 1) / lay.nodes_per_page;

  HIP_OK(hipMalloc(&pages.p, (size_t)(lay.num_pages * kPageSize)));
  HIP_OK(hipMemsetAsync(pages.p, 0, (size_t)(lay.num_pages * kPageSize), st));
  GLayout G{pages.as<uint8_t>(), n, lay.nodes_per_page, lay.node_size, lay.data_size, dim, prm.R};
  hipLaunchKernelGGL(init_pages_kernel<T>, dim3((unsigned)grid_of(n * (lay.data_size / 4 + 1), 256)), dim3(256), 0,
                     st, G, d_base);
  HIP_OK(hipGetLastError());
  HIP_OK(hipStreamSynchronize(st));
  // (both buffers are make_index's from its first line on, also when it throws)
  uint8_t *const d_pages = pages.as<uint8_t>(), *const d_codes = codes.as<uint8_t>();
  pages.p = codes.p = nullptr;
  std::unique_ptr<qv_index, void (*)(qv_index*)> ix(make_index(device, lay, pq, d_pages, d_codes, false),
                                                     release_index);

  // insertion order: seeded Fisher-Yates
  std::vector<int32_t> order((size_t)n);
  std::iota(order.begin(), order.end(), 0);
  for (int64_t i = n - 1; i > 0; i--) {
    const int64_t j = (int64_t)(rng_u64(prm.seed, 21, (uint64_t)i) % (uint64_t)(i + 1));
    std::swap(order[(size_t)i], order[(size_t)j]);
  }
  const int64_t max_batch = std::max<int64_t>(1024, std::min<int64_t>(262144, n / 40));
  const int rec_cap = 256;
  DevBuf d_order, d_q, d_rec, d_recd, d_hops, d_pairs, d_sorted, d_heads, d_cnt, d_tmp;
  HIP_OK(hipMalloc(&d_order.p, sizeof(int32_t) * (size_t)n));
  HIP_OK(hipMemcpy(d_order.p, order.data(), sizeof(int32_t) * (size_t)n, hipMemcpyHostToDevice));
  HIP_OK(hipMalloc(&d_q.p, sizeof(float) * (size_t)(max_batch * dim)));
  HIP_OK(hipMalloc(&d_rec.p, sizeof(int32_t) * (size_t)(max_batch * rec_cap)));
  HIP_OK(hipMalloc(&d_recd.p, sizeof(float) * (size_t)(max_batch * rec_cap)));
  HIP_OK(hipMalloc(&d_hops.p, sizeof(int32_t) * (size_t)max_batch));
  HIP_OK(hipMalloc(&d_pairs.p, sizeof(uint64_t) * (size_t)(max_batch * prm.R)));
  HIP_OK(hipMalloc(&d_sorted.p, sizeof(uint64_t) * (size_t)(max_batch * prm.R)));
  HIP_OK(hipMalloc(&d_heads.p, sizeof(int32_t) * (size_t)(max_batch * prm.R)));
  HIP_OK(hipMalloc(&d_cnt.p, 64));
  // graph slack (DiskANN's GRAPH_SLACK_FACTOR 1.3): up to P reverse edges per
  // node wait beside its record's R slots until a prune folds them in
  const int P = (int)std::ceil(0.3 * prm.R);
  DevBuf d_pend, d_pcnt, d_marks, d_flush;
  HIP_OK(hipMalloc(&d_pend.p, sizeof(uint32_t) * (size_t)n * (size_t)P));
  HIP_OK(hipMalloc(&d_pcnt.p, sizeof(int32_t) * (size_t)n));
  HIP_OK(hipMemsetAsync(d_pcnt.p, 0, sizeof(int32_t) * (size_t)n, st));
  HIP_OK(hipMalloc(&d_marks.p, sizeof(int32_t) * (size_t)(max_batch * prm.R)));
  HIP_OK(hipMalloc(&d_flush.p, sizeof(int32_t) * (size_t)n));
  size_t tmp_bytes = 0;
  HIP_OK(rocprim::radix_sort_keys(nullptr, tmp_bytes, d_pairs.as<uint64_t>(), d_sorted.as<uint64_t>(),
                                  (size_t)(max_batch * prm.R), 0, 64, st));
  HIP_OK(hipMalloc(&d_tmp.p, tmp_bytes));

  // Prune geometry: rows of `stride` dwords (16-byte pieces, an odd number of
  // them, so 16 lanes reading 16 different rows hit distinct banks), G lanes
  // per cooperative row fetch, and the candidate capacity: the largest with
  // which four prunes (two of long rows) fit a CU.  The capacity cuts the
  // candidates, so it is part of what graph a build gives: its rule counts the
  // rows, keys and lists only.
  const int ds4 = (int)(lay.data_size / 4);
  int stride4 = (ds4 + 3) / 4;
  if (stride4 % 2 == 0) stride4++;
  const int stride = 4 * stride4;
  int fetch_lanes = 4;
  while (fetch_lanes < 64 && fetch_lanes * 4 < ds4) fetch_lanes *= 2;
  int lds_cu = 0;
  HIP_OK(hipDeviceGetAttribute(&lds_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, device));
  auto prunes_at = [&](int c) {
    const int bytes = (prune_lds_plan(c, stride, prm.R).rule + 1023) & ~1023;
    return lds_cu / bytes;
  };
  int cmax = 256;
  while (cmax > 192 && prunes_at(cmax) < 4) cmax -= 8;
  if (prunes_at(cmax) < 4) {
    cmax = 256;
    while (cmax > 64 && prunes_at(cmax) < 2) cmax -= 8;
  }
  const size_t prune_lds = (size_t)prune_lds_plan(cmax, stride, prm.R).total;
  // the candidate's row in registers where its 16-byte pieces fit
  const int q4 = (ds4 + 3) / 4;
  void (*prune)(PruneArgs) = q4 <= 8 ? prune_kernel<T, 8> : prune_kernel<T, 0>;
  if constexpr (sizeof(T) == 4) {
    if (q4 > 8 && q4 <= 32) prune = q4 <= 24 ? prune_kernel<T, 24> : prune_kernel<T, 32>;
  }
  HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(prune), hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)prune_lds));
  auto launch_prune = [&](const PruneArgs& args) {
    hipLaunchKernelGGL(prune, dim3((unsigned)std::min<int64_t>(args.num_centers, 65536)), dim3(kPruneThreads), prune_lds,
                       st, args);
    HIP_OK(hipGetLastError());
  };

  const int passes = std::max(1, std::min(2, prm.passes));
  // QV_BUILD_PROGRESS=1: a progress line on stderr at most every 10 s (long builds)
  const bool progress = std::getenv("QV_BUILD_PROGRESS") != nullptr;
  auto last_note = std::chrono::steady_clock::now();
  for (int pass = 0; pass < passes; pass++) {
    const float alpha = (passes == 2 && pass == 0) ? 1.0f : prm.alpha;
    int64_t done = 0, bsz = 1;
    while (done < n) {
      const int64_t nb = std::min(n - done, pass == 0 ? std::min(bsz, max_batch) : max_batch);
      const int32_t* ids = d_order.as<int32_t>() + done;
      hipLaunchKernelGGL(gather_rows_f32<T>, dim3((unsigned)grid_of(nb * dim, 256)), dim3(256), 0, st, d_base, dim,
                         ids, nb, d_q.as<float>());
      HIP_OK(hipGetLastError());
      HIP_OK(hipStreamSynchronize(st));
      SearchRecord rec;
      rec.ids = d_rec.as<int32_t>();
      rec.dists = d_recd.as<float>();
      rec.cap = rec_cap;
      search_record(ix.get(), d_q.as<float>(), nb, std::min(prm.L, kMaxEfShared), rec, d_hops.as<int32_t>(), 0);

      PruneArgs pa{};
      pa.L = G;
      pa.mode = 0;
      pa.centers = ids;
      pa.num_centers = nb;
      pa.rec_ids = d_rec.as<int32_t>();
      pa.hops = d_hops.as<int32_t>();
      pa.rec_cap = rec_cap;
      pa.pend = d_pend.as<uint32_t>();
      pa.pcnt = d_pcnt.as<int32_t>();
      pa.P = P;
      pa.alpha = alpha;
      pa.cmax = cmax;
      pa.stride = stride;
      pa.G = fetch_lanes;
      launch_prune(pa);

      HIP_OK(hipMemsetAsync(d_cnt.p, 0, 64, st));
      const int64_t np = nb * prm.R;
      hipLaunchKernelGGL(emit_pairs_kernel, dim3((unsigned)grid_of(np, 256)), dim3(256), 0, st, G, ids, nb,
                         d_pairs.as<uint64_t>(), d_cnt.as<unsigned long long>());
      HIP_OK(hipGetLastError());
      HIP_OK(rocprim::radix_sort_keys(d_tmp.p, tmp_bytes, d_pairs.as<uint64_t>(), d_sorted.as<uint64_t>(),
                                      (size_t)np, 0, 64, st));
      unsigned long long nvalid = 0;
      HIP_OK(hipMemcpyAsync(&nvalid, d_cnt.p, sizeof(nvalid), hipMemcpyDeviceToHost, st));
      HIP_OK(hipStreamSynchronize(st));
      if (nvalid > 0) {
        unsigned int* d_nh = reinterpret_cast<unsigned int*>(d_cnt.as<char>() + 32);
        unsigned int* d_nm = reinterpret_cast<unsigned int*>(d_cnt.as<char>() + 40);
        HIP_OK(hipMemsetAsync(d_nh, 0, 16, st));
        hipLaunchKernelGGL(heads_kernel, dim3((unsigned)grid_of((int64_t)nvalid, 256)), dim3(256), 0, st,
                           d_sorted.as<uint64_t>(), (int64_t)nvalid, d_heads.as<int32_t>(), d_nh);
        HIP_OK(hipGetLastError());
        unsigned int nheads = 0;
        HIP_OK(hipMemcpyAsync(&nheads, d_nh, 4, hipMemcpyDeviceToHost, st));
        HIP_OK(hipStreamSynchronize(st));
        // append reverse edges where the list or its slack has room; mark the rest
        hipLaunchKernelGGL(reverse_insert_kernel, dim3((unsigned)std::min<unsigned>(nheads, 65536u)), dim3(64), 0,
                           st, G, d_sorted.as<uint64_t>(), d_heads.as<int32_t>(), (int64_t)nheads,
                           (int64_t)nvalid, d_pend.as<uint32_t>(), d_pcnt.as<int32_t>(), P,
                           d_marks.as<int32_t>(), d_nm);
        HIP_OK(hipGetLastError());
        unsigned int nmarks = 0;
        HIP_OK(hipMemcpyAsync(&nmarks, d_nm, 4, hipMemcpyDeviceToHost, st));
        HIP_OK(hipStreamSynchronize(st));
        if (nmarks > 0) {
          PruneArgs ra = pa;
          ra.mode = 1;
          ra.centers = nullptr;
          ra.num_centers = nmarks;
          ra.pairs = d_sorted.as<uint64_t>();
          ra.heads = d_heads.as<int32_t>();
          ra.marks = d_marks.as<int32_t>();
          ra.num_pairs = (int64_t)nvalid;
          launch_prune(ra);
          HIP_OK(hipStreamSynchronize(st));
        }
      }
      done += nb;
      bsz = std::min<int64_t>(bsz * 2, max_batch);  // capped: no overflow on long builds
      if (progress && std::chrono::steady_clock::now() - last_note > std::chrono::seconds(10)) {
        last_note = std::chrono::steady_clock::now();
        std::fprintf(stderr, "[qv build] pass %d/%d: %lld of %lld points inserted\n", pass + 1, passes,
                     (long long)done, (long long)n);
        std::fflush(stderr);
      }
    }
    // end of the pass: fold every node's pending edges into its list (DiskANN's
    // final prune of lists longer than R)
    unsigned int* d_nf = reinterpret_cast<unsigned int*>(d_cnt.as<char>() + 48);
    HIP_OK(hipMemsetAsync(d_nf, 0, 4, st));
    hipLaunchKernelGGL(pending_nodes_kernel, dim3((unsigned)grid_of(n, 256)), dim3(256), 0, st,
                       d_pcnt.as<int32_t>(), n, d_flush.as<int32_t>(), d_nf);
    HIP_OK(hipGetLastError());
    unsigned int nflush = 0;
    HIP_OK(hipMemcpyAsync(&nflush, d_nf, 4, hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    if (nflush > 0) {
      PruneArgs fa{};
      fa.L = G;
      fa.mode = 2;
      fa.centers = d_flush.as<int32_t>();
      fa.num_centers = nflush;
      fa.pend = d_pend.as<uint32_t>();
      fa.pcnt = d_pcnt.as<int32_t>();
      fa.P = P;
      fa.alpha = alpha;
      fa.cmax = cmax;
      fa.stride = stride;
      fa.G = fetch_lanes;
      launch_prune(fa);
      HIP_OK(hipStreamSynchronize(st));
    }
  }
  (void)t_start;
  return ix.release();
}

}  // namespace

extern "C" {

int qv_build_index_gpu(const void* d_base, int32_t data_type, int64_t n, int32_t dim,
                       const qv_build_params* params, int device, qv_index** out) {
  return qv::guard([&] {
    if (!d_base || !out || dim <= 0) qv::fail(QV_EINVAL, "bad argument");
    *out = nullptr;
    if (n <= 1 || n > (int64_t)INT32_MAX - 64) qv::fail(QV_EINVAL, "n must be in [2, 2^31 - 64)");
    qv_build_params p;
    qv_build_params_default(&p);
    if (params) p = *params;
    if (p.R <= 0 || p.R > kMaxBuildDegree) qv::fail(QV_EINVAL, "R must be in [1, 128]");
    if (p.L < p.R) qv::fail(QV_EINVAL, "L must be >= R");
    HIP_OK(hipSetDevice(device));
    if (data_type == QV_UINT8)
      *out = build_gpu_t<uint8_t>(static_cast<const uint8_t*>(d_base), data_type, n, dim, p, device);
    else if (data_type == QV_INT8)
      *out = build_gpu_t<int8_t>(static_cast<const int8_t*>(d_base), data_type, n, dim, p, device);
    else if (data_type == QV_FLOAT)
      *out = build_gpu_t<float>(static_cast<const float*>(d_base), data_type, n, dim, p, device);
    else
      qv::fail(QV_EINVAL, "bad data type");
    qv::validate_graph(*out);
  });
}

}  // extern "C"
