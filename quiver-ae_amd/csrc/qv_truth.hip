// qv_truth.hip -- brute-force exact nearest neighbours (ground truth) on the GPU.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <type_traits>

#include "qv_common.hpp"
#include "qv_device.hpp"
#include "qv_hip_util.hpp"
#include "qv_index_impl.hpp"

using namespace qv;
using namespace qv::dev;

namespace {

// ---- brute-force ground truth ----------------------------------------------

constexpr int kGtQ = 8;

__device__ __forceinline__ void gt_offer(uint64_t& tk, int k, uint64_t key) {
  uint64_t cand = __ballot(key < (((uint64_t)(uint32_t)__shfl((int)(uint32_t)(tk >> 32), k - 1) << 32) |
                                  (uint32_t)__shfl((int)(uint32_t)tk, k - 1)));
  while (cand) {
    const int l = __ffsll((long long)cand) - 1;
    cand &= cand - 1;
    const uint64_t ck = ((uint64_t)(uint32_t)__shfl((int)(uint32_t)(key >> 32), l) << 32) |
                        (uint32_t)__shfl((int)(uint32_t)key, l);
    const uint64_t th = ((uint64_t)(uint32_t)__shfl((int)(uint32_t)(tk >> 32), k - 1) << 32) |
                        (uint32_t)__shfl((int)(uint32_t)tk, k - 1);
    if (ck < th) {
      const int lane = lane_id();
      const int pos = __popcll(__ballot(lane < k && tk < ck));
      const uint64_t prev = ((uint64_t)(uint32_t)__shfl_up((int)(uint32_t)(tk >> 32), 1) << 32) |
                            (uint32_t)__shfl_up((int)(uint32_t)tk, 1);
      if (lane < k) {
        if (lane == pos) tk = ck;
        else if (lane > pos) tk = prev;
      }
    }
  }
}

// Block (query group, base slice): 4 waves stream the slice, each lane one base
// row at a time, distances to kGtQ queries in fp32 (exact for 8-bit data).
// which: (direct kernels) the call's numbers of the nq queries, null for all.
template <class T>
__global__ __launch_bounds__(256) void gt_kernel(const T* __restrict__ base, int64_t n, int dim,
                                                 const float* __restrict__ queries, const int64_t* __restrict__ which,
                                                 int64_t nq, int k, int64_t slice, int S,
                                                 uint64_t* __restrict__ part) {
  extern __shared__ __align__(16) char smem[];
  float* q = reinterpret_cast<float*>(smem);
  uint64_t* xk = reinterpret_cast<uint64_t*>(q + kGtQ * dim);
  const int64_t q0 = (int64_t)blockIdx.x * kGtQ;
  const int s = blockIdx.y;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  for (int i = tid; i < kGtQ * dim; i += 256) {
    const int64_t qi = q0 + i / dim;
    q[i] = qi < nq ? queries[(which ? which[qi] : qi) * dim + (i % dim)] : 0.f;
  }
  __syncthreads();
  uint64_t tk[kGtQ];
#pragma unroll
  for (int t = 0; t < kGtQ; t++) tk[t] = kPadKey;
  const int64_t r0 = (int64_t)s * slice, r1 = min(n, r0 + slice);
  for (int64_t rb = r0 + wave * kWave; rb < r1; rb += 4 * kWave) {
    const int64_t r = rb + lane;
    float acc[kGtQ];
#pragma unroll
    for (int t = 0; t < kGtQ; t++) acc[t] = 0.f;
    if (r < r1) {
      // rows are read a dword at a time (dim * sizeof(T) is a multiple of 4)
      constexpr int per = 4 / (int)sizeof(T);
      const uint32_t* x32 = reinterpret_cast<const uint32_t*>(base + r * dim);
      for (int w = 0; w < dim / per; w++) {
        const uint32_t word = x32[w];
#pragma unroll
        for (int e = 0; e < per; e++) {
          float xv;
          if constexpr (sizeof(T) == 4) xv = __uint_as_float(word);
          else if constexpr (std::is_signed<T>::value) xv = (float)(int8_t)(word >> (8 * e));
          else xv = (float)((word >> (8 * e)) & 0xffu);
          const int j = w * per + e;
#pragma unroll
          for (int t = 0; t < kGtQ; t++) {
            const float d = q[t * dim + j] - xv;
            acc[t] = __fmaf_rn(d, d, acc[t]);
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < kGtQ; t++) {
      const uint64_t key = r < r1 ? (((uint64_t)__float_as_uint(acc[t]) << 32) | (uint64_t)r) : kPadKey;
      gt_offer(tk[t], k, key);
    }
  }
#pragma unroll
  for (int t = 0; t < kGtQ; t++) {
    xk[(t * 4 + wave) * kWave + lane] = tk[t];
  }
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int t = 0; t < kGtQ; t++) {
      uint64_t m = tk[t];
      for (int w = 1; w < 4; w++) gt_offer(m, k, lane < k ? xk[(t * 4 + w) * kWave + lane] : kPadKey);
      const int64_t qi = q0 + t;
      if (qi < nq && lane < k) part[(qi * S + s) * k + lane] = m;
    }
  }
}

__global__ void gt_final_kernel(const uint64_t* __restrict__ part, const int64_t* __restrict__ which, int64_t nq, int S,
                                int k, int32_t* __restrict__ ids, float* __restrict__ dists) {
  const int lane = lane_id();
  for (int64_t qi = blockIdx.x; qi < nq; qi += gridDim.x) {
    uint64_t tk = kPadKey;
    for (int s = 0; s < S; s++) gt_offer(tk, k, lane < k ? part[(qi * S + s) * k + lane] : kPadKey);
    if (lane < k) {
      const int64_t at = (which ? which[qi] : qi) * k + lane;
      ids[at] = tk == kPadKey ? -1 : (int32_t)(uint32_t)tk;
      dists[at] = tk == kPadKey ? __int_as_float(0x7f800000) : __uint_as_float((uint32_t)(tk >> 32));
    }
  }
}

// Ground truth for 8-bit data with integer dot products: each lane owns one
// query (its elements packed four to a register, zero past dim <= 128), tiles
// of kGtTile consecutive base rows are staged in LDS with coalesced loads
// (rows of kGtStride words: nine 16-byte pieces, an odd count, so the row-per-
// thread norm pass is conflict-free) and every lane compares its query with
// each staged row: d = |q|^2 + |x|^2 - 2 q.x, exact in int32 and in fp32
// (< 2^24), so keys (d, id) -- and the top-k with ties to the smaller id --
// equal the floating-point kernel's.
constexpr int kGtTile = 256;
constexpr int kGtWords = 32;
constexpr int kGtStride = 36;
constexpr int kGtMaxK = 16;

template <class T>
__device__ __forceinline__ uint32_t dot4(uint32_t a, uint32_t b, uint32_t acc) {
  if constexpr (std::is_signed<T>::value)
    return (uint32_t)__builtin_amdgcn_sdot4((int)a, (int)b, (int)acc, false);
  else
    return __builtin_amdgcn_udot4(a, b, acc, false);
}

template <class T>
__global__ __launch_bounds__(256) void gt_int_kernel(const T* __restrict__ base, int64_t n, int dim,
                                                     const float* __restrict__ queries,
                                                     const int64_t* __restrict__ which, int64_t nq, int k,
                                                     int64_t slice, int S, uint64_t* __restrict__ part) {
  __shared__ __align__(16) uint32_t rows[kGtTile * kGtStride];
  __shared__ int32_t norms[kGtTile];
  const int tid = threadIdx.x;
  const int64_t qi = (int64_t)blockIdx.x * 256 + tid;
  const int s = blockIdx.y;
  const int d4 = dim / 4;
  const int64_t query = qi < nq && which ? which[qi] : qi;
  uint32_t qw[kGtWords];
#pragma unroll
  for (int w = 0; w < kGtWords; w++) {
    uint32_t packed = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int j = 4 * w + e;
      const int v = qi < nq && j < dim ? (int)queries[query * dim + j] : 0;
      packed |= ((uint32_t)v & 0xffu) << (8 * e);
    }
    qw[w] = packed;
  }
  uint32_t qn = 0;
#pragma unroll
  for (int w = 0; w < kGtWords; w++) qn = dot4<T>(qw[w], qw[w], qn);
  for (int i = tid; i < kGtTile * kGtStride; i += 256) rows[i] = 0u;  // pads stay zero
  uint64_t tk[kGtMaxK];
#pragma unroll
  for (int i = 0; i < kGtMaxK; i++) tk[i] = kPadKey;
  uint64_t thr = kPadKey;
  const int64_t r0 = (int64_t)s * slice, r1 = min(n, r0 + slice);
  __syncthreads();
  for (int64_t t0 = r0; t0 < r1; t0 += kGtTile) {
    const int here = (int)min<int64_t>(kGtTile, r1 - t0);
    const uint8_t* src = reinterpret_cast<const uint8_t*>(base + t0 * dim);
    if ((d4 & 3) == 0) {
      const int pr = d4 / 4;  // 16-byte pieces per row
      const uint4* s4 = reinterpret_cast<const uint4*>(src);
      for (int u = tid; u < here * pr; u += 256) {
        const int r = u / pr, c = u - r * pr;
        *reinterpret_cast<uint4*>(rows + r * kGtStride + 4 * c) = s4[u];
      }
    } else {
      const uint32_t* s1 = reinterpret_cast<const uint32_t*>(src);
      for (int u = tid; u < here * d4; u += 256) {
        const int r = u / d4, c = u - r * d4;
        rows[r * kGtStride + c] = s1[u];
      }
    }
    __syncthreads();
    if (tid < here) {
      const uint4* rp = reinterpret_cast<const uint4*>(rows + tid * kGtStride);
      uint32_t nn = 0;
#pragma unroll
      for (int pc = 0; pc < kGtWords / 4; pc++) {
        const uint4 x = rp[pc];
        nn = dot4<T>(x.x, x.x, nn);
        nn = dot4<T>(x.y, x.y, nn);
        nn = dot4<T>(x.z, x.z, nn);
        nn = dot4<T>(x.w, x.w, nn);
      }
      norms[tid] = (int32_t)nn;
    }
    __syncthreads();
    for (int r = 0; r < here; r++) {
      const uint4* rp = reinterpret_cast<const uint4*>(rows + r * kGtStride);
      uint32_t acc = 0;
#pragma unroll
      for (int pc = 0; pc < kGtWords / 4; pc++) {
        const uint4 x = rp[pc];
        acc = dot4<T>(qw[4 * pc + 0], x.x, acc);
        acc = dot4<T>(qw[4 * pc + 1], x.y, acc);
        acc = dot4<T>(qw[4 * pc + 2], x.z, acc);
        acc = dot4<T>(qw[4 * pc + 3], x.w, acc);
      }
      const int32_t d = (int32_t)qn + norms[r] - 2 * (int32_t)acc;
      const uint64_t key = ((uint64_t)__float_as_uint((float)d) << 32) | (uint64_t)(t0 + r);
      if (key < thr) {
#pragma unroll
        for (int i = kGtMaxK - 1; i > 0; i--) {
          const uint64_t lo = tk[i - 1], cur = tk[i];
          tk[i] = key < lo ? lo : (key < cur ? key : cur);
        }
        tk[0] = key < tk[0] ? key : tk[0];
        uint64_t t = tk[0];
#pragma unroll
        for (int i = 1; i < kGtMaxK; i++) t = i == k - 1 ? tk[i] : t;
        thr = t;
      }
    }
    __syncthreads();
  }
  if (qi < nq) {
#pragma unroll
    for (int i = 0; i < kGtMaxK; i++)
      if (i < k) part[(qi * S + s) * k + i] = tk[i];
  }
}

// Sets *bad when a query element is not an integer of the element type's range
// (then the 8-bit kernel does not apply).
template <class T>
__global__ void gt_query_check(const float* __restrict__ q, int64_t count, int32_t* __restrict__ bad) {
  const float lo = std::is_signed<T>::value ? -128.f : 0.f, hi = std::is_signed<T>::value ? 127.f : 255.f;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x) {
    const float v = q[i];
    if (!(v >= lo && v <= hi && v == rintf(v))) *bad = 1;
  }
}

// ---- ground truth on the matrix cores ---------------------------------------
//
// A scan over base rows that only has to find, per query, the rows that may
// still be among its k nearest: the products q.x of 32 rows and 32 queries at
// a time come from MFMA, one compare against the query's threshold drops all
// but a few hundred rows per query, and those few are ranked exactly
// (gt_pick_kernel), so ids, distances and ties equal the direct kernels'.
//   * 8-bit data: bytes shifted to int8 (a distance does not change), q.x exact
//     in int32 (v_mfma_i32_32x32x32_i8).
//   * float: rows and queries split into two bf16 parts (x = hi + lo + r,
//     |r| <= 2^-17 |x|), q.x = hi hi + hi lo + lo hi in fp32
//     (v_mfma_f32_32x32x16_bf16): only a bound.  Its error against the real
//     q.x, the norms' and the ranked distance's own rounding together are
//     below kGtEps (|q|^2 + |x|^2) for dim <= 128 (2^-15 |q||x| of dropped
//     parts and 2^-15.4 of 3 x 128 accumulations, twice, plus 2^-16 for the
//     sums of squares and 2^-22 for the differences to the point below: under
//     2^-12.9), so a row is only dropped when its
//     distance is above the threshold whatever the rounding.  The candidates'
//     distances are the fp32 chain of the direct kernel.
// Thresholds come from the rows already scanned.  Level 0 takes every S-th row
// (S = 4^m, a few hundred rows) and keeps them all; level j the rows whose
// number modulo S lies in [w, 4 w), w = 4^(j - 1), so every level scans three
// times the rows of all before it, spread over the whole base, and about 3 k
// of them pass the k-th distance found so far.
// Queries the scan cannot finish (8-bit: no whole numbers of the element type;
// float: a norm that is no number or overflows; a list that overflows: data ordered against the period, more than a list of
// float rows within the bound's slack of the k-th) are left out of its further
// levels and go to the direct kernels, by themselves, as soon as the next
// level's list is known not to hold them (gt_pick_kernel); once half of a batch
// has left, all of it does and its scans end early.
// The slack is relative to the norms, so float rows and queries are taken
// relative to a point amid the data (gt_start_kernel); a distance does not
// change.  (Per dimension the median of 16 rows: a few rows far out do not
// move it, as they would a mean.)
//
// What bounds it: the matrix pipes need 4 x 32 cycles per 32 x 32 pairs of 128
// bytes (1.25 M of the last level's 3.1 M cycles at the sizes below), the rest
// is the compare (8 max3 and a compare per 1,024 pairs), the candidates' path
// and the barrier that ties a workgroup's waves to the slowest of them.  So
// one tile of rows in LDS serves four query tiles per wave (two for float, 24
// MFMA per operand pair) while the next is in flight in registers, and a
// candidate costs no wait: it goes to a pool in LDS, 64 of them to the lists
// in one round trip of counter atomics.  Two query tiles per wave and twice
// the waves: 1.69 ms for the last level instead of 1.44 (float, one instead of
// two: 0.74 instead of 0.48).
// Measured, whole call: 10,000 queries x 1M x 128 uint8, k = 10: 2.4 ms
// (18.8 ms with one query per lane and dot4); 2,001 x 500,001 x 96 float: 0.96
// ms (12.1 ms with 8 queries per workgroup and fp32 FMA).

typedef int32_t gt_i4 __attribute__((ext_vector_type(4)));
typedef int32_t gt_i16 __attribute__((ext_vector_type(16)));
typedef float gt_f16 __attribute__((ext_vector_type(16)));
typedef __bf16 gt_b8 __attribute__((ext_vector_type(8)));

constexpr int kGtRows = 64;          // base rows per LDS tile
constexpr int64_t kGtBatch = 32768;  // queries per scan: the lists' memory (4 KB a query up to k = 16, 16 KB beyond)
constexpr int kGtPool = 128;         // candidates a wave gathers in LDS before it appends them to the lists
constexpr float kGtEps = 1.0f / 4096.0f;
constexpr float kGtHuge = 1e37f;     // |x|^2 above this: the row is never dropped, the query leaves the scan
constexpr int kGtDrop = -(1 << 29);  // (8-bit) accumulator start of rows past the end
constexpr int kGtCenter = 128;       // (float) dimensions of the point amid the data, zero past the rows'
constexpr uint32_t kGtLeft = 1u << 31;  // count of a query that has left the scan (no list entry is written past cap)

// A batch's queries that have left the scan.
struct GtLeft {
  int32_t count;  // of them
  int32_t all;    // set with the count at `limit`: the whole batch leaves, its scans end early
};
// What the host reads at the end of a call.
struct GtCall {
  unsigned long long direct;  // queries listed for the direct kernels
  int32_t fractional;         // set when an 8-bit index's query is no whole number of the element type
  int32_t pad;
};

__device__ __forceinline__ void gt_leave(GtLeft* left, int limit) {
  if (atomicAdd(&left->count, 1) + 1 >= limit) left->all = 1;
}

struct ScanArgs {
  const uint8_t* base;
  int64_t row_bytes;
  int64_t rows;         // rows of this level (gt_base_row)
  int64_t period;       // S
  int32_t shift;        // log2 w, -1 at level 0
  int64_t nq;
  int groups, slices;   // query groups, row slices (a multiple of 8)
  const uint8_t* qp;    // packed queries, [padded nq][planes * KS * 32] bytes
  const uint32_t* qn;   // |q|^2 (int32 or float bits), [padded nq]
  const uint32_t* thr;  // accumulator threshold (int32 or float bits), [padded nq]
  const uint64_t* tkey; // (8-bit) key no candidate may exceed, [padded nq]
  uint32_t* cnt;        // [padded nq] candidates listed
  uint64_t* list;       // [nq][cap] keys (8-bit) or row ids (float)
  int cap;
  const float* center;  // (float) [kGtCenter] point the rows and queries are taken relative to
  GtLeft* left;
  int limit;
};

// Base row of a level's row i: every S-th row at level 0, else row i of the
// runs [S b + w, S b + 4 w).
__device__ __forceinline__ int64_t gt_base_row(const ScanArgs& a, uint32_t i) {
  if (a.shift < 0) return (int64_t)i * a.period;
  const uint32_t u = i >> a.shift, b = u / 3u;
  return (int64_t)b * a.period + ((int64_t)(u - 3u * b + 1u) << a.shift) + (int64_t)(i & ((1u << a.shift) - 1u));
}

template <class T>
struct GtKind {
  static constexpr bool kFloat = sizeof(T) == 4;
  static constexpr int kPlanes = kFloat ? 2 : 1;
  static constexpr int kPieceBytes = kFloat ? 32 : 16;  // source bytes behind one 16-byte LDS piece
  using Acc = std::conditional_t<kFloat, gt_f16, gt_i16>;
  using One = std::conditional_t<kFloat, float, int32_t>;
};

// LDS bytes of one tile row: its planes, then 16 bytes so that the row is an
// odd number of 16-byte pieces (lanes reading one piece of 32 rows spread over
// all banks).
template <class T>
constexpr int gt_row_lds(int KS) {
  return GtKind<T>::kPlanes * KS * 32 + 16;
}
// Lanes that stage one row, a 16-byte LDS piece of each plane per lane.
constexpr int gt_lanes(int KS) { return KS <= 2 ? 4 : (KS <= 4 ? 8 : 16); }
template <class T>
constexpr int gt_scan_lds(int KS, int QT) {
  return 2 * kGtRows * (gt_row_lds<T>(KS) + 8) + 4 * kGtPool * 12 +
         (GtKind<T>::kFloat ? gt_lanes(KS) * 32 : 128 * QT * 12) + 8;
}

// bf16 parts of 8 floats: hi rounded to nearest, lo the rounded rest.
__device__ __forceinline__ void gt_split(const float (&x)[8], gt_b8& hi, gt_b8& lo) {
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const __bf16 h = (__bf16)x[j];
    hi[j] = h;
    lo[j] = (__bf16)(x[j] - (float)h);
  }
}

// Four source words of a row of nwords 32-bit words from w0 on, zero past its
// end.
__device__ __forceinline__ gt_i4 gt_words(const uint32_t* row, int w0, int nwords) {
  typedef gt_i4 gt_i4u __attribute__((aligned(4)));  // rows are 4-byte aligned
  gt_i4 v = {0, 0, 0, 0};
  if (w0 + 4 <= nwords) {
    v = *reinterpret_cast<const gt_i4u*>(row + w0);
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (w0 + e < nwords) v[e] = (int32_t)row[w0 + e];
  }
  return v;
}

// uint8 words as int8 (x - 128), zero past the row's end.
template <class T>
__device__ __forceinline__ gt_i4 gt_shift(gt_i4 v, int w0, int nwords) {
  if constexpr (!std::is_signed<T>::value && sizeof(T) == 1) {
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = w0 + e < nwords ? (int32_t)((uint32_t)v[e] ^ 0x80808080u) : 0;
  }
  return v;
}

// Start of a call: its counts cleared (words of 4 bytes), and float: the point
// amid the data, per dimension the median of 16 rows spread over the base (0
// where there is none that is finite and not enormous).  One workgroup, a
// thread per dimension.
template <class T>
__global__ __launch_bounds__(kGtCenter) void gt_start_kernel(const T* __restrict__ base, int64_t n, int dim,
                                                             uint32_t* __restrict__ state, int64_t words,
                                                             float* __restrict__ center) {
  const int j = threadIdx.x;
  for (int64_t i = j; i < words; i += kGtCenter) state[i] = 0u;
  if constexpr (sizeof(T) == 4) {
    constexpr int kRows = 16;
    float c = 0.f;
    if (j < dim) {
      float v[kRows];
#pragma unroll
      for (int i = 0; i < kRows; i++) v[i] = base[(i * n / kRows) * dim + j];
#pragma unroll
      for (int i = 0; i < kRows; i++) {
        int below = 0;
#pragma unroll
        for (int o = 0; o < kRows; o++) below += v[o] < v[i] || (v[o] == v[i] && o < i) ? 1 : 0;
        if (below == kRows / 2) c = v[i];
      }
      if (!(fabsf(c) <= 1e15f)) c = 0.f;
    }
    center[j] = c;
  }
}

// Queries into the scan's operand layout, with their norms, an open threshold
// and an empty list.  An 8-bit index's query that is not a whole number of the
// element type's range leaves the scan here, and a float one without a finite
// norm that its bound could use: as zeros, since a NaN reaches any threshold
// (one such query of 2,000 x 500,000 x 96 would take the scan from 1.0 to 6.1
// ms).  One wave per query slot; slots past nq never match.
template <class T, int KS>
__global__ __launch_bounds__(64) void gt_pack_kernel(const float* __restrict__ queries, int64_t nq, int dim,
                                                     uint8_t* __restrict__ qp, uint32_t* __restrict__ qn,
                                                     uint32_t* __restrict__ thr, uint64_t* __restrict__ tkey,
                                                     uint32_t* __restrict__ cnt, const float* __restrict__ center,
                                                     GtLeft* __restrict__ left, int limit, GtCall* __restrict__ call) {
  using K = GtKind<T>;
  const int lane = lane_id();
  const int64_t q = blockIdx.x;
  const bool live = q < nq;
  uint8_t* const out = qp + q * (int64_t)(K::kPlanes * KS * 32);
  bool fractional = false, leaves = false;
  if constexpr (K::kFloat) {
    float s = 0.f, x[8];
    if (lane < KS * 2) {
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int i = lane * 8 + j;
        x[j] = live && i < dim ? queries[q * dim + i] - center[i] : 0.f;
        s = __fmaf_rn(x[j], x[j], s);
      }
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    leaves = !(s <= kGtHuge);
    if (lane < KS * 2) {
      gt_b8 hi, lo;
      if (leaves) {
#pragma unroll
        for (int j = 0; j < 8; j++) x[j] = 0.f;
      }
      gt_split(x, hi, lo);
      *reinterpret_cast<gt_b8*>(out + lane * 16) = hi;
      *reinterpret_cast<gt_b8*>(out + KS * 32 + lane * 16) = lo;
    }
    if (lane == 0) {
      qn[q] = __float_as_uint(s);
      thr[q] = live && !leaves ? 0xff800000u : 0x7f800000u;
    }
  } else {
    const float lo = std::is_signed<T>::value ? -128.f : 0.f, hi = std::is_signed<T>::value ? 127.f : 255.f;
    constexpr int kShift = std::is_signed<T>::value ? 0 : 128;
    int32_t s = 0;
    bool wrong = false;
    for (int w = lane; w < KS * 8; w += kWave) {
      uint32_t packed = 0;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int i = 4 * w + e;
        if (live && i < dim) {
          const float v = queries[q * dim + i];
          if (!(v >= lo && v <= hi && v == rintf(v))) wrong = true;
          packed |= ((uint32_t)((int)v - kShift) & 0xffu) << (8 * e);
        }
      }
      s = __builtin_amdgcn_sdot4((int)packed, (int)packed, s, false);
      reinterpret_cast<uint32_t*>(out)[w] = packed;
    }
    leaves = fractional = __ballot(wrong) != 0;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) {
      qn[q] = (uint32_t)s;
      thr[q] = (uint32_t)(live && !fractional ? INT32_MIN : INT32_MAX);
    }
  }
  if (lane == 0) {
    tkey[q] = kPadKey;
    cnt[q] = leaves ? kGtLeft : 0u;
    if (fractional) call->fractional = 1;
    if (leaves) gt_leave(left, limit);
  }
}

// One workgroup: 4 waves of QT x 32 queries each, over the row tiles of one
// slice.  Rows are D's rows and queries its columns, so a lane's 16 sums all
// belong to one query and one register holds its threshold; the accumulators
// start at minus half the rows' norms, so that "sum >= threshold" is the whole
// test.  Workgroups that share a slice run on one XCD (round-robin over 8 by
// workgroup number), whose L2 then serves its rows to all query groups.
template <class T, int KS, int QT>
__global__ __launch_bounds__(256, 2) void gt_scan_kernel(ScanArgs a) {
  using K = GtKind<T>;
  using Acc = typename K::Acc;
  using One = typename K::One;
  constexpr int P = K::kPlanes;
  constexpr int kPieces = KS * 2;                                                // per plane and row
  constexpr int kGroup = gt_lanes(KS);
  constexpr int kRounds = kGtRows * kGroup / 256;
  constexpr int kLoads = K::kPieceBytes / 16;
  constexpr int kStride = gt_row_lds<T>(KS);
  extern __shared__ __align__(16) char smem[];
  char* const tile = smem;                                                       // [2][kGtRows][kStride]
  One* const start = reinterpret_cast<One*>(smem + 2 * kGtRows * kStride);       // [2][kGtRows]
  One* const odds = start + 2 * kGtRows;                                         // (8-bit) |x|^2 & 1
  // one wave's pool: level rows, query slots of the wave and (8-bit) sums
  int32_t* const pools = reinterpret_cast<int32_t*>(odds + 2 * kGtRows);         // [4 waves][3][kGtPool]
  uint32_t* const pool_at = reinterpret_cast<uint32_t*>(pools + (threadIdx.x / kWave) * 3 * kGtPool);
  int32_t* const pool_q = reinterpret_cast<int32_t*>(pool_at + kGtPool);
  int32_t* const pool_sum = pool_q + kGtPool;
  // (float) a.center; (8-bit) the workgroup's queries' key limits and norms
  const float4* const center = reinterpret_cast<const float4*>(pools + 4 * 3 * kGtPool);
  uint64_t* const tkey = reinterpret_cast<uint64_t*>(pools + 4 * 3 * kGtPool);
  int32_t* const qnorm = reinterpret_cast<int32_t*>(tkey + 128 * QT);
  int32_t* const ended = reinterpret_cast<int32_t*>(smem + gt_scan_lds<T>(KS, QT) - 8);  // [2]

  const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  const int col = lane & 31, half = lane >> 5;
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int group = j % a.groups, slice = (j / a.groups) * 8 + xcd;
  const int64_t q0 = ((int64_t)group * 4 + wave) * (32 * QT) + col;
  const int64_t tiles = (a.rows + kGtRows - 1) / kGtRows;
  const int nwords = (int)(a.row_bytes / 4);

  gt_i4 b[QT][P][KS];
  One thr[QT];
#pragma unroll
  for (int t = 0; t < QT; t++) {
    const uint8_t* const src = a.qp + (q0 + 32 * t) * (int64_t)(P * KS * 32) + half * 16;
#pragma unroll
    for (int p = 0; p < P; p++)
#pragma unroll
      for (int s = 0; s < KS; s++) b[t][p][s] = *reinterpret_cast<const gt_i4*>(src + (p * KS + s) * 32);
    const uint32_t bits = a.thr[q0 + 32 * t];
    if constexpr (K::kFloat) thr[t] = __uint_as_float(bits);
    else thr[t] = (int32_t)bits;
  }

  const int piece = tid % kGroup;
  gt_i4 in[kRounds][kLoads];
  auto request = [&](int64_t t) {
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
      const int64_t i = t * kGtRows + tid / kGroup + r * (256 / kGroup);
      const bool ok = piece < kPieces && i < a.rows;
      const uint32_t* const src = reinterpret_cast<const uint32_t*>(a.base + gt_base_row(a, ok ? (uint32_t)i : 0u) * a.row_bytes);
#pragma unroll
      for (int l = 0; l < kLoads; l++)
        in[r][l] = ok ? gt_words(src, piece * (K::kPieceBytes / 4) + 4 * l, nwords) : gt_i4{0, 0, 0, 0};
    }
  };
  auto stage = [&](int64_t t, int buf) {
    float4 c0, c1;
    if constexpr (K::kFloat) c0 = center[2 * piece], c1 = center[2 * piece + 1];
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
      const int row = tid / kGroup + r * (256 / kGroup);
      char* const dst = tile + (buf * kGtRows + row) * kStride + piece * 16;
      const bool live = t * kGtRows + row < a.rows;
      One s = 0;
      if constexpr (K::kFloat) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = __int_as_float(in[r][e / 4][e % 4]);
        x[0] -= c0.x, x[1] -= c0.y, x[2] -= c0.z, x[3] -= c0.w;
        x[4] -= c1.x, x[5] -= c1.y, x[6] -= c1.z, x[7] -= c1.w;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          s = __fmaf_rn(x[e], x[e], s);
        }
        for (int off = 1; off < kGroup; off <<= 1) s += __shfl_xor(s, off);
        const bool keep = !(s <= kGtHuge);  // never dropped: zero row, accumulators at +inf
        if (keep) {
#pragma unroll
          for (int e = 0; e < 8; e++) x[e] = 0.f;
        }
        gt_b8 hi, lo;
        gt_split(x, hi, lo);
        if (piece < kPieces) {
          *reinterpret_cast<gt_b8*>(dst) = hi;
          *reinterpret_cast<gt_b8*>(dst + KS * 32) = lo;
        }
        if (piece == 0) {
          const float inf = __int_as_float(0x7f800000);
          start[buf * kGtRows + row] = !live ? -inf : (keep ? inf : -0.5f * (1.f - kGtEps) * s);
        }
      } else {
        const gt_i4 v = gt_shift<T>(in[r][0], piece * 4, live ? nwords : 0);
#pragma unroll
        for (int e = 0; e < 4; e++) s = __builtin_amdgcn_sdot4(v[e], v[e], s, false);
        for (int off = 1; off < kGroup; off <<= 1) s += __shfl_xor(s, off);
        if (piece < kPieces) *reinterpret_cast<gt_i4*>(dst) = v;
        if (piece == 0) {
          odds[buf * kGtRows + row] = s & 1;
          start[buf * kGtRows + row] = live ? -((s + 1) >> 1) : kGtDrop;
        }
      }
    }
  };

  // This wave's pooled candidates into their queries' lists, 64 at a time: one
  // round trip of counter atomics for 64 of them.
  int pooled = 0;
  auto flush = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    // a batch that has left adds nothing more (its counters would only be fought over)
    if (pooled > 0 && __hip_atomic_load(&a.left->all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) pooled = 0;
    for (int i = lane; i < pooled; i += kWave) {
      const uint32_t at = pool_at[i];
      const int lq = wave * 32 * QT + pool_q[i];
      const int64_t q = (int64_t)group * (128 * QT) + lq;
      uint64_t entry = 0;
      bool take = q < a.nq && (int64_t)at < a.rows;
      if (take) entry = (uint64_t)gt_base_row(a, at);
      if constexpr (!K::kFloat) {
        const int32_t dist = qnorm[lq] - pool_sum[i];
        entry |= (uint64_t)__float_as_uint((float)dist) << 32;
        take = take && entry <= tkey[lq];
      }
      if (take) {
        const uint32_t pos = atomicAdd(a.cnt + q, 1u);
        if (pos < (uint32_t)a.cap) a.list[q * a.cap + pos] = entry;
        else if (pos == (uint32_t)a.cap) gt_leave(a.left, a.limit);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    pooled = 0;
  };

  // The rows of one 32 x 32 tile that reach their query's threshold, into the
  // pool, without a wait: 8-bit candidates leave with |q|^2 - dist = 2 sum +
  // (|x|^2 & 1) (odd: the rows' norm parities), which flush turns into the key.
  auto harvest = [&](const Acc& d, One limit, int qt, int rt, uint32_t odd, int64_t t) {
    const uint32_t at = (uint32_t)(t * kGtRows) + (uint32_t)(rt * 32 + 4 * half);  // level row of element 0 (< 2^31)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const bool take = !(d[i] < limit);
      const uint64_t m = __ballot(take);
      if (m != 0) {
        const int row = 8 * (i / 4) + (i & 3);
        if (take) {
          const int to = pooled + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
          pool_at[to] = at + row;
          pool_q[to] = 32 * qt + col;
          if constexpr (!K::kFloat) pool_sum[to] = 2 * d[i] + (int32_t)((odd >> row) & 1u);
        }
        pooled += (int)__popcll(m);
        if (pooled > kGtPool - kWave) flush();
      }
    }
  };

  int64_t t = slice;
  if (t >= tiles) return;  // the whole workgroup
  request(t);
  if constexpr (K::kFloat) {
    if (tid < kGroup * 8) reinterpret_cast<float*>(pools + 4 * 3 * kGtPool)[tid] = a.center[tid];
    __syncthreads();
  } else {
    for (int i = tid; i < 128 * QT; i += 256) {
      tkey[i] = a.tkey[(int64_t)group * (128 * QT) + i];
      qnorm[i] = (int32_t)a.qn[(int64_t)group * (128 * QT) + i];
    }
  }
  stage(t, 0);
  __syncthreads();
  int buf = 0;
  while (true) {
    const int64_t tn = t + a.slices;
    const int32_t lost = __hip_atomic_load(&a.left->all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tn < tiles) request(tn);
    uint64_t parity = 0;
    if constexpr (!K::kFloat) parity = __ballot(odds[buf * kGtRows + lane] != 0);
#pragma unroll 1
    for (int rt = 0; rt < kGtRows / 32; rt++) {
      const char* const arow = tile + (buf * kGtRows + rt * 32 + col) * kStride + half * 16;
      const int r0 = buf * kGtRows + rt * 32;
      gt_i4 av[P][KS];
#pragma unroll
      for (int p = 0; p < P; p++)
#pragma unroll
        for (int s = 0; s < KS; s++) av[p][s] = *reinterpret_cast<const gt_i4*>(arow + (p * KS + s) * 32);
      // D element 4 g + e of a lane: row 8 g + 4 half + e of the tile
      Acc c;
#pragma unroll
      for (int g = 0; g < 4; g++)
#pragma unroll
        for (int e = 0; e < 4; e++) c[4 * g + e] = start[r0 + 8 * g + 4 * half + e];
      Acc d[QT];
#pragma unroll
      for (int s = 0; s < KS; s++) {
#pragma unroll
        for (int qt = 0; qt < QT; qt++) {
          const Acc& in_c = s == 0 ? c : d[qt];
          if constexpr (K::kFloat) {
            const gt_b8 ah = __builtin_bit_cast(gt_b8, av[0][s]), al = __builtin_bit_cast(gt_b8, av[P - 1][s]);
            const gt_b8 bh = __builtin_bit_cast(gt_b8, b[qt][0][s]), bl = __builtin_bit_cast(gt_b8, b[qt][P - 1][s]);
            d[qt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, in_c, 0, 0, 0);
            d[qt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, d[qt], 0, 0, 0);
            d[qt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, d[qt], 0, 0, 0);
          } else {
            d[qt] = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[0][s], b[qt][0][s], in_c, 0, 0, 0);
          }
        }
      }
      bool pass[QT], any = false;
#pragma unroll
      for (int qt = 0; qt < QT; qt++) {
        One top = d[qt][0];
#pragma unroll
        for (int i = 1; i < 16; i++) {
          if constexpr (K::kFloat) top = fmaxf(top, d[qt][i]);
          else top = max(top, d[qt][i]);
        }
        pass[qt] = !(top < thr[qt]);
        any |= pass[qt];
      }
      if (__ballot(any) == 0) continue;
      uint32_t hits = 0;
#pragma unroll
      for (int qt = 0; qt < QT; qt++) hits |= __ballot(pass[qt]) != 0 ? 1u << qt : 0u;
      uint32_t odd = 0;
      if constexpr (!K::kFloat) odd = (uint32_t)(parity >> (rt * 32)) >> (4 * half);
      // one copy of the harvest for every query tile (its code, not its moves, is the cost)
#pragma unroll 1
      while (hits != 0) {
        const int qt = __builtin_ctz(hits);
        hits &= hits - 1;
        Acc x = d[0];
        One limit = thr[0];
#pragma unroll
        for (int o = 1; o < QT; o++) {
          if (qt == o) {
            x = d[o];
            limit = thr[o];
          }
        }
        harvest(x, limit, qt, rt, odd, t);
      }
    }
    if (tn >= tiles) break;
    stage(tn, buf ^ 1);
    if (tid == 0) ended[buf ^ 1] = lost;
    __syncthreads();
    buf ^= 1;
    t = tn;
    if (ended[buf]) break;  // the same word for every wave
  }
  flush();
}

// The k nearest of each query's listed rows, one wave per query: float rows
// get their distance here (the direct kernel's fp32 chain over the
// dimensions).  Before the last level: the threshold for the next one, and a
// list of just these, or the query leaves the scan; at the last: the results,
// or for a query that has left its number in the direct kernels' list.
template <class T>
__global__ __launch_bounds__(256) void gt_pick_kernel(const uint8_t* __restrict__ base, int64_t row_bytes, int dim,
                                                      const float* __restrict__ queries, int64_t nq, int k,
                                                      const uint32_t* __restrict__ qn, uint32_t* __restrict__ thr,
                                                      uint64_t* __restrict__ tkey, uint32_t* __restrict__ cnt,
                                                      uint64_t* __restrict__ list, int cap, int level, bool last,
                                                      int32_t* __restrict__ ids, float* __restrict__ dists,
                                                      GtLeft* __restrict__ left, int limit, int64_t first_query,
                                                      GtCall* __restrict__ call, int64_t* __restrict__ direct) {
  __shared__ float qs[4][128];
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t q = (int64_t)blockIdx.x * 4 + wave;
  constexpr bool kFloat = sizeof(T) == 4;
  if constexpr (kFloat) {
    for (int i = lane; i < dim; i += kWave) qs[wave][i] = q < nq ? queries[q * dim + i] : 0.f;
    __syncthreads();
  }
  if (q >= nq) return;
  const uint32_t listed = cnt[q];
  const bool all_left = __hip_atomic_load(&left->all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  // (a query whose list ran over, or is about to in the next level, leaves)
  auto leave = [&]() {
    if (lane == 0) {
      if (last) {
        direct[atomicAdd(&call->direct, 1ull)] = first_query + q;
      } else if (listed < kGtLeft) {
        if (listed <= (uint32_t)cap) gt_leave(left, limit);  // (past cap: counted by the scan)
        cnt[q] = kGtLeft;
        thr[q] = kFloat ? 0x7f800000u : (uint32_t)INT32_MAX;
      }
    }
  };
  if (all_left || listed > (uint32_t)cap) {
    leave();
    return;
  }
  const int m = (int)listed;
  uint64_t tk = kPadKey;
  for (int i0 = 0; i0 < m; i0 += kWave) {
    uint64_t key = kPadKey;
    if (i0 + lane < m) {
      key = list[q * cap + i0 + lane];
      if constexpr (kFloat) {
        typedef float gt_f4u __attribute__((ext_vector_type(4), aligned(4)));
        const float* const x = reinterpret_cast<const float*>(base + (int64_t)key * row_bytes);
        float s = 0.f;
        int i = 0;
        for (; i + 4 <= dim; i += 4) {
          const gt_f4u v = *reinterpret_cast<const gt_f4u*>(x + i);
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float d = qs[wave][i + e] - v[e];
            s = __fmaf_rn(d, d, s);
          }
        }
        for (; i < dim; i++) {
          const float d = qs[wave][i] - x[i];
          s = __fmaf_rn(d, d, s);
        }
        key |= (uint64_t)__float_as_uint(s) << 32;
        if (level > 0 && !last && m > cap / 4) list[q * cap + i0 + lane] = key;  // (read again below)
      }
    }
    // the first 64 sorted at once, the others offered one by one
    if (i0 == 0) {
      tk = ~wave_sort_desc(~key);
      if (lane >= k) tk = kPadKey;
    } else {
      gt_offer(tk, k, key);
    }
  }
  if (last) {
    if (lane < k) {
      ids[q * k + lane] = tk == kPadKey ? -1 : (int32_t)(uint32_t)tk;
      dists[q * k + lane] = tk == kPadKey ? __int_as_float(0x7f800000) : __uint_as_float((uint32_t)(tk >> 32));
    }
    return;
  }
  if constexpr (kFloat) {
    // The next level has three times the rows of all before it, and of these
    // the ones that would pass the new threshold are in the list: the ones not
    // further than the k-th and the bound's slack (about 2 eps |q|^2 for a row
    // near the query).
    if (level > 0 && m > cap / 4) {
      const float kth = __uint_as_float(read_lane_u32((uint32_t)(tk >> 32), k - 1));
      const float reach = kth + 2.f * kGtEps * __uint_as_float(qn[q]);
      int near = 0;
      for (int i = lane; i < m; i += kWave) near += __uint_as_float((uint32_t)(list[q * cap + i] >> 32)) <= reach ? 1 : 0;
      for (int off = 32; off > 0; off >>= 1) near += __shfl_xor(near, off);
      if (3 * near > cap) {
        leave();
        return;
      }
    }
  }
  // the k found so far open the next level's list
  const uint64_t have = __ballot(lane < k && tk != kPadKey);
  if (lane < k && tk != kPadKey) list[q * cap + lane] = kFloat ? (uint64_t)(uint32_t)tk : tk;
  if (lane == k - 1) {
    cnt[q] = (uint32_t)__popcll(have);
    const float d = __uint_as_float((uint32_t)(tk >> 32));
    if constexpr (kFloat) {
      // a row is dropped when q.x (the bound) < ((1 - eps)(|q|^2 + |x|^2) - d) / 2;
      // with no bound for the query (distance not finite) none is
      const float n2 = __uint_as_float(qn[q]);
      const double at = 0.5 * ((1.0 - (double)kGtEps) * (double)n2 - (double)d) - 1e-30;
      thr[q] = __float_as_uint(tk != kPadKey && n2 <= kGtHuge && d <= kGtHuge ? __double2float_rd(at)
                                                                              : -__int_as_float(0x7f800000));
    } else {
      // dist = |q|^2 - 2 sum - (|x|^2 & 1) <= d needs sum >= (|q|^2 - d - 1) / 2
      tkey[q] = tk;
      thr[q] = (uint32_t)(tk != kPadKey ? ((int32_t)qn[q] - (int32_t)d) >> 1 : INT32_MIN);
    }
  }
}

// Memory of a call, given back in its stream's order, also when the call fails.
struct CallMemory {
  hipStream_t st;
  void* p = nullptr;
  explicit CallMemory(hipStream_t s) : st(s) {}
  CallMemory(const CallMemory&) = delete;
  CallMemory& operator=(const CallMemory&) = delete;
  ~CallMemory() {
    if (p) (void)hipFreeAsync(p, st);
  }
  hipError_t take(size_t bytes) { return hipMallocAsync(&p, bytes, st); }
  template <class U>
  U* as() const {
    return static_cast<U*>(p);
  }
};

int grid_of(int64_t work, int block) {
  return (int)std::max<int64_t>(1, std::min<int64_t>((work + block - 1) / block, 1 << 20));
}

// The scan of one batch of queries, all levels (see above).
template <class T, int KS, int QT>
void gt_levels(const T* d_base, int64_t n, int dim, const float* d_q, int64_t nq, int k, int32_t* d_ids,
               float* d_dists, int cap, int64_t resident, uint8_t* work, const float* center, GtLeft* left,
               int64_t first_query, GtCall* call, int64_t* direct, hipStream_t st) {
  const int64_t groups = (nq + 128 * QT - 1) / (128 * QT), padded = groups * 128 * QT;
  uint64_t* const list = reinterpret_cast<uint64_t*>(work);
  uint64_t* const tkey = list + nq * cap;
  uint32_t* const qn = reinterpret_cast<uint32_t*>(tkey + padded);
  uint32_t* const thr = qn + padded;
  uint32_t* const cnt = thr + padded;
  uint8_t* const qp = reinterpret_cast<uint8_t*>(cnt + padded);
  const int limit = (int)((nq + 1) / 2);
  hipLaunchKernelGGL((gt_pack_kernel<T, KS>), dim3((unsigned)padded), dim3(64), 0, st, d_q, nq, dim, qp, qn, thr, tkey,
                     cnt, center, left, limit, call);
  HIP_OK(hipGetLastError());
  ScanArgs a{};
  a.base = reinterpret_cast<const uint8_t*>(d_base);
  a.row_bytes = (int64_t)dim * (int64_t)sizeof(T);
  a.nq = nq;
  a.groups = (int)groups;
  a.qp = qp;
  a.qn = qn;
  a.thr = thr;
  a.tkey = tkey;
  a.cnt = cnt;
  a.list = list;
  a.cap = cap;
  a.center = center;
  a.left = left;
  a.limit = limit;
  int levels = 1;  // S = 4^(levels - 1): level 0 keeps all of its rows, at least k where n allows
  a.period = 1;
  while (n / (4 * a.period) >= (k <= 16 ? 64 : 256)) {
    a.period *= 4;
    levels++;
  }
  for (int l = 0; l < levels; l++) {
    const int64_t w = l == 0 ? 1 : (int64_t)1 << (2 * (l - 1)), width = l == 0 ? 1 : 3 * w;
    a.shift = l == 0 ? -1 : 2 * (l - 1);
    a.rows = n / a.period * width +
             std::max<int64_t>(0, std::min<int64_t>(n % a.period - (l == 0 ? 0 : w), width));
    const int64_t tiles = (a.rows + kGtRows - 1) / kGtRows;
    // as many workgroups as are resident at once, in eighths (one per XCD)
    a.slices = (int)(8 * std::max<int64_t>(1, std::min<int64_t>((tiles + 7) / 8, resident / (8 * groups))));
    hipLaunchKernelGGL((gt_scan_kernel<T, KS, QT>), dim3((unsigned)(groups * a.slices)), dim3(256),
                       (size_t)gt_scan_lds<T>(KS, QT), st, a);
    HIP_OK(hipGetLastError());
    hipLaunchKernelGGL(gt_pick_kernel<T>, dim3((unsigned)((nq + 3) / 4)), dim3(256), 0, st, a.base, a.row_bytes, dim,
                       d_q, nq, k, qn, thr, tkey, cnt, list, cap, l, l == levels - 1, d_ids, d_dists, left, limit,
                       first_query, call, direct);
    HIP_OK(hipGetLastError());
  }
}

// The direct kernels for the nq queries listed in which (null: the call's
// first nq).  whole: every one of them is a whole number of T's range.
template <class T>
void gt_direct(const T* d_base, int64_t n, int dim, const float* d_q, const int64_t* which, int64_t nq, int k,
               int32_t* d_ids, float* d_dists, bool whole, hipStream_t st) {
  CallMemory partial(st);
  int S = 0;
  if (sizeof(T) == 1 && whole && dim <= 4 * kGtWords && k <= kGtMaxK) {
    if constexpr (sizeof(T) == 1) {
      const int64_t groups = (nq + 255) / 256;
      const int64_t tiles = (n + kGtTile - 1) / kGtTile;
      S = (int)std::max<int64_t>(1, std::min<int64_t>({256, tiles, (2048 + groups - 1) / groups}));
      const int64_t slice = (tiles + S - 1) / S * kGtTile;
      HIP_OK(partial.take(sizeof(uint64_t) * (size_t)(nq * S * k)));
      hipLaunchKernelGGL(gt_int_kernel<T>, dim3((unsigned)groups, (unsigned)S), dim3(256), 0, st, d_base, n, dim, d_q,
                         which, nq, k, slice, S, partial.as<uint64_t>());
    }
  } else {
    S = (int)std::max<int64_t>(1, std::min<int64_t>(64, 4096 / std::max<int64_t>(1, (nq + kGtQ - 1) / kGtQ)));
    const int64_t slice = (n + S - 1) / S;
    HIP_OK(partial.take(sizeof(uint64_t) * (size_t)(nq * S * k)));
    const size_t lds = (size_t)kGtQ * dim * 4 + (size_t)kGtQ * 4 * kWave * 8;
    hipLaunchKernelGGL(gt_kernel<T>, dim3((unsigned)((nq + kGtQ - 1) / kGtQ), (unsigned)S), dim3(256), lds, st, d_base,
                       n, dim, d_q, which, nq, k, slice, S, partial.as<uint64_t>());
  }
  HIP_OK(hipGetLastError());
  hipLaunchKernelGGL(gt_final_kernel, dim3((unsigned)std::min<int64_t>(nq, 65536)), dim3(64), 0, st,
                     partial.as<uint64_t>(), which, nq, S, k, d_ids, d_dists);
  HIP_OK(hipGetLastError());
}

// The whole call by the scan, then the direct kernels for the queries that
// left it (*direct of them).  false: nothing was launched, its memory (lists of
// 4 KB a query up to k = 16, of 16 KB beyond) could not be had.
template <class T, int KS, int QT>
bool gt_matrix_ks(const T* d_base, int64_t n, int dim, const float* d_q, int64_t nq, int k, int32_t* d_ids,
                  float* d_dists, int device, int64_t* direct, hipStream_t st) {
  const void* const fn = reinterpret_cast<const void*>(&gt_scan_kernel<T, KS, QT>);
  HIP_OK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, gt_scan_lds<T>(KS, QT)));
  int per_cu = 0, cus = 0;
  HIP_OK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, 256, (size_t)gt_scan_lds<T>(KS, QT)));
  HIP_OK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  const int cap = k <= 16 ? 512 : 2048;  // level 0 keeps up to 256 (1024) rows, a later one about 3 k
  const int64_t batch = std::min<int64_t>(nq, kGtBatch), batches = (nq + batch - 1) / batch;
  const int64_t padded = (batch + 128 * QT - 1) / (128 * QT) * (128 * QT);
  const size_t lists = (size_t)batch * cap * 8 + (size_t)padded * (8 + 12 + GtKind<T>::kPlanes * KS * 32);
  const size_t state = sizeof(GtCall) + (size_t)batches * sizeof(GtLeft);
  CallMemory memory(st);
  const hipError_t got = memory.take(lists + state + (size_t)nq * 8 + kGtCenter * 4);
  if (got == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    return false;
  }
  HIP_OK(got);
  uint8_t* const work = memory.as<uint8_t>();
  GtCall* const call = reinterpret_cast<GtCall*>(work + lists);
  GtLeft* const left = reinterpret_cast<GtLeft*>(call + 1);
  int64_t* const listed = reinterpret_cast<int64_t*>(left + batches);
  float* const center = reinterpret_cast<float*>(listed + nq);
  hipLaunchKernelGGL(gt_start_kernel<T>, dim3(1), dim3(kGtCenter), 0, st, d_base, n, dim, reinterpret_cast<uint32_t*>(call),
                     (int64_t)state / 4, center);
  HIP_OK(hipGetLastError());
  for (int64_t q = 0, b = 0; q < nq; q += batch, b++)
    gt_levels<T, KS, QT>(d_base, n, dim, d_q + q * dim, std::min(batch, nq - q), k, d_ids + q * k, d_dists + q * k, cap,
                         (int64_t)per_cu * cus, work, center, left + b, q, call, listed, st);
  GtCall host{};
  HIP_OK(hipMemcpyAsync(&host, call, sizeof(host), hipMemcpyDeviceToHost, st));
  HIP_OK(hipStreamSynchronize(st));
  *direct = (int64_t)host.direct;
  if (host.direct > 0) {
    gt_direct<T>(d_base, n, dim, d_q, listed, (int64_t)host.direct, k, d_ids, d_dists, !host.fractional, st);
    HIP_OK(hipStreamSynchronize(st));
  }
  return true;
}

// The matrix-core path where it applies; false for rows longer than its tiles
// and where its memory cannot be had.
template <class T>
bool gt_matrix(const T* d_base, int64_t n, int dim, const float* d_q, int64_t nq, int k, int32_t* d_ids,
               float* d_dists, int device, int64_t* direct, hipStream_t st) {
  const bool few = nq <= 256;  // one query tile per wave: a workgroup then holds 128 queries, not 256 or 512
#define QV_GT(KS, QT) return gt_matrix_ks<T, KS, QT>(d_base, n, dim, d_q, nq, k, d_ids, d_dists, device, direct, st)
  if constexpr (sizeof(T) == 4) {
    if (dim > 128) return false;
    if (few) {
      if (dim <= 32) QV_GT(2, 1);
      if (dim <= 64) QV_GT(4, 1);
      if (dim <= 96) QV_GT(6, 1);
      QV_GT(8, 1);
    }
    if (dim <= 32) QV_GT(2, 2);
    if (dim <= 64) QV_GT(4, 2);
    if (dim <= 96) QV_GT(6, 2);
    QV_GT(8, 2);
  } else {
    if (dim > 256) return false;
    if (few) {
      if (dim <= 64) QV_GT(2, 1);
      if (dim <= 128) QV_GT(4, 1);
      QV_GT(8, 1);
    }
    if (dim <= 64) QV_GT(2, 4);
    if (dim <= 128) QV_GT(4, 4);
    QV_GT(8, 2);
  }
#undef QV_GT
}

// Whether a call is too small for the scan's levels, whose launches and lists
// cost more than they save.  Float rows: up to half a million pairs (1,000 rows
// x 100 queries x 96: 0.16 ms direct, 0.19 by the scan; 1,000 x 1,000: 0.33 and
// 0.26) over few rows, which the direct kernel spreads over 64 workgroups per 8
// queries (4,000 rows x 1 query: 0.20 and 0.18).  8-bit rows with more queries than one
// small workgroup of the scan takes (with fewer the scan is the faster one at
// any size): five million pairs of the integer kernel (60 x 1,000 x 128: 0.20
// and 0.26; 300 x 10,000: 0.31 and 0.34; 2,000 x 10,000: 0.44 and 0.37), of the
// fp32 kernel 600,000 (300 x 300, k = 50: 0.25 and 0.28; 1,000 x 1,000: 0.39
// and 0.34).
template <class T>
bool gt_small(int64_t n, int dim, int64_t nq, int k) {
  if (sizeof(T) == 4) return n <= 2048 && n * nq <= 500000;
  return dim <= 4 * kGtWords && nq > 256 && n * nq <= (k <= kGtMaxK ? 5000000 : 600000);
}

// direct: how many of the queries the direct kernels answered.
template <class T>
void ground_truth_t(const T* d_base, int64_t n, int dim, const float* d_q, int64_t nq, int k, int32_t* d_ids,
                    float* d_dists, int device, bool scan_small, int64_t* direct, hipStream_t st) {
  if ((scan_small || !gt_small<T>(n, dim, nq, k)) &&
      gt_matrix<T>(d_base, n, dim, d_q, nq, k, d_ids, d_dists, device, direct, st)) return;
  *direct = nq;
  int32_t bad = 1;
  if constexpr (sizeof(T) == 1) {
    if (dim <= 4 * kGtWords && k <= kGtMaxK) {
      CallMemory flag(st);
      HIP_OK(flag.take(sizeof(int32_t)));
      HIP_OK(hipMemsetAsync(flag.p, 0, sizeof(int32_t), st));
      hipLaunchKernelGGL(gt_query_check<T>, dim3((unsigned)grid_of(nq * dim, 256)), dim3(256), 0, st, d_q, nq * dim,
                         flag.as<int32_t>());
      HIP_OK(hipGetLastError());
      HIP_OK(hipMemcpyAsync(&bad, flag.p, sizeof(bad), hipMemcpyDeviceToHost, st));
      HIP_OK(hipStreamSynchronize(st));
    }
  }
  gt_direct<T>(d_base, n, dim, d_q, nullptr, nq, k, d_ids, d_dists, !bad, st);
  HIP_OK(hipStreamSynchronize(st));
}

}  // namespace

extern "C" {

int qv_ground_truth_counted(const void* d_base, int32_t data_type, int64_t n, int32_t dim, const float* d_queries,
                            int64_t nq, int32_t k, int32_t* d_ids, float* d_dists, int device, int32_t scan_small,
                            int64_t* direct) {
  return qv::guard([&] {
    if (!d_base || !d_queries || !d_ids || !d_dists) qv::fail(QV_EINVAL, "null argument");
    if (k <= 0 || k > 64 || n <= 0 || n > INT32_MAX || nq <= 0 || dim <= 0) qv::fail(QV_EINVAL, "bad shape");
    if ((dim * (data_type == QV_FLOAT ? 4 : 1)) % 4) qv::fail(QV_EUNSUPPORTED, "row bytes must be a multiple of 4");
    HIP_OK(hipSetDevice(device));
    hipStream_t st;
    HIP_OK(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
    std::unique_ptr<std::remove_pointer<hipStream_t>::type, void (*)(hipStream_t)> owned(
        st, [](hipStream_t s) { (void)hipStreamDestroy(s); });
    auto go = [&](auto* base) {
      ground_truth_t(base, n, dim, d_queries, nq, k, d_ids, d_dists, device, scan_small != 0, direct, st);
    };
    if (data_type == QV_UINT8) go(static_cast<const uint8_t*>(d_base));
    else if (data_type == QV_INT8) go(static_cast<const int8_t*>(d_base));
    else go(static_cast<const float*>(d_base));
  });
}

int qv_ground_truth(const void* d_base, int32_t data_type, int64_t n, int32_t dim, const float* d_queries,
                    int64_t nq, int32_t k, int32_t* d_ids, float* d_dists, int device) {
  int64_t direct = 0;
  return qv_ground_truth_counted(d_base, data_type, n, dim, d_queries, nq, k, d_ids, d_dists, device, 0, &direct);
}

}  // extern "C"
