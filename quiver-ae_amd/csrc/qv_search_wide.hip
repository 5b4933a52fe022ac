// qv_search_wide.hip -- the per-query-LUT search kernels for a top-k above 64
// (the reference's retset_push_32 path, gpu_primitives.cuh:99-138, for any
// k): entries 0 .. 63 in the wave's registers as in every other kernel,
// entries 64 .. k - 1 in LDS after the query's area.  Kept apart from the
// other kernels so theirs stay exactly as they are; every element type, PQ
// layout and neighbour-slot count, beams of Q = 2, 4, 7, 10 or 16 positions
// per lane.
#include "qv_search_kernels.hpp"

namespace {

template <class T, int Q, int NPL>
KernelFn wide_mc(int M) {
  if constexpr (NPL == 1 && Q <= 7) {
    if (M == 32) return search_kernel_team<T, Q, 32, true>;
    if (M == 48) return search_kernel_team<T, Q, 48, true>;
  } else {
    if (M == 32) return search_kernel<T, Q, 32, NPL, true>;
    if (M == 48) return search_kernel<T, Q, 48, NPL, true>;
  }
  return search_kernel<T, Q, 0, NPL, true>;
}

// The one-wave kernel where it holds half again as many queries per CU as the
// team (launch_plan): 48-chunk LUTs beside beams of four positions per lane,
// three instead of two.
template <class T>
KernelFn one_wave(int Q, int M) {
  return Q == 4 && M == 48 ? search_kernel<T, 4, 48, 1, true> : nullptr;
}

template <class T, int NPL>
KernelFn wide_q(int Q, int M) {
  switch (Q) {
    case 2: return wide_mc<T, 2, NPL>(M);
    case 4: return wide_mc<T, 4, NPL>(M);
    case 7: return wide_mc<T, 7, NPL>(M);
    case 10: return wide_mc<T, 10, NPL>(M);
    case 16: return wide_mc<T, 16, NPL>(M);
    default: return nullptr;
  }
}

template <class T>
KernelFn wide_npl(int Q, int M, int npl) {
  return npl > 1 ? wide_q<T, 2>(Q, M) : wide_q<T, 1>(Q, M);
}

}  // namespace

namespace qv {
namespace sk {

KernelFn pick_kernel_wide(int dtype, int Q, int M, int npl) {
  if (dtype == QV_UINT8) return wide_npl<uint8_t>(Q, M, npl);
  if (dtype == QV_INT8) return wide_npl<int8_t>(Q, M, npl);
  return wide_npl<float>(Q, M, npl);
}

KernelFn pick_kernel_wide_one_wave(int dtype, int Q, int M) {
  if (dtype == QV_UINT8) return one_wave<uint8_t>(Q, M);
  if (dtype == QV_INT8) return one_wave<int8_t>(Q, M);
  return one_wave<float>(Q, M);
}

}  // namespace sk
}  // namespace qv
