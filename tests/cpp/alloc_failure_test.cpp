// The library's host code when an allocation fails, without a GPU: this
// program defines the HIP calls that libquiver_hip.so makes ("device" memory
// is host memory, a kernel launch does nothing), so the library binds to them,
// and one allocation after the other is refused.
//   alloc_failure_test build  a GPU build refused its i-th allocation, for
//                             every i the call reaches, fails and frees
//                             nothing twice
//   alloc_failure_test truth  ground truth whose first allocation (the matrix
//                             scan's lists) is refused still runs, and whichever
//                             is refused leaves no memory and no stream behind
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <vector>

#include "quiver_hip.h"

namespace {

std::set<void*> live;       // allocations not freed yet
long allocs = 0;            // allocations asked for
long refuse = 0;            // the one to refuse (from 1; 0: none)
long double_frees = 0;
long launches = 0;
long streams = 0;           // created and not destroyed

hipError_t take(void** p, size_t bytes) {
  *p = nullptr;
  if (++allocs == refuse) return hipErrorOutOfMemory;
  *p = std::calloc(1, bytes > 0 ? bytes : 1);
  live.insert(*p);
  return hipSuccess;
}
// (the memory itself is kept: an address is handed out once)
hipError_t give(void* p) {
  if (p != nullptr && live.erase(p) == 0) double_frees++;
  return hipSuccess;
}

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n); }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return take(p, n); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipFreeAsync(void* p, hipStream_t) { return give(p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(8);
  return streams++, hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return streams--, hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(8), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) {
  std::memset(a, 0, sizeof(*a));
  a->maxThreadsPerBlock = 1024;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { return *n = 2, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256
       : a == hipDeviceAttributeMaxSharedMemoryPerMultiprocessor ? 160 * 1024
       : a == hipDeviceAttributeWarpSize ? 64 : 1;
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // (the header's macro names its current form)
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  return hipSuccess;
}
// launches: the configuration is only passed through
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return launches++, hipSuccess; }
}

static int build_refused() {
  const int64_t n = 300;
  const int32_t dim = 32;
  std::vector<uint8_t> base((size_t)n * dim);
  for (size_t i = 0; i < base.size(); i++) base[i] = (uint8_t)(i * 37 % 251);
  qv_build_params p;
  qv_build_params_default(&p);
  p.R = 8;
  p.L = 16;
  p.num_chunks = 8;
  p.kmeans_iters = 1;
  long reached = 0;
  for (refuse = 1; refuse < 1000; refuse++) {
    allocs = 0;
    qv_index* ix = nullptr;
    const int rc = qv_build_index_gpu(base.data(), QV_UINT8, n, dim, &p, 0, &ix);
    if (allocs < refuse) break;  // everything it asks for was given (no kernel ran: it fails in its first search)
    reached = refuse;
    if (rc != QV_ENOMEM || ix != nullptr || double_frees != 0) {
      std::printf("allocation %ld refused: status %d (%s), %ld double frees\n", refuse, rc, qv_last_error(), double_frees);
      return 1;
    }
  }
  std::printf("%ld allocations refused in turn, %ld launches, nothing freed twice\n", reached, launches);
  return reached >= 20 ? 0 : 1;
}

static int truth_refused() {
  const int64_t n = 5000, nq = 300;
  const int32_t dim = 32, k = 50;
  std::vector<float> base((size_t)n * dim, 1.f), q((size_t)nq * dim, 2.f), dists((size_t)nq * k);
  std::vector<int32_t> ids((size_t)nq * k);
  for (int32_t type : {QV_UINT8, QV_INT8, QV_FLOAT}) {
    for (refuse = 0; refuse <= 1; refuse++) {
      allocs = launches = 0;
      const int rc = qv_ground_truth(base.data(), type, n, dim, q.data(), nq, k, ids.data(), dists.data(), 0);
      if (rc != QV_OK || launches < 2 || !live.empty() || double_frees != 0) {
        std::printf("type %d, allocation %ld refused: status %d (%s), %ld launches, %zu allocations left\n", type, refuse,
                    rc, qv_last_error(), launches, live.size());
        return 1;
      }
    }
    // few rows: the direct kernels' own check and partial results
    for (int32_t kk : {10, 50}) {
      for (refuse = 1;; refuse++) {
        allocs = 0;
        const int rc = qv_ground_truth(base.data(), type, 100, dim, q.data(), nq, kk, ids.data(), dists.data(), 0);
        if (!live.empty() || streams != 0 || double_frees != 0 || (rc != QV_OK && rc != QV_ENOMEM)) {
          std::printf("type %d, k %d, allocation %ld refused: status %d (%s), %zu allocations and %ld streams left\n", type,
                      kk, refuse, rc, qv_last_error(), live.size(), streams);
          return 1;
        }
        if (allocs < refuse) break;
      }
    }
  }
  std::printf("ground truth ran without its first allocation\n");
  return 0;
}

int main(int argc, char** argv) {
  if (argc == 2 && std::strcmp(argv[1], "build") == 0) return build_refused();
  if (argc == 2 && std::strcmp(argv[1], "truth") == 0) return truth_refused();
  std::fprintf(stderr, "usage: alloc_failure_test build|truth\n");
  return 2;
}
