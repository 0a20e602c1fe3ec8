// The host side of src/kernels/blas.hip against a HIP runtime and a rocBLAS
// that only write down their calls: in what order do products queued on
// several streams reach the library's one workspace?  No GPU.  Prints "ok".
#include <hip/hip_runtime_api.h>
#include <rocblas/rocblas.h>

#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "mk_kernels.h"

namespace {
typedef std::set<int> Done;           // products that are finished before ...
std::map<hipStream_t, Done> g_after;  // ... whatever a stream takes next
std::map<hipEvent_t, Done> g_event;
std::map<hipStream_t, bool> g_capturing;
std::vector<std::pair<int, Done>> g_products[2];  // by device: product, what it waits for
int g_device = 0, g_next = 0, g_own = 0, g_events = 0, g_synced = 0;
bool g_record_fails = false;
hipStream_t g_blas_stream[2];

hipStream_t stream(int i) { return reinterpret_cast<hipStream_t>(uintptr_t(16 * (i + 1))); }

int product(int s, int64_t m = 256) {
  static uint16_t a[64], c[64];
  return mk_gemm_blas(stream(s), MK_BF16, MK_BF16, 1, m, 256, 256, a, 0, 256, 1, a, 0, 256, 1, c, 0, 256, 1.f, 0.f);
}

// every product on a device waits for all before it
bool ordered(int dev) {
  for (size_t i = 0; i < g_products[dev].size(); ++i)
    for (size_t j = 0; j < i; ++j)
      if (!g_products[dev][i].second.count(g_products[dev][j].first)) return false;
  return true;
}

void expect(bool ok, const char* what) {
  if (ok) return;
  std::printf("FAILED: %s\n", what);
  std::exit(1);
}
}  // namespace

// ---------------------------------------------------------------- the runtime
extern "C" {
hipError_t hipGetDevice(int* d) { return *d = g_device, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(uintptr_t(0x1000 + 16 * ++g_events));
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (g_record_fails) return hipErrorUnknown;
  g_event[e] = g_after[s];
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  g_after[s].insert(g_event[e].begin(), g_event[e].end());
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  ++g_synced;
  for (int i = 0; i < 4; ++i) g_after[stream(i)].insert(g_after[s].begin(), g_after[s].end());
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) {
  const auto at = g_capturing.find(s);  // asked by threads outside any lock
  *c = at != g_capturing.end() && at->second ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }

// ---------------------------------------------------------------- the library
rocblas_status rocblas_create_handle(rocblas_handle* h) {
  *h = reinterpret_cast<rocblas_handle>(uintptr_t(1 + g_device));
  return rocblas_status_success;
}
rocblas_status rocblas_set_pointer_mode(rocblas_handle, rocblas_pointer_mode) { return rocblas_status_success; }
rocblas_status rocblas_set_stream(rocblas_handle h, hipStream_t s) {
  g_blas_stream[reinterpret_cast<uintptr_t>(h) - 1] = s;
  return rocblas_status_success;
}
const char* rocblas_status_to_string(rocblas_status) { return "status"; }
rocblas_status rocblas_gemm_strided_batched_ex(rocblas_handle h, rocblas_operation, rocblas_operation, rocblas_int,
                                               rocblas_int, rocblas_int, const void*, const void*, rocblas_datatype,
                                               rocblas_int, rocblas_stride, const void*, rocblas_datatype, rocblas_int,
                                               rocblas_stride, const void*, const void*, rocblas_datatype, rocblas_int,
                                               rocblas_stride, void*, rocblas_datatype, rocblas_int, rocblas_stride,
                                               rocblas_int, rocblas_datatype, rocblas_gemm_algo, int32_t, uint32_t) {
  const int dev = int(reinterpret_cast<uintptr_t>(h)) - 1;
  const hipStream_t s = g_blas_stream[dev];
  expect(!g_capturing[s], "a library kernel in a captured graph");
  g_products[dev].push_back({g_next, g_after[s]});
  g_after[s].insert(g_next++);
  return rocblas_status_success;
}
}

// ---------------------------------------------------------------- the rest of this library
namespace mk {
void clear_error() {}
int fail(int code, const std::string&) { return code; }
int check_launch(const char*) { return MK_OK; }
int gemm_own(hipStream_t, int, int, int64_t, int64_t, int64_t, int64_t, const void*, int64_t, int64_t, int64_t,
             const void*, int64_t, int64_t, int64_t, void*, int64_t, int64_t, float, float) {
  return ++g_own, MK_OK;
}
}  // namespace mk

int main() {
  for (int s : {0, 1, 0, 0, 2, 1}) expect(product(s) == MK_OK, "product");
  expect(g_products[0].size() == 6 && ordered(0), "products on three streams share the workspace one at a time");

  // the split form's batched product too
  static float w[64];
  const int rc = mk_gemm_blas_splitk(stream(2), MK_BF16, 256, 256, 512, w, 512, 1, w, 256, 1, w, 256, 2, w);
  expect(rc == MK_OK && g_products[0].size() == 7 && ordered(0), "the split form takes its turn");

  // refused products leave the order as it is
  expect(mk_gemm_blas(stream(1), MK_BF16, MK_BF16, 1, 8, 8, 8, nullptr, 0, 8, 1, w, 0, 8, 1, w, 0, 8, 1.f, 0.f) ==
             MK_ERR_INVALID, "null operand");
  product(1);
  expect(g_products[0].size() == 8 && ordered(0), "a refused product between");

  // captured: no library kernel, no event of the eager order in the graph
  g_capturing[stream(3)] = true;
  const Done before = g_after[stream(3)];
  expect(product(3) == MK_OK && g_own == 1, "a captured product runs on this library's kernels");
  expect(g_products[0].size() == 8 && g_after[stream(3)] == before, "and waits for nothing outside its graph");
  g_capturing[stream(3)] = false;
  product(3);
  expect(g_products[0].size() == 9 && ordered(0), "eager products after a capture");

  // GPUs have orders of their own
  g_device = 1;
  product(0), product(1);
  expect(g_products[1].size() == 2 && ordered(1), "the second GPU");
  g_device = 0;

  // an event that cannot be recorded: the turn ends when its kernels have
  g_record_fails = true;
  product(0);
  g_record_fails = false;
  product(1);
  expect(g_synced == 1 && ordered(0), "no event");

  // several threads
  std::vector<std::thread> threads;
  for (int t = 0; t < 4; ++t) threads.emplace_back([t] { for (int i = 0; i < 50; ++i) product(t); });
  for (auto& t : threads) t.join();
  expect(ordered(0), "four threads, a stream each");
  std::printf("ok\n");
}
