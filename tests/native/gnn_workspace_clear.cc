// The network workspace is cleared on the stream that uses it, and a workspace
// that could not be cleared is not handed out. The HIP runtime is replaced by
// the few functions below; no GPU is needed.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>

#include "ba_learned.h"

static size_t g_allocated = 0;
static int g_live = 0, g_clears = 0, g_null_clears = 0;
static hipStream_t g_stream = nullptr;
static size_t g_cleared = 0;
static hipError_t g_malloc_result = hipSuccess, g_memset_result = hipSuccess;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (g_malloc_result != hipSuccess) return g_malloc_result;
  *p = std::malloc(n);
  g_allocated = n;
  ++g_live;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::free(p);
  --g_live;
  return hipSuccess;
}
hipError_t hipMemset(void*, int, size_t) {
  ++g_null_clears;
  return g_memset_result;
}
hipError_t hipMemsetAsync(void*, int, size_t n, hipStream_t s) {
  ++g_clears;
  g_stream = s;
  g_cleared = n;
  return g_memset_result;
}
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipErrorUnknown; }
hipError_t hipDeviceSynchronize() { return hipErrorUnknown; }
hipError_t hipGetLastError() { return hipErrorUnknown; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipErrorUnknown; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipErrorUnknown; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipErrorUnknown; }
// The host half of a HIP object registers its kernels before main.
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
}

#define CHECK(x)                                       \
  do {                                                 \
    if (!(x)) {                                        \
      std::printf("line %d: %s\n", __LINE__, #x);      \
      return 1;                                        \
    }                                                  \
  } while (0)

int main() {
  const hipStream_t s = reinterpret_cast<hipStream_t>(0x1234);
  for (bool training : {false, true}) {
    mlba::GnnWorkspace* w = mlba::gnn_workspace_create(s, 300, 4000, training);
    CHECK(w);
    CHECK(g_clears == 1 && g_null_clears == 0);
    CHECK(g_stream == s);
    CHECK(g_cleared == g_allocated);
    mlba::gnn_workspace_destroy(w);
    CHECK(g_live == 0);
    g_clears = 0;
  }
  g_memset_result = hipErrorUnknown;
  CHECK(mlba::gnn_workspace_create(s, 300, 4000, false) == nullptr);
  CHECK(g_live == 0);
  g_memset_result = hipSuccess;
  g_malloc_result = hipErrorOutOfMemory;
  CHECK(mlba::gnn_workspace_create(s, 300, 4000, false) == nullptr);
  CHECK(g_live == 0);
  std::printf("ok\n");
  return 0;
}
