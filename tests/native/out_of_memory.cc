// mlba_create and mlba_set_landmark_active where host or device memory runs
// out: every allocation of a small map is failed in turn, alone and with all
// that follow it. Neither call may end the process; they return a status, and
// a handle that could not be rebuilt refuses to run until it is. The HIP
// runtime is replaced by the functions below (device memory is host memory,
// launches do nothing); no GPU is needed.
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "maplab_ba.h"

static std::atomic<long> g_left{-1};  // allocations until one fails; < 0: none does
static std::atomic<bool> g_all{false};  // all that follow fail too
static std::atomic<long> g_count{0}, g_live{0};

static bool fails() {
  ++g_count;
  if (g_left < 0) return false;
  const long left = g_left.fetch_sub(1);
  if (left > 0) return false;
  if (g_all) g_left = 0;
  return true;
}
static void* host(std::size_t n) {
  if (fails()) throw std::bad_alloc();
  void* p = std::malloc(n ? n : 1);
  if (!p) std::abort();
  return p;
}
void* operator new(std::size_t n) { return host(n); }
void* operator new[](std::size_t n) { return host(n); }
void* operator new(std::size_t n, const std::nothrow_t&) noexcept { return fails() ? nullptr : std::malloc(n); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete[](void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
void operator delete[](void* p, std::size_t) noexcept { std::free(p); }

static hipError_t device(void** p, size_t n) {
  *p = nullptr;
  if (fails()) return hipErrorOutOfMemory;
  *p = std::malloc(n ? n : 1);
  ++g_live;
  return hipSuccess;
}
extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return device(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return device(p, n); }
hipError_t hipFree(void* p) {
  if (p) --g_live;
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = reinterpret_cast<hipStream_t>(8);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(8);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
}

#define CHECK(x)                                                                          \
  do {                                                                                    \
    if (!(x)) {                                                                           \
      std::printf("line %d: %s (allocation %ld, all %d)\n", __LINE__, #x, n, (int)all);   \
      return 1;                                                                           \
    }                                                                                     \
  } while (0)

int main() {
  // 40 vertices on a line, each landmark seen by six neighbours.
  const int P = 40, L = 400;
  std::vector<double> vert, lm(3 * L, 1.0), kp, sigma;
  std::vector<int32_t> mission(P, 0), store(L), ov, ol, oc;
  for (int v = 0; v < P; ++v)
    for (double x : {0.0, 0.0, 0.0, 1.0, 0.1 * v, 0.0, 0.0}) vert.push_back(x);
  for (int l = 0; l < L; ++l) {
    store[l] = l % P;
    for (int k = 0; k < 6; ++k) {
      ov.push_back((l + k) % P);
      ol.push_back(l);
      oc.push_back(0);
      kp.insert(kp.end(), {100.0, 100.0});
      sigma.push_back(1.0);
    }
  }
  const double frame[7] = {0, 0, 0, 1, 0, 0, 0}, intr[4] = {400, 400, 300, 200}, dist[4] = {0, 0, 0, 0};
  const int32_t dtype = 0, size[2] = {640, 480};
  std::vector<uint8_t> vconst(P, 0);
  vconst[0] = 1;
  mlba_problem_desc d;
  std::memset(&d, 0, sizeof(d));
  d.num_vertices = P;
  d.num_missions = 1;
  d.num_cameras = 1;
  d.num_landmarks = L;
  d.num_observations = (int32_t)ov.size();
  d.vertex_q_IM__M_p_MI = vert.data();
  d.vertex_mission = mission.data();
  d.vertex_constant = vconst.data();
  d.baseframe_q_GM__G_p_GM = frame;
  d.camera_q_CI__C_p_CI = frame;
  d.camera_intrinsics = intr;
  d.camera_distortion = dist;
  d.camera_distortion_type = &dtype;
  d.camera_resolution = size;
  d.landmark_p_B = lm.data();
  d.landmark_store_vertex = store.data();
  d.obs_vertex = ov.data();
  d.obs_landmark = ol.data();
  d.obs_camera = oc.data();
  d.obs_keypoint = kp.data();
  d.obs_sigma = sigma.data();
  std::vector<uint8_t> some(L, 1), every(L, 1), good(L, 0);
  for (int l = 0; l < L; l += 3) some[l] = 0;
  mlba_quality_options q;
  mlba_quality_options_init(&q);
  long failed_create = 0, failed_mask = 0;
  for (bool all : {false, true})
    for (long n = 0;; ++n) {
      mlba_handle* h = nullptr;
      g_all = all;
      g_left = n;
      int32_t rc = mlba_create(&d, &h);
      const bool reached = g_left < 0 || (all && g_left == 0);
      g_left = -1;
      if (rc && rc != MLBA_ENOMEM) std::printf("%d: %s\n", rc, mlba_last_error(nullptr));
      CHECK(rc == MLBA_OK || (rc == MLBA_ENOMEM && h == nullptr));
      if (rc == MLBA_ENOMEM) {
        ++failed_create;
        CHECK(reached && mlba_last_error(nullptr) != nullptr);
        CHECK(g_live == 0);
        continue;
      }
      CHECK(mlba_destroy(h) == MLBA_OK && g_live == 0);
      if (!reached) break;
    }
  for (bool all : {false, true})
    for (long n = 0;; ++n) {
      mlba_handle* h = nullptr;
      int32_t rc = mlba_create(&d, &h);
      CHECK(rc == MLBA_OK && mlba_set_landmark_active(h, some.data()) == MLBA_OK);
      g_all = all;
      g_left = n;
      rc = mlba_set_landmark_active(h, every.data());
      const bool reached = g_left < 0 || (all && g_left == 0);
      g_left = -1;
      CHECK(rc == MLBA_OK || rc == MLBA_ENOMEM);
      CHECK(mlba_landmark_quality(h, &q, good.data()) == (rc == MLBA_OK ? MLBA_OK : MLBA_ESTATE));
      if (rc != MLBA_OK) {
        ++failed_mask;
        mlba_options o;
        mlba_options_init(&o);
        CHECK(mlba_solve(h, &o, nullptr) == MLBA_ESTATE);
        CHECK(mlba_set_landmark_active(h, every.data()) == MLBA_OK);
        CHECK(mlba_landmark_quality(h, &q, good.data()) == MLBA_OK);
      }
      CHECK(mlba_destroy(h) == MLBA_OK && g_live == 0);
      if (!reached) break;
    }
  std::printf("create failed %ld times, the mask %ld times\n", failed_create, failed_mask);
  return failed_create > 100 && failed_mask > 50 ? 0 : 2;
}
