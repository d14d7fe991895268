#include "standin.h"

#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <mutex>

namespace standin {
size_t limit = (size_t)1 << 40;
static std::mutex mu;
static std::map<const char*, size_t> blocks;
static size_t in_use = 0;
static hipError_t last = hipSuccess;  // as hipGetLastError would return it

size_t used() {
  std::lock_guard<std::mutex> lk(mu);
  return in_use;
}
size_t size_of(const void* p) {
  std::lock_guard<std::mutex> lk(mu);
  auto it = blocks.upper_bound((const char*)p);
  if (it == blocks.begin()) return 0;
  --it;
  return (const char*)p < it->first + it->second ? it->second : 0;
}
std::function<int(int, const sxc::ForwardArgs&)> on_forward;
std::function<int(int, bool, const sxc::PairArgs&)> on_pairs;
std::function<int(int, const sxc::ResolveArgs&)> on_resolve;
std::function<int(const sxc::LagPrepArgs&)> on_lag_prep;
std::function<int(bool, const sxc::LagPairArgs&)> on_lag_pairs;
}  // namespace standin

using namespace standin;

extern "C" {
#undef hipMalloc
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  *p = nullptr;
  if (n > limit || in_use > limit - n) return last = hipErrorOutOfMemory;
  *p = calloc(n ? n : 1, 1);
  blocks[(const char*)*p] = n;
  in_use += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(mu);
  auto it = blocks.find((const char*)p);
  if (it != blocks.end()) {
    in_use -= it->second;
    blocks.erase(it);
    free(p);
  }
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = malloc(n ? n : 1);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
  memset(d, v, n);
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
  return hipSuccess;
}
}

namespace sxc {
template <typename F, typename... A>
static hipError_t call(const F& f, const A&... a) {
  return f && f(a...) ? hipErrorLaunchFailure : hipGetLastError();  // the launchers report it
}
hipError_t launch_forward(int R, const ForwardArgs& a, hipStream_t) {
  if (a.zero) *a.zero = 0u;
  return call(on_forward, R, a);
}
hipError_t launch_pairs(int R, bool full, const PairArgs& a, int, hipStream_t) { return call(on_pairs, R, full, a); }
hipError_t launch_resolve(int R, const ResolveArgs& a, int, hipStream_t) { return call(on_resolve, R, a); }
hipError_t launch_lag_prep(const LagPrepArgs& a, hipStream_t) { return call(on_lag_prep, a); }
hipError_t launch_lag_pairs(bool bf16x3, LagPairArgs a, hipStream_t) { return call(on_lag_pairs, bf16x3, a); }
hipError_t launch_lag_tiles(bool bf16x3, const LagPairArgs& a, hipStream_t) { return call(on_lag_pairs, bf16x3, a); }
hipError_t launch_fill_u32(unsigned* p, unsigned v, int n, hipStream_t) {
  for (int k = 0; k < n; ++k) p[k] = v;
  return hipSuccess;
}
hipError_t launch_copy_f4(float4*, const float4*, long long, hipStream_t) { return hipSuccess; }
hipError_t launch_topk(const float*, const int*, int, int, int, float*, int*, int*, hipStream_t) { return hipSuccess; }
hipError_t launch_topk_split(const float*, const int*, int, int, int, int, float*, int*, int*, float*, int*, int*,
                             hipStream_t) {
  return hipSuccess;
}
hipError_t launch_hist_threshold(const HistArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_lag_resolve(const LagResolveArgs&, int, hipStream_t) { return hipSuccess; }
hipError_t launch_pack_block(const PackBlockArgs&, hipStream_t) { return hipSuccess; }
}  // namespace sxc
