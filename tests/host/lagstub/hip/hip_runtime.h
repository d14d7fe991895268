// Host stand-in of the few HIP names xc_lag.hip uses, so that its load
// addresses can be checked lane by lane on the CPU.  Buffer loads record the
// bytes they touch; matrix products leave the accumulator as it is.
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>

#define __device__
#define __host__
#define __global__ [[maybe_unused]]
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)

struct dim3 { unsigned x = 1, y = 1, z = 1; dim3(unsigned a = 1) : x(a) {} };
static dim3 threadIdx(0), blockIdx(0), gridDim(1);
struct int2 { int x, y; };
struct int4 { int x, y, z, w; };
inline int2 make_int2(int a, int b) { return {a, b}; }
inline int4 make_int4(int a, int b, int c, int d) { return {a, b, c, d}; }
typedef void* hipStream_t;
enum hipError_t { hipSuccess = 0 };
inline hipError_t hipGetLastError() { return hipSuccess; }
#define hipLaunchKernelGGL(...) ((void)0)  // no kernel body is compiled

template <typename T> T min(T a, T b) { return a < b ? a : b; }
template <typename T> T max(T a, T b) { return a > b ? a : b; }
inline unsigned __float_as_uint(float f) { unsigned u; memcpy(&u, &f, 4); return u; }
inline int __float_as_int(float f) { int u; memcpy(&u, &f, 4); return u; }
inline float __uint_as_float(unsigned u) { float f; memcpy(&f, &u, 4); return f; }
inline float __int_as_float(int u) { float f; memcpy(&f, &u, 4); return f; }
inline void __syncthreads() {}
template <typename T> T __shfl_xor(T v, int, int) { return v; }
inline unsigned long long __ballot(bool b) { return b; }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline unsigned atomicAdd(unsigned* p, unsigned v) { unsigned o = *p; *p += v; return o; }
#define __builtin_amdgcn_readfirstlane(x) (x)

struct BufferRsrc { const void* base; int bytes; };
#define __amdgpu_buffer_rsrc_t BufferRsrc
#define __builtin_amdgcn_make_buffer_rsrc(p, stride, n, flags) BufferRsrc{p, n}
typedef unsigned stub_u32x4 __attribute__((ext_vector_type(4)));
void on_buffer_load(const BufferRsrc& r, int voff, int soff, int bytes);
inline stub_u32x4 stub_load_b128(BufferRsrc r, int voff, int soff) {
  on_buffer_load(r, voff, soff, 16);
  return stub_u32x4{0, 0, 0, 0};
}
#define __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, aux) stub_load_b128(r, voff, soff)
#define __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, x, y, z) (c)
#define __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, x, y, z) (c)
