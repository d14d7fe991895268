// HIP kernels for the FP32-FFT form of the all-pairs normalized
// cross-correlation (gfx950).
//
// Reference path these kernels replace, as one fused pipeline:
//   cuFFT R2C x2          Correlation_in_CUDA/correlation_cuda.cu:615-636
//   EWM_Linear            Correlation_in_CUDA/correlation_cuda.cu:23-75
//   cuFFT C2R             Correlation_in_CUDA/correlation_cuda.cu:424-428,450
//   FE_Linear             Correlation_in_CUDA/correlation_cuda.cu:78-152
//   scan/normalise rule   Correlation_in_OMP/correlation_c.cpp:102-136
//
// Math.  The reference multiplies X_i by R_j = rfft(pad(flip(x_j))), which is
// exp(-2 pi i (L-1) k / P) * conj(X_j), inverse-transforms and scans
// corr_t[L + i], i in [-S, S), as lag i + 1.  corr_t[L + i] equals
// P * c[(i + 1) mod P] with c the period-P circular cross-correlation
// c[l] = sum_n x_i[n] x_j[n - l], so these kernels form X_i * conj(X_j)
// directly and read lag l at index l mod P; no reversed copy is needed.
//
// Spectra are pre-normalised in the forward kernel: Xhat = X / sqrt(E*C*P)
// with the energy E summed in FP64 on the device, so the inverse transform of
// sum_c Xhat_ic conj(Xhat_jc) is directly the channel-averaged normalized
// coefficient.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "xc_fft.hpp"
#include "xc_kernels.h"

#ifndef SXC_R
#error "compile once per R with -DSXC_R=8|16|24|32|40|48|64"
#endif

namespace sxc {

// ----------------------------------------------------------------------------
// small helpers
// ----------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

#if SXC_R == 8
// Histogram + threshold pass (Correlation_in_OMP/correlation_c.cpp:114-136):
// pos value v -> class v >= 1 ? n-1 : int(v / delta), neg value u -> class
// u <= -1 ? n-1 : int(-u / delta) (FP32 division, truncation), counted before
// the threshold; then pos kept if v > threshold, neg if u < -threshold, else
// (0, 0).  The class index is clamped to n-1 (the reference can index one
// past the end when v / delta rounds up to n).  Block-local histograms in LDS
// when 2 n ints fit 64 KiB, else direct global atomics.
__global__ __launch_bounds__(256) void k_hist_threshold(HistArgs a) {
  extern __shared__ int hs[];
  const int nc = a.n_classes;
  const bool lds = 2 * nc <= 16384;
  if (lds) {
    for (int k = threadIdx.x; k < 2 * nc; k += 256) hs[k] = 0;
    __syncthreads();
  }
  for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < a.n; e += (long long)gridDim.x * 256) {
    const float v = a.vpos[e], u = a.vneg[e];
    const int bp = v >= 1.f ? nc - 1 : max(0, min((int)__fdiv_rn(v, a.delta), nc - 1));
    const int bn = u <= -1.f ? nc - 1 : max(0, min((int)__fdiv_rn(-u, a.delta), nc - 1));
    if (lds) {
      atomicAdd(&hs[bp], 1);
      atomicAdd(&hs[nc + bn], 1);
    } else {
      atomicAdd(&a.hist_pos[bp], 1);
      atomicAdd(&a.hist_neg[bn], 1);
    }
    if (!(v > a.threshold)) {
      a.vpos[e] = 0.f;
      a.lpos[e] = 0;
    }
    if (!(u < -a.threshold)) {
      a.vneg[e] = 0.f;
      a.lneg[e] = 0;
    }
  }
  if (lds) {
    __syncthreads();
    for (int k = threadIdx.x; k < nc; k += 256) {
      if (hs[k]) atomicAdd(&a.hist_pos[k], hs[k]);
      if (hs[nc + k]) atomicAdd(&a.hist_neg[k], hs[nc + k]);
    }
  }
}

hipError_t launch_hist_threshold(const HistArgs& a, hipStream_t st) {
  if (a.n <= 0 || a.n_classes < 1) return hipSuccess;
  const long long g = (a.n + 255) / 256;
  const size_t lds = 2 * a.n_classes <= 16384 ? (size_t)2 * a.n_classes * sizeof(int) : 0;
  hipLaunchKernelGGL(k_hist_threshold, dim3((unsigned)(g < 2048 ? g : 2048)), dim3(256), lds, st, a);
  return hipGetLastError();
}

__global__ void k_fill_u32(unsigned* p, unsigned v, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
#endif

// ----------------------------------------------------------------------------
// forward: one wave per (event, channel) row
// ----------------------------------------------------------------------------
// Reads row r (samples n < in_len, zero beyond), optionally demeans the first
// L samples in FP64, sums the energy of the first L samples in FP64, and
// writes Xhat[k] = rfft(x)[k] * scale for k = 0..M, scale = 1/sqrt(E*C*P)
// (0 for a zero-energy row).
// A workgroup of fwd_waves<R>() waves stages the twiddle tables once and
// walks rows (blockIdx.x + g gridDim.x) W + wave; each wave keeps one buffer
// of max(kWaveLds, M) entries for its transposes and, after its FFT, for the
// natural-order Z (in-order LDS accesses within a wave let the two share it).
template <int R>
constexpr int fwd_wave_buf() {
  return 64 * R > kWaveLds ? 64 * R : kWaveLds;
}
template <int R>
constexpr int fwd_waves() {
  constexpr int w = (160 * 1024 - TwLayout<R>::kFft * 8) / (fwd_wave_buf<R>() * 8);
  return w > 8 ? 8 : (w < 1 ? 1 : w);
}

// The row's samples in registers -> its scaled half spectrum in memory.
template <int R>
__device__ __forceinline__ void forward_finish(const ForwardArgs& a, cf (&d)[R], float scale, float2* out,
                                               const float2* twl, float2* wl, float2* zl, int lane) {
  constexpr int M = 64 * R;
  constexpr int P = 2 * M;
  // the first post-twiddles are requested before the transform where registers
  // allow (N = 16, P = 4096 spilled: 49 -> 56 us), those of the next four steps
  // before the stores of this four (which the compiler cannot move loads across)
  constexpr int kStep = 4;
  static_assert((R / 2) % kStep == 0, "whole steps");
  float2 tw[kStep];
  auto first_tw = [&] {
#pragma unroll
    for (int u = 0; u < kStep; ++u) tw[u] = a.post_tw[lane + 64 * u];
  };
  if constexpr (R <= 24) first_tw();

  wave_fft<R, -1>(d, twl, wl, lane);
#pragma unroll
  for (int r = 0; r < R; ++r) zl[wave_out_index<R>(lane, r)] = c2f(d[r]);
  wave_lds_fence();

  auto emit = [&](int k, cf X) {
    if (a.reversed) {
      // X * exp(+2 pi i q / P), q = k * rev_shift mod P, from the table of
      // exp(-2 pi i k / P), k <= M: conj(post[q]) for q <= M, post[P - q] above
      const int q = (int)(((long long)k * a.rev_shift) % P);
      const cf pq = f2c(a.post_tw[q <= M ? q : P - q]);
      const cf ph = cmk(pq.x, q <= M ? -pq.y : pq.y);
      X = cmul(X, ph);
      X.y = -X.y;  // stored conjugated: the pair kernel conjugates its column operand
    }
    if (k == 0 || k == M) X.y = 0.f;
    out[k] = make_float2(X.x * scale, X.y * scale);
  };
  // X[k] = E + O e^{-2 pi i k/P} and, E and O of the mirrored bin being
  // conjugates, X[M-k] = conj(E - O e^{-2 pi i k/P}), with
  // E = (Z[k] + conj Z[M-k])/2, O = -i/2 (Z[k] - conj Z[M-k]), Z[M] = Z[0]
  auto convert = [&](int k, float2 t) {
    const cf z = f2c(zl[k]);
    cf zm = f2c(zl[k > 0 ? M - k : 0]);
    zm.y = -zm.y;
    const cf e = cmk(0.5f * (z.x + zm.x), 0.5f * (z.y + zm.y));
    const cf dd = csub(z, zm);
    const cf od = cmul(cmk(0.5f * dd.y, -0.5f * dd.x), f2c(t));
    emit(k, cadd(e, od));
    if (2 * k != M) emit(M - k, cmk(e.x - od.x, od.y - e.y));
  };
  if constexpr (R > 24) first_tw();
#pragma unroll 1
  for (int k0 = lane; k0 < M / 2; k0 += 64 * kStep) {
    float2 t[kStep];
#pragma unroll
    for (int u = 0; u < kStep; ++u) t[u] = tw[u];
#pragma unroll
    for (int u = 0; u < kStep; ++u) tw[u] = a.post_tw[min(k0 + 64 * (kStep + u), M)];
#pragma unroll
    for (int u = 0; u < kStep; ++u) convert(k0 + 64 * u, t[u]);
  }
  if (lane == 0) convert(M / 2, a.post_tw[M / 2]);
}

template <int R>
__device__ __forceinline__ void forward_row(const ForwardArgs& a, int row, const float2* twl, float2* wl,
                                            float2* zl, int lane) {
  constexpr int M = 64 * R;
  constexpr int P = 2 * M;
  wave_lds_fence();  // the previous row's reads of this wave's buffer come first
  const float* x = a.in + (long long)row * a.in_stride;
  int in_len = a.in_len, L = a.L;
  if (a.row_len) {  // uneven lengths: this row's event sets both counts
    const int n = a.row_len[row / a.n_channels];
    in_len = n < (int)a.in_stride ? n : (int)a.in_stride;
    L = in_len;
  }
  if (in_len < 1) {  // empty row: zero spectrum
    for (int k = lane; k <= M; k += 64) a.spec[(long long)row * a.spec_stride + k] = make_float2(0.f, 0.f);
    if (lane == 0 && !a.reversed) a.norms[row] = 0.0;
    return;
  }
  // d[m] = x[2(t+64m)] + i x[2(t+64m)+1]; clamped loads + selects, no branches
  cf d[R];
  const int last = in_len > 0 ? in_len - 1 : 0;
#pragma unroll
  for (int m = 0; m < R; ++m) {
    const int n = 2 * (lane + 64 * m);
    const float e0 = x[min(n, last)], e1 = x[min(n + 1, last)];
    d[m].x = n < in_len ? e0 : 0.f;
    d[m].y = n + 1 < in_len ? e1 : 0.f;
  }
  // mean (from memory) and energy (from the registers) of the first L
  // samples in FP64 (a reversed row takes the energy of its forward row)
  double mean = 0.0, E = 0.0;
  if (a.reversed) {
    const double nr = a.norms_in[row];
    E = nr * nr;
  } else {
    if (a.demean) {
      double s1 = 0.0;
      for (int n = lane; n < L; n += 64) s1 += (double)(n < in_len ? x[n] : 0.f);
      mean = wave_sum_f64(s1) / (double)L;
#pragma unroll
      for (int m = 0; m < R; ++m) {
        const int n = 2 * (lane + 64 * m);
        const float u0 = (float)((double)d[m].x - mean), u1 = (float)((double)d[m].y - mean);
        d[m].x = n < L ? u0 : d[m].x;
        d[m].y = n + 1 < L ? u1 : d[m].y;
      }
    }
    double s2 = 0.0;
#pragma unroll
    for (int m = 0; m < R; ++m) {
      const int n = 2 * (lane + 64 * m);
      const double u0 = n < L ? (double)d[m].x : 0.0, u1 = n + 1 < L ? (double)d[m].y : 0.0;
      s2 += u0 * u0 + u1 * u1;
    }
    E = wave_sum_f64(s2);
  }
  if (a.out_traces) {
    float* o = a.out_traces + (long long)row * a.out_stride;
#pragma unroll
    for (int m = 0; m < R; ++m) {
      const int n = 2 * (lane + 64 * m);
      *reinterpret_cast<float2*>(o + n) = make_float2(d[m].x, d[m].y);
    }
  }
  if (lane == 0 && !a.reversed) a.norms[row] = sqrt(E);
  const float scale = E > 0.0 ? (float)(1.0 / sqrt(E * (double)a.n_channels * (double)P)) : 0.f;

  forward_finish<R>(a, d, scale, a.spec + (long long)row * a.spec_stride, twl, wl, zl, lane);
}

// Item v of a segment-mode launch: row v / (2 n_seg), segment v / 2 % n_seg, row
// side (v even) or column side; with one side, row v / n_seg, segment v % n_seg.  Every wave sums its row's mean and energy
// itself: a row is at most 8192 samples, which its 2 n_seg waves read from L2,
// and a launch of its own would cost a small job more.
template <int R>
__device__ __forceinline__ void forward_segment(const ForwardArgs& a, int v, const float2* twl, float2* wl,
                                                float2* zl, int lane) {
  constexpr int P = 128 * R;
  wave_lds_fence();  // the previous item's reads of this wave's buffer come first
  const bool col = a.seg_sides ? a.seg_sides == 2 : (v & 1) != 0;
  const int u = a.seg_sides ? v : v >> 1, row = u / a.n_seg, seg = u - row * a.n_seg, s0 = seg * a.seg_len;
  const float* x = a.in + (long long)row * a.in_stride;
  const int last = a.in_len - 1;
  constexpr int U = 8;  // 64-sample steps whose loads are in flight together
  auto sum = [&](auto&& term) {
    double s = 0.0;
    for (int n0 = lane; n0 < a.L; n0 += 64 * U) {
      float u[U];
#pragma unroll
      for (int k = 0; k < U; ++k) u[k] = x[min(n0 + 64 * k, last)];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const int n = n0 + 64 * k;
        s += n < a.L ? term(n < a.in_len ? u[k] : 0.f) : 0.0;
      }
    }
    return wave_sum_f64(s);
  };
  const double mean = a.demean ? sum([](float u) { return (double)u; }) / (double)a.L : 0.0;
  const double E = sum([&](float u) {
    const double w = (double)(a.demean ? (float)((double)u - mean) : u);
    return w * w;
  });
  // element m: sample n = s0 + m, or s0 + m - P before the segment (column side)
  const int end = s0 + a.seg_len + (col ? a.seg_ahead : 0), begin = s0 - (col ? a.seg_back : 0);
  auto sample = [&](int m) {
    int n = s0 + m;
    n -= n >= end ? P : 0;
    const float u = x[min(max(n, 0), last)], w = n < a.in_len ? u : 0.f;
    const float z = a.demean && n < a.L ? (float)((double)w - mean) : w;
    return n >= max(begin, 0) && n < end ? z : 0.f;
  };
  cf d[R];
#pragma unroll
  for (int m = 0; m < R; ++m) {
    const int n = 2 * (lane + 64 * m);
    d[m].x = sample(n);
    d[m].y = sample(n + 1);
  }
  if (!col) {
    if (a.out_traces) {
      float* o = a.out_traces + (long long)row * a.out_stride + s0;
      const int n_out = min(a.seg_len, (int)a.out_stride - s0);
#pragma unroll
      for (int m = 0; m < R; ++m) {
        const int n = 2 * (lane + 64 * m);
        if (n < n_out) o[n] = d[m].x;
        if (n + 1 < n_out) o[n + 1] = d[m].y;
      }
    }
    if (lane == 0 && seg == 0) a.norms[row] = sqrt(E);
  }
  const float scale = E > 0.0 ? (float)(1.0 / sqrt(E * (double)a.n_channels * (double)P)) : 0.f;
  float2* out = (col ? a.seg_cols : a.spec) + ((long long)row * a.n_seg + seg) * a.spec_stride;
  forward_finish<R>(a, d, scale, out, twl, wl, zl, lane);
}

template <int R, bool SEG>
__global__ __launch_bounds__(64 * fwd_waves<R>()) void k_forward(ForwardArgs a) {
  constexpr int M = 64 * R;
  constexpr int P = 2 * M;
  constexpr int W = fwd_waves<R>();
  extern __shared__ __align__(16) float2 smem[];
  float2* twl = smem;  // twiddle tables
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float2* wl = smem + TwLayout<R>::kFft + wv * fwd_wave_buf<R>();  // this wave's transposes, then Z
  float2* zl = wl;
  if (a.zero && blockIdx.x == 0 && threadIdx.x == 0) *a.zero = 0u;
  stage_twiddles<TwLayout<R>::kFft, 64 * W>(twl, a.tw, threadIdx.x);
  __syncthreads();
  const int n = SEG ? a.n_rows * a.n_seg * (a.seg_sides ? 1 : 2) : a.n_rows;
  for (int row = blockIdx.x * W + wv; row < n; row += gridDim.x * W) {
    if constexpr (SEG) forward_segment<R>(a, row, twl, wl, zl, lane);
    else forward_row<R>(a, row, twl, wl, zl, lane);
  }
}

// ----------------------------------------------------------------------------
// per-pair inverse transform (shared by the pair kernel and the resolver)
// ----------------------------------------------------------------------------
// Builds Y = sum_c Xhat_ic conj(Xhat_jc) for this lane's bins t + 64m (row i
// from LDS, row j from global), converts the half spectrum to the packed
// half-length sequence Z[k] = (Y[k] + conj Y[M-k]) + i e^{2 pi i k/P}
// (Y[k] - conj Y[M-k]) and runs the inverse wave FFT.  On return lane l,
// register r holds c[2q] (x) and c[2q+1] (y), q = wave_out_index(l, r).
// Largest divisor of R that is at most cap (R = 48, cap 32: 24), so the load
// groups tile the R bins of a lane exactly.
constexpr int load_group(int R, int cap) {
  int g = R < cap ? R : cap;
  while (R % g) --g;
  return g;
}

// Spectrum rows read from global memory go through a buffer resource: the
// row base is a scalar, one per-lane offset register (8 lane) serves a whole
// 4 KiB stretch through the instruction's immediate offset, and a channel's
// start is the scalar offset, so the loads need no per-pair vector address
// arithmetic.  `base` must be wave-uniform; a row of nch channels spans
// ((nch - 1) stride + M + 1) float2, at most 8 channels of 4097 bins (the
// plans' limits), far below the 2^31 bytes a resource can describe.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t spec_rsrc(const float2* base, long long stride, int nch, int M) {
  const long long bytes = 8 * ((long long)(nch - 1) * stride + M + 1);
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float2 spec_load(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
  return make_float2(__uint_as_float(v.x), __uint_as_float(v.y));
}

// Channels [0, n_lds) of row i are read from xi_lds (stride M + 1), the others from
// xi in memory (stride xj_stride).
enum class RowFrom { kLds, kMemory, kBoth };
// kChannels: channels loaded together.
template <int R, RowFrom kRow, int kChannels, int kLoadGroup = 32>
__device__ __forceinline__ void pair_inverse(cf (&y)[R], const float2* __restrict__ xi_lds, int n_lds,
                                             const float2* __restrict__ xi, const float2* __restrict__ xj,
                                             long long xj_stride, int nch, const float2* tw,
                                             float2* wl, int lane) {
  constexpr int M = 64 * R;
  float yN = 0.f;
  const __amdgpu_buffer_rsrc_t rj = spec_rsrc(xj, xj_stride, nch, M);
  const __amdgpu_buffer_rsrc_t ri = spec_rsrc(xi, xj_stride, nch, M);
  // Channels [c, c + kN): channel 0 initialises the accumulators, the others add to
  // them.
  auto channels = [&](int c, auto count_c, auto first_c, auto memory_c) {
    constexpr int kN = decltype(count_c)::value;
    constexpr bool kFirst = decltype(first_c)::value;
    constexpr bool XI_GLOBAL = decltype(memory_c)::value;
    // per-lane byte offset, redefined per channel (in the loads' block, with
    // a known range) so the bin offsets stay instruction immediates instead
    // of one hoisted offset register per load
    int lv = lane;
    asm volatile("" : "+v"(lv));
    const int vb = 8 * (lv & 63);
    float2 aN[kN], bN[kN];
    // All of a group's global loads are issued before the compiler fence so
    // they are in flight together (one L2 round trip per group, not per row).
    // Two channels at a time at P = 1024, where registers allow, and the Nyquist
    // bins with them: N = 1500, P = 1024, C = 6 .. 8 5%
    // faster, N = 16, C = 1, L = 4096, +-50 (5 segments) 37.4 -> 35.5 us.  At P = 2048
    // and 3072 the Nyquist bin's registers alone cost 1-3%.
    constexpr bool kEarly = kChannels > 1;
    constexpr int kGroup = load_group(R, kLoadGroup);
    static_assert(R % kGroup == 0, "load groups must tile the lane's bins");
#pragma unroll
    for (int m0 = 0; m0 < R; m0 += kGroup) {
      float2 Bv[kN][kGroup];
      float2 Av[kN][XI_GLOBAL ? kGroup : 1];
#pragma unroll
      for (int n = 0; n < kN; ++n) {
        const int soff = (int)(8 * (c + n) * xj_stride);
#pragma unroll
        for (int u = 0; u < kGroup; ++u) Bv[n][u] = spec_load(rj, vb + 512 * (m0 + u), soff);
        if constexpr (XI_GLOBAL) {
#pragma unroll
          for (int u = 0; u < kGroup; ++u) Av[n][u] = spec_load(ri, vb + 512 * (m0 + u), soff);
        }
        if (kEarly && m0 == 0) {
          bN[n] = spec_load(rj, 8 * M, soff);
          if constexpr (XI_GLOBAL) aN[n] = spec_load(ri, 8 * M, soff);
        }
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int n = 0; n < kN; ++n) {
        const float2* ai = xi_lds + (c + n) * (M + 1);
#pragma unroll
        for (int u = 0; u < kGroup; ++u) {
          const int m = m0 + u;
          cf A = f2c(XI_GLOBAL ? Av[n][XI_GLOBAL ? u : 0] : ai[lane + 64 * m]);
          cf B = f2c(Bv[n][u]);
          if (kFirst && n == 0) {
            y[m].x = __builtin_fmaf(A.x, B.x, A.y * B.y);
            y[m].y = __builtin_fmaf(A.y, B.x, -A.x * B.y);
          } else {
            y[m].x = __builtin_fmaf(A.x, B.x, __builtin_fmaf(A.y, B.y, y[m].x));
            y[m].y = __builtin_fmaf(A.y, B.x, __builtin_fmaf(-A.x, B.y, y[m].y));
          }
        }
      }
    }
#pragma unroll
    for (int n = 0; n < kN; ++n) {
      if constexpr (!XI_GLOBAL) aN[n] = xi_lds[(c + n) * (M + 1) + M];
      else if (!kEarly) aN[n] = xi[(c + n) * xj_stride + M];
      if (!kEarly) bN[n] = xj[(c + n) * xj_stride + M];
      yN = kFirst && n == 0 ? __builtin_fmaf(aN[n].x, bN[n].x, aN[n].y * bN[n].y)
                            : __builtin_fmaf(aN[n].x, bN[n].x, __builtin_fmaf(aN[n].y, bN[n].y, yN));
    }
  };
  constexpr std::integral_constant<int, 1> one{};
  // channels [0, n), kChannels at a time
  auto run = [&](int n, auto memory_c) {
    int c = 1;
    if constexpr (kChannels > 1) {
      constexpr std::integral_constant<int, kChannels> some{};
      if (n >= kChannels) {
        channels(0, some, std::true_type{}, memory_c);
        for (c = kChannels; c + kChannels <= n; c += kChannels) channels(c, some, std::false_type{}, memory_c);
      } else {
        channels(0, one, std::true_type{}, memory_c);
      }
    } else {
      channels(0, one, std::true_type{}, memory_c);
    }
    for (; c < n; ++c) channels(c, one, std::false_type{}, memory_c);
  };
  // Wave priority by phase (s_setprio; the arbiter issues from the waves of
  // a SIMD in priority order): 2 while the column spectra are loaded and
  // multiplied, 1 for the packing, 0 for the transform and the scan.  A wave
  // starting a pair then gets its loads out and its products done first,
  // which keeps the SIMD's waves staggered over the phases instead of all
  // waiting on memory or LDS at once (pair kernel 6% faster at P = 4096).
  __builtin_amdgcn_s_setprio(2);
  if constexpr (kRow == RowFrom::kMemory) run(nch, std::true_type{});
  else run(kRow == RowFrom::kLds ? nch : n_lds, std::false_type{});
  if constexpr (kRow == RowFrom::kBoth)
    for (int c = n_lds; c < nch; ++c) channels(c, one, std::false_type{}, std::true_type{});
  __builtin_amdgcn_s_setprio(1);
  // c2r ignores the imaginary parts of the DC and Nyquist bins
  if (lane == 0) y[0].y = 0.f;

  const cf u = f2c(tw[TwLayoutCT<R>::kPreL + lane]);
  // exp(+2 pi i (lane + 64 m) / P)
  auto pre_tw = [&](auto mc) -> cf { return twmul<decltype(mc)::value, 2 * R, 1>(u); };
  // With E = Y[k] + conj(Y[M-k]), D = Y[k] - conj(Y[M-k]), T = e^{2 pi i k/P}:
  // Z[k] = E + i T D and, as E and D of the mirrored bin are conj(E) and
  // -conj(D) and its factor -conj(T), Z[M-k] = conj(E - i T D).  One lane so
  // computes both bins from one product: 12 operations and one packing factor
  // for two bins instead of 16 and two (each bin by its own lane): the kernel is
  // bound by vector issue, and N = 4096, C = 3, P = 4096 went 33.00 -> 32.36 ms,
  // N = 1501, P = 8192 7.58 -> 7.40 ms, N = 1111, C = 2, P = 3072 2.00 -> 1.94 ms.
  // Lane t owns bin t + 64 m in register m; the lanes of the low registers
  // m < R/2 compute.  In chunks of Q low registers m = cQ + q, the registers
  // R - 1 - m that hold their mirrors are written to this wave's LDS buffer as
  // a linear range of bins (row r: register a0 + r; the bin above the range,
  // lane 0 of the next register or the Nyquist bin, as row Q), each lane reads
  // its mirror M - k at one address formula, writes Z[M-k] back to the same
  // place, and the owners read it.  Lane 0's lowest bin of a chunk, 64 a0,
  // mirrors into the next chunk: it stays unchanged and goes along as that
  // chunk's row Q; after the last chunk it is bin M/2, its own mirror.
  constexpr int HR = R / 2;
  constexpr int Q = load_group(HR, 8);
  static_assert(HR % Q == 0 && Q + 1 <= kWaveLds / 64, "mirror chunks");
  sfor<0, HR / Q>([&](auto cc) {
    constexpr int c = decltype(cc)::value;
    constexpr int a0 = R - Q - Q * c;  // first register of the chunk's mirrors
    cf am[Q];
    wave_lds_fence();  // earlier reads of the buffer come first
#pragma unroll
    for (int r = 0; r < Q; ++r) wl[64 * r + lane] = c2f(y[a0 + r]);
    wl[64 * Q + lane] = c == 0 ? make_float2(yN, 0.f) : c2f(y[c == 0 ? 0 : a0 + Q]);
    wave_lds_fence();
#pragma unroll
    for (int q = 0; q < Q; ++q) am[q] = f2c(wl[64 * (Q - q) - lane]);
    sfor<0, Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      constexpr int m = Q * c + q;
      const cf t = pre_tw(std::integral_constant<int, m>{});
      const cf a = y[m], b = am[q];
      const float ex = a.x + b.x, ey = a.y - b.y, dx = a.x - b.x, dy = a.y + b.y;
      const float re = __builtin_fmaf(t.x, dy, t.y * dx);   // -Re(i T D)
      const float im = __builtin_fmaf(t.x, dx, -t.y * dy);  // Im(i T D)
      y[m] = cmk(ex - re, ey + im);
      am[q] = cmk(ex + re, im - ey);
    });
    wave_lds_fence();
#pragma unroll
    for (int q = 0; q < Q; ++q) wl[64 * (Q - q) - lane] = c2f(am[q]);
    wave_lds_fence();
#pragma unroll
    for (int r = 0; r < Q; ++r) y[a0 + r] = f2c(wl[64 * r + lane]);
    if constexpr (c > 0) y[a0 + Q] = f2c(wl[64 * Q + lane]);  // lane 0's bin from this chunk's row Q
  });
  // bin M/2 (lane 0 of register R/2): E + i T D with Y its own mirror, T = i
  if (lane == 0) y[HR] = cmk(2.f * y[HR].x, -2.f * y[HR].y);
  wave_lds_fence();  // the FFT's transposes reuse the buffer
  __builtin_amdgcn_s_setprio(0);
  wave_fft<R, 1, true>(y, tw, wl, lane);
}

// lag of (lane, slot) where slot = 2*reg + {0: x, 1: y}
template <int R>
__host__ __device__ __forceinline__ int slot_lag(int lane, int slot) {
  constexpr int M = 64 * R;
  const int reg = slot >> 1;
  const int q = ((lane >> 3) + 8 * (reg >> 3)) + R * ((lane & 7) + 8 * (reg & 7));
  const int n = 2 * q + (slot & 1);
  return n <= M ? n : n - 2 * M;
}

// Registers a window can touch.  Register 8s + k of the transform's output
// holds, over the lanes and s, the run of 16 R lags from 16 R k on (k < 4) or
// 16 R (k - 8) (k >= 4).  A kernel built for G = 1 or 2 serves windows inside
// the 2G runs around lag 0 (k < G and k >= 8 - G): the other registers are
// neither scanned nor, as the compiler drops them, computed in the last
// radix-8 pass.  G = 4 serves every window, G = 0 scans every lag unmasked.
template <int R, int G>
constexpr int win_regs() { return G == 0 ? R : R / 8 * 2 * G; }
template <int R, int G>
constexpr int win_reg(int i) {  // i-th such register
  if (G == 0) return i;
  const int s = i / (2 * G), q = i % (2 * G);
  return 8 * s + (q < G ? q : 8 - 2 * G + q);
}

// In-window bit of every value (2 i + {0: x, 1: y}) of a lane's win_regs, built
// once per workgroup and applied with two operations per value (bit field
// extract, and).
template <int R, int G>
struct WinBits {
  static constexpr int kWords = (2 * win_regs<R, G>() + 31) / 32;
  unsigned w[kWords];
};
template <int R, int G>
__device__ __forceinline__ void win_bits(WinBits<R, G>& wb, int lane, int lo, int hi) {
  constexpr int M = 64 * R;
  const unsigned span = (unsigned)(hi - lo);
  const int base = 2 * ((lane >> 3) + R * (lane & 7)) - lo;  // lag - lo of (lane, register 0)
#pragma unroll
  for (int w = 0; w < WinBits<R, G>::kWords; ++w) wb.w[w] = 0u;
  sfor<0, 2 * win_regs<R, G>()>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    constexpr int reg = win_reg<R, G>(i >> 1), s = reg >> 3, k = reg & 7;
    constexpr int off = 2 * (8 * s + 8 * R * k) + (i & 1) - (k >= 4 ? 2 * M : 0);
    bool in = (unsigned)(base + off) <= span;
    if constexpr (k == 4 && s == 0 && (i & 1) == 0) in = in || (lane == 0 && hi >= M);  // lag M, not -M
    wb.w[i >> 5] |= in ? 1u << (i & 31) : 0u;
  });
}
// Zero every value whose lag is outside the window.
template <int R, int G>
__device__ __forceinline__ void apply_window(cf (&y)[R], const WinBits<R, G>& wb) {
  sfor<0, win_regs<R, G>()>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    constexpr int r = win_reg<R, G>(i);
    auto keep = [&](float v, int bit) {
      const int m = (int)(wb.w[bit >> 5] << (31 - (bit & 31))) >> 31;
      return __int_as_float(__float_as_int(v) & m);
    };
    y[r].x = keep(y[r].x, 2 * i);
    y[r].y = keep(y[r].y, 2 * i + 1);
  });
}

struct Best {
  float v;
  int lag;
};

// Wave-wide max / min with DPP row operations, read from lane 63 (so the
// result is wave-uniform).  Both run on the float bit patterns as integers,
// which DPP folds into the max itself (a float max would first quiet its DPP
// operand: three more instructions per step): the running max is >= +0 (it
// starts at 0), and non-negative floats order as signed integers (-0 maps to
// the smallest, equal in value to +0); the running min is <= 0, and
// non-positive floats order (reversed) as unsigned integers, with +0 below
// -0 below every negative.  Lanes whose DPP source is out of range read 0,
// which neither changes.
__device__ __forceinline__ int dpp_i(int v, int ctrl_sel) {
  switch (ctrl_sel) {
    case 0: return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);   // quad_perm [1,0,3,2]
    case 1: return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
    case 2: return __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true);  // row_half_mirror
    case 3: return __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, true);  // row_mirror
    case 4: return __builtin_amdgcn_update_dpp(0, v, 0x142, 0xF, 0xF, true);  // row_bcast:15
    default: return __builtin_amdgcn_update_dpp(0, v, 0x143, 0xF, 0xF, true); // row_bcast:31
  }
}
__device__ __forceinline__ void wave_maxmin(float& mx, float& mn) {
  int imx = __float_as_int(mx);
  unsigned umn = __float_as_uint(mn);
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    imx = max(imx, dpp_i(imx, k));
    umn = max(umn, (unsigned)dpp_i((int)umn, k));
  }
  mx = __int_as_float(__builtin_amdgcn_readlane(imx, 63));
  mn = __int_as_float(__builtin_amdgcn_readlane((int)umn, 63));
}

// Reference scan rule over the wave's values: strict > (<) starting from
// (0, lag 0), first occurrence.  Pass 1 keeps the max (min) of each group of
// four registers (8 values; two registers for G = 1) and reduces them to the exact extrema (DPP wave
// reduction); pass 2 ballots each group maximum (minimum) against extremum
// -/+ tol, and only for the rare groups where that ballot is non-zero
// ballots the group's values separately: the ballot counts are summed
// on the scalar unit, and the last slot whose ballot is non-zero (with its
// lane mask) locates the extremum.  More than one value within tol flags a
// near tie, which the FP64 resolver settles.
template <int R, int G>
__device__ __forceinline__ void scan_wave(const cf (&y)[R], int lane, float tol, float thr,
                                          Best& pos, Best& neg, bool& tie_p, bool& tie_n) {
  constexpr int N = win_regs<R, G>(), S = G == 1 ? 2 : 4;  // registers scanned, and per group
  static_assert(N % S == 0, "whole groups of registers");
  constexpr int NG = N / S;
  float gp[NG], gn[NG];
  float mx = 0.f, mn = 0.f;
  sfor<0, NG>([&](auto gc) {
    constexpr int g = decltype(gc)::value;
    // chained so that each three-operand max (min) takes two new values
    float hi = y[win_reg<R, G>(S * g)].x, lo = hi;
    sfor<1, 2 * S>([&](auto qc) {
      constexpr int q = decltype(qc)::value, r = win_reg<R, G>(S * g + (q >> 1));
      const float v = (q & 1) ? y[r].y : y[r].x;
      hi = fmaxf(hi, v);
      lo = fminf(lo, v);
    });
    gp[g] = hi;
    gn[g] = lo;
    mx = fmaxf(mx, hi);
    mn = fminf(mn, lo);
  });
  wave_maxmin(mx, mn);
  const bool want_p = mx > thr && mx > 0.f;
  const bool want_n = mn < -thr && mn < 0.f;
  const float cp = mx - tol, cn = mn + tol;
  int cnt_p = 0, cnt_n = 0, slot_p = -1, slot_n = -1;
  unsigned long long msk_p = 0, msk_n = 0;
  if (want_p || want_n) {
    sfor<0, NG>([&](auto gc) {
      constexpr int g = decltype(gc)::value;
      if (__ballot(gp[g] >= cp)) {
        sfor<0, 2 * S>([&](auto qc) {
          constexpr int q = decltype(qc)::value, r = win_reg<R, G>(S * g + (q >> 1));
          const float v = (q & 1) ? y[r].y : y[r].x;
          const unsigned long long b = __ballot(v >= cp);
          cnt_p += __popcll(b);
          if (b) { slot_p = 2 * r + (q & 1); msk_p = b; }
        });
      }
      if (__ballot(gn[g] <= cn)) {
        sfor<0, 2 * S>([&](auto qc) {
          constexpr int q = decltype(qc)::value, r = win_reg<R, G>(S * g + (q >> 1));
          const float v = (q & 1) ? y[r].y : y[r].x;
          const unsigned long long b = __ballot(v <= cn);
          cnt_n += __popcll(b);
          if (b) { slot_n = 2 * r + (q & 1); msk_n = b; }
        });
      }
    });
  }
  pos.v = want_p ? mx : (mx > 0.f ? mx : 0.f);
  pos.lag = (want_p && slot_p >= 0) ? slot_lag<R>(__ffsll((long long)msk_p) - 1, slot_p) : 0;
  neg.v = want_n ? mn : (mn < 0.f ? mn : 0.f);
  neg.lag = (want_n && slot_n >= 0) ? slot_lag<R>(__ffsll((long long)msk_n) - 1, slot_n) : 0;
  // also near 0, the scan's starting state; with kScanNoise, no value outside the
  // window of an unmasked scan decides whether a pair is recorded
  tie_p = want_p && (cnt_p > 1 || cp <= kScanNoise);
  tie_n = want_n && (cnt_n > 1 || cn >= -kScanNoise);
}

__device__ __forceinline__ long long packed_index(int i, int j, int n) {
  return (long long)i * n - (long long)i * (i - 1) / 2 + (j - i);
}

// ----------------------------------------------------------------------------
// pair kernel: one workgroup (kWaves waves) per work item (row i, column chunk)
// ----------------------------------------------------------------------------
// The row spectra of a work item are staged in LDS for the workgroup's waves: all
// of them (kRow = kLds) or, with many channels at a long period, the first
// a.n_lds, the rest being read from memory by every wave (kBoth).
// Compact twiddle tables (9 KB instead of 66 KB at P = 8192, one extra complex
// multiply per twiddle; fewer LDS reads per pair).
// G: the registers scanned (win_regs).  kPerSimd: waves per SIMD the register
// budget leaves room for.
template <int R, int G, int kWaves, int kPerSimd, RowFrom kRow>
__global__ __launch_bounds__(kWaves * 64, kPerSimd) void k_pairs(PairArgs a) {
  constexpr int M = 64 * R;
  constexpr int kTab = TwLayoutCT<R>::kInv;
  extern __shared__ __align__(16) float2 smem[];
  const int lane = threadIdx.x & 63;
  // wave index as a scalar: column indices and spectrum addresses then stay
  // in scalar registers (loads use a scalar base and a per-lane offset)
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_lds = kRow == RowFrom::kLds ? a.n_channels : a.n_lds;
  float2* twl = smem;
  float2* xi_lds = smem + kTab;
  float2* wl = xi_lds + n_lds * (M + 1) + wv * kWaveLds;

  stage_twiddles<kTab, 64 * kWaves>(twl, a.tw, threadIdx.x);
  WinBits<R, G> wb;
  if constexpr (G > 0) win_bits<R, G>(wb, lane, a.lag_lo, a.lag_hi);

  // XCD-aware walk: workgroups are dispatched round-robin over the 8 XCDs,
  // so XCD x = blockIdx % 8 takes its own contiguous eighth of the
  // chunk-major work list and keeps one column chunk hot in its L2.
  const int n_xcd = (gridDim.x % 8 == 0) ? 8 : 1;  // pair_grid: a multiple of 8
  const int xcd = blockIdx.x % n_xcd, local = blockIdx.x / n_xcd, n_local = gridDim.x / n_xcd;
  const int seg = (a.n_work + n_xcd - 1) / n_xcd;
  const int seg_end = min(a.n_work, (xcd + 1) * seg);
  auto fetch = [&](int e) -> int2 {
    return a.work ? a.work[e] : make_int2(e % a.n_rows, e / a.n_rows * a.chunk);
  };
  int item = xcd * seg + local;
  int2 wk = item < seg_end ? fetch(item) : make_int2(0, 0);
  for (; item < seg_end; item += n_local) {
    const int i = wk.x;
    const int jb = wk.y;
    if (item + n_local < seg_end) wk = fetch(item + n_local);  // early: its load is done by the next turn
    const int je = min((jb / a.chunk + 1) * a.chunk, a.n_events);  // end of jb's column chunk
    const bool dense = a.dense_cols > 0;
    const float2* src = a.spec + (long long)i * a.n_channels * a.spec_stride;
    {
      // a channel's loads, or four channels' at short periods, are all in flight
      // before their first store
      constexpr int T = 64 * kWaves, kPer = (M + T - 1) / T, kCh = kPer > 3 ? 1 : 4;
      auto stage = [&](int c, auto count_c) {
        constexpr int kN = decltype(count_c)::value;
        float2 v[kN][kPer];
#pragma unroll
        for (int n = 0; n < kN; ++n)
#pragma unroll
          for (int u = 0; u < kPer; ++u) v[n][u] = src[(c + n) * a.spec_stride + min((int)threadIdx.x + u * T, M)];
#pragma unroll
        for (int n = 0; n < kN; ++n)
#pragma unroll
          for (int u = 0; u < kPer; ++u)
            if (M % T == 0 || (int)threadIdx.x + u * T < M) xi_lds[(c + n) * (M + 1) + threadIdx.x + u * T] = v[n][u];
      };
      __syncthreads();
      int c = 0;
      for (; c + kCh <= n_lds; c += kCh) stage(c, std::integral_constant<int, kCh>{});
      if constexpr (kCh > 1) {
        if (c + 2 <= n_lds) {
          stage(c, std::integral_constant<int, 2>{});
          c += 2;
        }
        if (c < n_lds) stage(c, std::integral_constant<int, 1>{});
      }
      if ((int)threadIdx.x < n_lds) xi_lds[threadIdx.x * (M + 1) + M] = src[threadIdx.x * a.spec_stride + M];
      __syncthreads();
    }

    const float2* cols = a.col_spec ? a.col_spec : a.spec;
    for (int j = (dense ? jb : max(jb, i)) + wv; j < je; j += kWaves) {
      cf y[R];
      const float2* xj = cols + (long long)j * a.n_channels * a.spec_stride;
      // smaller load groups where registers are short: the budget of 4 waves
      // per SIMD (128 VGPRs), and at P >= 6144 channels from memory (twice
      // the loads in flight) and the budget of 3
      pair_inverse<R, kRow, R == 8 ? 2 : 1, (kPerSimd >= 4 || (R >= 48 && (kRow != RowFrom::kLds || kPerSimd == 3))) ? 16 : 32>(
          y, xi_lds, n_lds, src, xj, a.spec_stride, a.n_channels, twl, wl, lane);
      if constexpr (G > 0) apply_window<R, G>(y, wb);
      Best pos, neg;
      bool tp, tn;
      scan_wave<R, G>(y, lane, a.tie_tol, a.threshold, pos, neg, tp, tn);
      if (lane == 0) {
        const long long idx = dense ? (long long)i * a.dense_cols + j : packed_index(i, j, a.n_events);
        const bool kp = pos.v > a.threshold, kn = neg.v < -a.threshold;
        a.vpos[idx] = kp ? pos.v : 0.f;
        a.lpos[idx] = kp ? pos.lag : 0;
        if (!a.pos_only) {
          a.vneg[idx] = kn ? neg.v : 0.f;
          a.lneg[idx] = kn ? neg.lag : 0;
        }
        if ((tp || tn) && a.tie_cap > 0) {
          unsigned slot = atomicAdd(a.tie_count, 1u);
          if (slot < (unsigned)a.tie_cap) a.ties[slot] = make_int4(i, j, (tp ? 1 : 0) | (tn ? 2 : 0), 0);
        }
      }
    }
  }
}

// ----------------------------------------------------------------------------
// FP64 near-tie resolver: one wave per recorded pair
// ----------------------------------------------------------------------------
// Recomputes the pair's FP32 correlation, collects every in-window lag whose
// value is within tol of the winner, evaluates those lags as FP64 direct
// sums over the time-domain traces and keeps the largest (smallest) with
// ties to the smaller lag; starting state (0, lag 0) as in the reference scan.
//
// FP64 sums for NQ lags at once (callers repeat one to fill unused slots),
// as shifts in [0, P):
//   conv = false: sum_n ti[n] tj[(n - shift_q) mod P], the circular
//                 correlation at lag shift_q;
//   conv = true:  sum_m ti[m] tj[(shift_q - m) mod P], the circular
//                 convolution with a reversed row, which is the reference's
//                 own sum for reversed rows (Correlation_in_OMP/
//                 correlation_c.cpp:270, :63, :102-103): its lag-l value is
//                 corr_t[L - 1 + l], this sum at shift_q = L - 1 + l.
// Each ti sample is read once for all NQ, the loads of 8 steps (4 for
// four lags) are issued together (a record is a serial chain: one memory round
// trip per 512 or 256 samples instead of one per 128), and two sets of partial sums per lane keep the FP64
// FMA chains short.  The results are wave-uniform.
template <int NQ>
__device__ __forceinline__ void corrn_f64(const float* __restrict__ ti, int len_i, const float* __restrict__ tj,
                                          int len_j, int P, const int (&shift)[4], bool conv, int lane,
                                          double (&out)[4]) {
  constexpr int U = NQ > 2 ? 4 : 8;  // 64-sample steps whose loads are in flight together
  double sa[NQ], sb[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) sa[q] = sb[q] = 0.0;
  for (int n0 = lane; n0 < len_i; n0 += 64 * U) {
    float x[U], b[U][NQ];
    bool ok[U][NQ];
#pragma unroll
    for (int s = 0; s < U; ++s) {
      const int n = n0 + 64 * s;
      const bool in = n < len_i;
      x[s] = ti[in ? n : 0];
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        int u = conv ? shift[q] - n : n - shift[q];  // n, shift in [0, P): one wrap suffices
        u += u < 0 ? P : 0;
        ok[s][q] = in && u < len_j;
        b[s][q] = tj[ok[s][q] ? u : 0];  // always in bounds
      }
    }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int s = 0; s < U; ++s) {
      const double xs = (double)x[s];
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        double& acc = (s & 1) ? sb[q] : sa[q];
        acc += ok[s][q] ? xs * (double)b[s][q] : 0.0;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) out[q] = wave_sum_f64(sa[q] + sb[q]);
}

template <int R>
__global__ __launch_bounds__(64) void k_resolve(ResolveArgs a) {
  constexpr int M = 64 * R;
  extern __shared__ __align__(16) float2 smem[];
  const int lane = threadIdx.x;
  // records [begin, end): tie_begin, when set, holds the count before the
  // pair launches whose records this launch resolves (the launch groups of
  // a blocked host-buffer call)
  const unsigned end = min(*a.tie_count, (unsigned)a.tie_cap);
  const unsigned begin = a.tie_begin ? min(*a.tie_begin, end) : 0u;
  const unsigned total = end - begin;
  // XCD-aware walk: XCD x = blockIdx % 8 resolves its own contiguous eighth
  // of the record list (records arrive roughly grouped by tile or row), so
  // the traces a record re-reads are usually still in that XCD's L2
  const unsigned n_xcd = (gridDim.x % 8 == 0) ? 8 : 1;
  const unsigned xcd = blockIdx.x % n_xcd, local = blockIdx.x / n_xcd, n_local = gridDim.x / n_xcd;
  const unsigned seg = (total + n_xcd - 1) / n_xcd;
  const unsigned rec0 = xcd * seg + local, seg_end = min(total, (xcd + 1) * seg);
  if (rec0 >= seg_end) return;  // no record for this workgroup
  // compact tables (as the pair kernel): 11.8 KB of LDS at P = 4096
  float2* twl = smem;
  float2* wl = smem + TwLayoutCT<R>::kInv;
  int4 t = a.ties[begin + rec0];  // its load runs beside the tables'
  stage_twiddles<TwLayoutCT<R>::kInv, 64>(twl, a.tw, lane);
  for (unsigned rec = rec0; rec < seg_end; rec += n_local) {
    if (rec != rec0) t = a.ties[begin + rec];
    const int i = __builtin_amdgcn_readfirstlane(t.x), j = __builtin_amdgcn_readfirstlane(t.y);
    const int side = __builtin_amdgcn_readfirstlane(t.z);
    wave_lds_fence();
    cf y[R];
    const float2* cols = a.col_spec ? a.col_spec : a.spec;
    pair_inverse<R, RowFrom::kMemory, R == 8 ? 2 : 1>(y, nullptr, 0, a.spec + (long long)i * a.n_spec * a.spec_stride,
                                      cols + (long long)j * a.n_spec * a.spec_stride, a.spec_stride, a.n_spec, twl,
                                      wl, lane);
    {
      WinBits<R, 4> wb;
      win_bits<R, 4>(wb, lane, a.lag_lo, a.lag_hi);
      apply_window<R, 4>(y, wb);
    }
    const long long idx = a.out_ld ? (long long)(i - a.out_row0) * a.out_ld + (j - a.out_col0)
                                   : packed_index(i, j, a.n_events);
    // candidate slots of both sides first (one ballot per slot, kept in this
    // wave's LDS buffer, free after the transform), so the transform's
    // registers are dead during the FP64 evaluation
    unsigned long long* cmask = reinterpret_cast<unsigned long long*>(wl);  // [side][2R]
    for (int sd = 0; sd < 2; ++sd) {
      if (!(side & (1 << sd))) continue;
      const float sg = sd == 0 ? 1.f : -1.f;
      // FP32 winner of this side
      float bv = 0.f;
      sfor<0, 2 * R>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        const float v = sg * ((s & 1) ? y[s >> 1].y : y[s >> 1].x);
        bv = fmaxf(bv, v);
      });
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) bv = fmaxf(bv, __shfl_xor(bv, o, 64));
      const float cut = bv - a.tie_tol;
      sfor<0, 2 * R>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        const float v = sg * ((s & 1) ? y[s >> 1].y : y[s >> 1].x);
        const int lg = slot_lag<R>(lane, s);
        const bool inw = lg >= a.lag_lo && lg <= a.lag_hi;
        const unsigned long long m = __ballot(inw && v >= cut && v > 0.f);
        if (lane == 0) cmask[sd * 2 * R + s] = m;
      });
    }
    wave_lds_fence();
    // lane c: the norms of channel c
    const int nc = min(lane, a.n_channels - 1);
    const double norm_i = a.norms[(long long)i * a.n_channels + nc], norm_j = a.norms[(long long)j * a.n_channels + nc];
    for (int sd = 0; sd < 2; ++sd) {
      if (!(side & (1 << sd))) continue;
      const double sg = sd == 0 ? 1.0 : -1.0;
      double best = 0.0;
      int best_lag = 0;
      bool have = false;
      // the candidates in batches of four, each batch one pass over the traces
      // per channel (the FP64 sums of the reference's own arithmetic: the
      // convolution with the caller's reversed row when there is one)
      int batch[4] = {0, 0, 0, 0};
      int nb = 0;
      auto flush = [&]() {
        if (nb == 0) return;
        for (int q = nb; q < 4; ++q) batch[q] = batch[0];
        int shift[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          int t = a.rev_traces ? (batch[q] + a.rev_shift) % a.period : batch[q];
          shift[q] = t < 0 ? t + a.period : t;
        }
        double acc[4] = {0.0, 0.0, 0.0, 0.0};
        for (int c = 0; c < a.n_channels; ++c) {
          const double ni = __shfl(norm_i, c, 64), nj = __shfl(norm_j, c, 64);
          if (!(ni > 0.0 && nj > 0.0)) continue;
          const float* ti = a.traces + ((long long)i * a.n_channels + c) * a.tr_stride;
          double sum[4] = {0.0, 0.0, 0.0, 0.0};
          // a side's usual two candidates in a two-lag pass
          if (a.rev_traces) {
            const float* rj = a.rev_traces + ((long long)j * a.n_channels + c) * a.rev_stride;
            if (nb <= 2) corrn_f64<2>(ti, a.tr_len, rj, a.rev_len, a.period, shift, true, lane, sum);
            else corrn_f64<4>(ti, a.tr_len, rj, a.rev_len, a.period, shift, true, lane, sum);
          } else {
            const float* tj = a.traces + ((long long)j * a.n_channels + c) * a.tr_stride;
            if (nb <= 2) corrn_f64<2>(ti, a.tr_len, tj, a.tr_len, a.period, shift, false, lane, sum);
            else corrn_f64<4>(ti, a.tr_len, tj, a.tr_len, a.period, shift, false, lane, sum);
          }
          const double w = ni * nj * (double)a.n_channels;
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[q] += sum[q] / w;
        }
        for (int q = 0; q < nb; ++q) {
          const double v = sg * acc[q];
          if (v > 0.0 && (!have || v > best || (v == best && batch[q] < best_lag))) {
            best = v;
            best_lag = batch[q];
            have = true;
          }
        }
        nb = 0;
      };
      // 64 slots' masks at a time, one per lane; only slots with a candidate are
      // visited (reading each slot's mask in turn was 2R LDS round trips)
      for (int s0 = 0; s0 < 2 * R; s0 += 64) {
        const unsigned long long ms = s0 + lane < 2 * R ? cmask[sd * 2 * R + s0 + lane] : 0ull;
        unsigned long long hit = __ballot(ms != 0ull);
        while (hit) {
          const int u = __ffsll((long long)hit) - 1;
          hit &= hit - 1;
          unsigned long long mask =
              ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(ms >> 32), u) << 32) |
              (unsigned)__builtin_amdgcn_readlane((int)(unsigned)ms, u);
          while (mask) {
            const int src = __ffsll((long long)mask) - 1;
            mask &= mask - 1;
            batch[nb++] = slot_lag<R>(src, s0 + u);
            if (nb == 4) flush();
          }
        }
      }
      flush();
      if (lane == 0) {
        const float v = (float)best;
        if (sd == 0) {
          const bool keep = have && v > a.threshold;
          a.vpos[idx] = keep ? v : 0.f;
          a.lpos[idx] = keep ? best_lag : 0;
        } else {
          const bool keep = have && -v < -a.threshold;
          a.vneg[idx] = keep ? -v : 0.f;
          a.lneg[idx] = keep ? best_lag : 0;
        }
      }
    }
    wave_lds_fence();  // the next record rewrites the buffer
  }
}

// ----------------------------------------------------------------------------
// launchers (this translation unit instantiates one R, given by SXC_R)
// ----------------------------------------------------------------------------
template <int R>
hipError_t launch_forward_r(const ForwardArgs& a, hipStream_t st) {
  if (a.n_rows <= 0) return hipSuccess;
  constexpr int W = fwd_waves<R>();
  const size_t lds = (size_t)(TwLayout<R>::kFft + W * fwd_wave_buf<R>()) * sizeof(float2);
  auto kernel = a.n_seg > 0 ? k_forward<R, true> : k_forward<R, false>;
  hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  const long long groups = ((long long)a.n_rows * (a.n_seg > 0 ? a.n_seg * (a.seg_sides ? 1 : 2) : 1) + W - 1) / W;
  hipLaunchKernelGGL(kernel, dim3(groups < 1024 ? (int)groups : 1024), dim3(64 * W), lds, st, a);
  return hipGetLastError();
}

template <int R, int G, int W, int S, RowFrom kRow>
static hipError_t launch_pairs_rfw(const PairArgs& a, int grid, hipStream_t st) {
  const size_t lds = pair_lds_bytes(R, kRow == RowFrom::kLds ? a.n_channels : a.n_lds, W);
  static_assert(TwLayoutCT<R>::kInv == 640 + 8 * R, "compact twiddle layout");
  hipError_t e = hipFuncSetAttribute((const void*)k_pairs<R, G, W, S, kRow>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_pairs<R, G, W, S, kRow>), dim3(grid), dim3(W * 64), lds, st, a);
  return hipGetLastError();
}

// Narrow windows (G = 1, 2) where the build is kept (kNarrow); every window
// otherwise.
template <int R, int W, int S, RowFrom kRow, bool kNarrow>
static hipError_t launch_pairs_rw(int groups, const PairArgs& a, int grid, hipStream_t st) {
  if (groups == 0) return launch_pairs_rfw<R, 0, W, S, kRow>(a, grid, st);
  if constexpr (kNarrow) {
    if (groups == 1) return launch_pairs_rfw<R, 1, W, S, kRow>(a, grid, st);
    if (groups == 2) return launch_pairs_rfw<R, 2, W, S, kRow>(a, grid, st);
  }
  return launch_pairs_rfw<R, 4, W, S, kRow>(a, grid, st);
}

// Narrow-window builds go with the shapes of up to four channels (eight at the
// periods that cut rows use, P <= 2048);
// as many channels in LDS as the last shape holds when none holds all.
template <int R, int I>
static hipError_t launch_pairs_fit(int groups, const PairArgs& a, int grid, hipStream_t st) {
  constexpr PairShape k = pair_shape(R, I);
  if constexpr (k.waves > 0) {
    constexpr bool kNarrow = I == 0 || !pair_shape_fits(R, R <= 16 ? 8 : 4, pair_shape(R, I - (I > 0)));
    if (pair_shape_fits(R, a.n_channels, k))
      return launch_pairs_rw<R, k.waves, k.per_simd, RowFrom::kLds, kNarrow>(groups, a, grid, st);
    return launch_pairs_fit<R, I + 1>(groups, a, grid, st);
  } else {
    constexpr PairShape last = pair_shape(R, I - 1);
    if constexpr (!pair_shape_fits(R, 8, last)) {
      PairArgs b = a;
      for (b.n_lds = 1; pair_shape_fits(R, b.n_lds + 1, last);) ++b.n_lds;
      return launch_pairs_rw<R, last.waves, last.per_simd, RowFrom::kBoth, false>(groups, b, grid, st);
    }
  }
  return hipErrorInvalidValue;  // not reached: the last shape holds 8 channels, a plan's most
}

template <int R>
hipError_t launch_pairs_r(bool full, const PairArgs& a, int grid, hipStream_t st) {
  // Runs of 16 R lags the window reaches into on either side of lag 0: the
  // narrowest build that holds them (win_regs).  Measured at N = 3001, C = 3,
  // P = 4096: +-512 (G = 2) 20.2 ms -> 18.0
  // with every value masked by a per-slot lane mask before; N = 3000, C = 3,
  // P = 2048, every overlapping lag (G = 4) 10.8 -> 9.4.
  constexpr int kRun = 16 * R;
  const int runs = (a.lag_hi >= 0 ? a.lag_hi / kRun + 1 : 0), below = (a.lag_lo < 0 ? (-a.lag_lo + kRun - 1) / kRun : 0);
  const int need = runs > below ? runs : below;
  const int groups = full ? 0 : (need <= 1 ? 1 : (need == 2 ? 2 : 4));
  return launch_pairs_fit<R, 0>(groups, a, grid, st);
}

template <int R>
hipError_t launch_resolve_r(const ResolveArgs& a, int grid, hipStream_t st) {
  size_t lds = (size_t)(TwLayoutCT<R>::kInv + kWaveLds) * sizeof(float2);
  hipError_t e = hipFuncSetAttribute((const void*)k_resolve<R>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_resolve<R>, dim3(grid), dim3(64), lds, st, a);
  return hipGetLastError();
}

template hipError_t launch_forward_r<SXC_R>(const ForwardArgs&, hipStream_t);
template hipError_t launch_pairs_r<SXC_R>(bool, const PairArgs&, int, hipStream_t);
template hipError_t launch_resolve_r<SXC_R>(const ResolveArgs&, int, hipStream_t);

#if SXC_R == 8
// Plain streaming copy of n float4 (device bandwidth reference for profiling).
__global__ __launch_bounds__(256) void k_copy_f4(float4* __restrict__ dst, const float4* __restrict__ src,
                                                 long long n) {
  for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    dst[i] = src[i];
}

hipError_t launch_copy_f4(float4* dst, const float4* src, long long n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  long long blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_copy_f4, dim3((unsigned)blocks), dim3(256), 0, st, dst, src, n);
  return hipGetLastError();
}

// Top k of a row (or of a slice of its columns), larger value first, then the
// smaller column -> out[(row * slices + slice) * k ...] as (value, lag, idx_in[c]
// when given, else the column c), padded with (-inf, 0, -1).
//
// A latency chain, so nothing waits on a barrier until the end: every wave walks
// its own share of the columns, 64 kV at a time in registers (each lane's sorted,
// so that its best is at hand), with its k best in lanes 0 .. k-1, best first; a
// round takes the largest of what is left (one DPP reduction over values, one
// over columns), shifts it into the list and stops at the first that is no better
// than the k-th.  The first wave then absorbs the others' lists the same way.
// 4096 columns, k = 10, one row 8.5 us (two launches of 20.7 with a sorted list per
// thread and k rounds of shuffles before; 16 waves of 4 values and 4 of 16, unsorted
// and shifted by shuffles, 18.9 and 23.5).
constexpr int kTopkMax = 32;
constexpr int kTopkWaves = 8;
typedef unsigned long long u64;
// A candidate: its value's bits in unsigned order (-0 as +0), then ~column; 0: none,
// which is what a NaN gives.
__device__ __forceinline__ u64 topk_cand(float v, int c) {
  const unsigned u = __float_as_uint(v + 0.f);
  const unsigned key = (u >> 31) ? ~u : u | 0x80000000u;
  return v != v ? 0ull : (u64)key << 32 | ~(unsigned)c;
}
__device__ __forceinline__ float topk_value(u64 c) {
  const unsigned key = (unsigned)(c >> 32);
  return __uint_as_float((key >> 31) ? key & 0x7fffffffu : ~key);
}
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
#pragma unroll
  for (int k = 0; k < 6; ++k) v = max(v, (unsigned)dpp_i((int)v, k));
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
// A lane's V candidates in descending order (Batcher's odd-even merge network).
template <int V>
__device__ __forceinline__ void topk_sort(u64 (&c)[V]) {
#pragma unroll
  for (int p = 1; p < V; p *= 2)
#pragma unroll
    for (int q = p; q >= 1; q /= 2)
#pragma unroll
      for (int a = 0; a + q < V; ++a)
        if (a >= q % p && (a - q % p) / q % 2 == 0 && a / (2 * p) == (a + q) / (2 * p)) {
          const u64 x = c[a], y = c[a + q];
          c[a] = x > y ? x : y;
          c[a + q] = x > y ? y : x;
        }
}
// Every lane's candidates (sorted; used up) into the list t.
template <int V>
__device__ __forceinline__ void topk_absorb(u64& t, int k, int lane, u64 (&c)[V]) {
  for (;;) {
    const unsigned hi = (unsigned)(c[0] >> 32), m = wave_max_u32(hi);
    if (m == 0u) return;
    const unsigned w = wave_max_u32(hi == m ? (unsigned)c[0] : 0u);
    const u64 best = (u64)m << 32 | w;
    const u64 last = (u64)(unsigned)__builtin_amdgcn_readlane((int)(t >> 32), k - 1) << 32 |
                     (unsigned)__builtin_amdgcn_readlane((int)t, k - 1);
    if (best <= last) return;
    const int rank = __popcll(__ballot(t > best));
    // the lane before's entry (wave shift right by one)
    const u64 before = (u64)(unsigned)__builtin_amdgcn_update_dpp(0, (int)(t >> 32), 0x138, 0xF, 0xF, true) << 32 |
                       (unsigned)__builtin_amdgcn_update_dpp(0, (int)t, 0x138, 0xF, 0xF, true);
    t = lane == rank ? best : (lane > rank ? before : t);
    const bool owner = c[0] == best;
#pragma unroll
    for (int u = 0; u < V; ++u) c[u] = owner ? (u + 1 < V ? c[u + 1 < V ? u + 1 : u] : 0ull) : c[u];
  }
}
__global__ __launch_bounds__(64 * kTopkWaves) void k_topk(const float* __restrict__ v, const int* __restrict__ l,
                                                          const int* __restrict__ idx_in, long long row_stride,
                                                          int n_cols, int k, float* out_v, int* out_l, int* out_idx) {
  constexpr int kV = 8;
  __shared__ u64 lists[kTopkWaves * kTopkMax];
  const int row = blockIdx.x, slice = blockIdx.y, n_slices = gridDim.y;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int width = (n_cols + n_slices - 1) / n_slices;
  const int cb = slice * width, ce = min(n_cols, cb + width);
  const long long base = (long long)row * row_stride;
  u64 t = 0ull;
  for (int c0 = cb + wv * 64 * kV; c0 < ce; c0 += kTopkWaves * 64 * kV) {
    float x[kV];
    u64 c[kV];
#pragma unroll
    for (int u = 0; u < kV; ++u) x[u] = v[base + min(c0 + 64 * u + lane, ce - 1)];
#pragma unroll
    for (int u = 0; u < kV; ++u) {
      const int col = c0 + 64 * u + lane;
      c[u] = col < ce ? topk_cand(x[u], col) : 0ull;
    }
    topk_sort<kV>(c);
    topk_absorb<kV>(t, k, lane, c);
  }
  if (lane < kTopkMax) lists[wv * kTopkMax + lane] = t;
  __syncthreads();
  if (wv != 0) return;
  constexpr int kL = kTopkWaves * kTopkMax / 64;
  u64 c[kL];
#pragma unroll
  for (int u = 0; u < kL; ++u) {
    const int e = lane + 64 * u;  // list 0 is this wave's own
    c[u] = e >= kTopkMax && e % kTopkMax < k ? lists[e] : 0ull;
  }
  topk_sort<kL>(c);
  topk_absorb<kL>(t, k, lane, c);
  if (lane < k) {
    const long long o = ((long long)row * n_slices + slice) * k + lane;
    const bool ok = t != 0ull;
    const int col = (int)~(unsigned)t;
    out_v[o] = ok ? topk_value(t) : -INFINITY;
    out_idx[o] = ok ? (idx_in ? idx_in[base + col] : col) : -1;
    out_l[o] = ok ? l[base + col] : 0;
  }
}

static void launch_topk_any(const float* v, const int* l, const int* idx_in, long long row_stride, int n_rows,
                            int n_slices, int n_cols, int k, float* out_v, int* out_l, int* out_idx,
                            hipStream_t st) {
  hipLaunchKernelGGL(k_topk, dim3(n_rows, n_slices), dim3(64 * kTopkWaves), 0, st, v, l, idx_in, row_stride, n_cols,
                     k, out_v, out_l, out_idx);
}

hipError_t launch_topk(const float* v, const int* l, int n_rows, int n_cols, int k, float* out_v,
                       int* out_l, int* out_idx, hipStream_t st) {
  if (n_rows <= 0) return hipSuccess;
  if (k < 1 || k > kTopkMax) return hipErrorInvalidValue;
  launch_topk_any(v, l, nullptr, n_cols, n_rows, 1, n_cols, k, out_v, out_l, out_idx, st);
  return hipGetLastError();
}

hipError_t launch_topk_split(const float* v, const int* l, int n_rows, int n_cols, int k, int n_slices,
                             float* tmp_v, int* tmp_l, int* tmp_idx, float* out_v, int* out_l, int* out_idx,
                             hipStream_t st) {
  if (n_rows <= 0) return hipSuccess;
  if (k < 1 || k > kTopkMax || n_slices < 1 || n_slices > kTopkMaxSlices) return hipErrorInvalidValue;
  if (n_slices == 1) return launch_topk(v, l, n_rows, n_cols, k, out_v, out_l, out_idx, st);
  launch_topk_any(v, l, nullptr, n_cols, n_rows, n_slices, n_cols, k, tmp_v, tmp_l, tmp_idx, st);
  const int m = n_slices * k;  // candidates per row
  launch_topk_any(tmp_v, tmp_l, tmp_idx, m, n_rows, 1, m, k, out_v, out_l, out_idx, st);
  return hipGetLastError();
}

hipError_t launch_fill_u32(unsigned* p, unsigned v, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill_u32, dim3((n + 255) / 256), dim3(256), 0, st, p, v, n);
  return hipGetLastError();
}
#endif

}  // namespace sxc
