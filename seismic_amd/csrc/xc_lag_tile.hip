// Lag-window form on MFMA (gfx950) for windows of few lags on many samples: the
// correlation as a product per lag over tiles of 32 x 32 pairs.
//
// For pairs (i, j) in a 32 x 32 tile and a block of kTileLags (16) consecutive lags
// l = lb + d, the coefficient c_ij(l) = sum_c sum_n xh_ic[n] xh_jc[n - l] is a
// 32 x 32 x K product per lag with K running over all samples and channels:
//   A (32 x 16) = row traces xh_i[n0 .. n0+16)       (held per K step)
//   B (16 x 32) = column traces xh_j[n0 - l .. )      (a shifted window)
// on v_mfma_f32_32x32x16_{bf16,f16}.  Each lane loads one 24-element window
// of its column trace per K step and forms the 16 shifted operands with
// v_alignbyte (odd shifts) or plain register selection (even shifts).  The
// 16 lag accumulators (32 x 32 FP32 each) live in the accumulation registers.
//
// The product over lags (xc_lag.hip) loads an operand for every 32 x 32 products of
// 32 lags and one row, and with one or two blocks of lags is bound by those loads
// once the traces no longer stay in the caches; here 16 lags of a tile share
// them.  lag_tiles (xc_lag.h) says which windows run here.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "xc_lag.h"

namespace sxc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// ----------------------------------------------------------------------------
// tile kernel: one workgroup (4 waves) per 32 x 32 tile of pairs
// ----------------------------------------------------------------------------
// MFMA 32x32x16 operand layout: lane l supplies A[l % 32][8*(l/32) + e] and
// B[8*(l/32) + e][l % 32], e < 8; result register r of lane l holds
// D[8*(r/4) + 4*(l/32) + r%4][l % 32].
__device__ __forceinline__ int mfma_row(int lane, int r) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

template <int B, int E, typename F>
__device__ __forceinline__ void sfor_tile(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    sfor_tile<B + 1, E>(f);
  }
}

// One K step's operands for this lane: A (row) 8 samples and the B (column)
// window of 24 samples, hi and (bf16x3) lo planes.
struct StepData {
  u32x4 ah, al;
  u32x4 bh[3], bl[3];
};

// One K step's operands from this lane's row (A) and column window (B)
// bases, `off` elements into the plane row (the step's channel and sample).
template <bool BF16X3>
__device__ __forceinline__ void load_step(StepData& s, const unsigned short* __restrict__ ahi,
                                          const unsigned short* __restrict__ alo,
                                          const unsigned short* __restrict__ bhi,
                                          const unsigned short* __restrict__ blo, int off) {
  s.ah = *reinterpret_cast<const u32x4*>(ahi + off);
#pragma unroll
  for (int q = 0; q < 3; ++q) s.bh[q] = *reinterpret_cast<const u32x4*>(bhi + off + 8 * q);
  if constexpr (BF16X3) {
    s.al = *reinterpret_cast<const u32x4*>(alo + off);
#pragma unroll
    for (int q = 0; q < 3; ++q) s.bl[q] = *reinterpret_cast<const u32x4*>(blo + off + 8 * q);
  }
}

// 12 dwords (24 elements) -> the 4 dwords starting at element O (0 <= O <= 16)
template <int O>
__device__ __forceinline__ u32x4 window_frag3(const u32x4 (&w)[3]) {
  auto word = [&](int k) { return w[k >> 2][k & 3]; };
  u32x4 r;
  if constexpr ((O & 1) == 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = word(O / 2 + k);
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = __builtin_amdgcn_alignbyte(word((O + 1) / 2 + k), word((O - 1) / 2 + k), 2);
  }
  return r;
}

template <bool BF16X3>
__device__ __forceinline__ void mfma_step(f32x16 (&acc)[kTileLags], const StepData& s) {
  // lag lb + d uses window elements 15 - d .. 22 - d
  auto step = [&](auto dc) {
    constexpr int d = decltype(dc)::value;
    const u32x4 b_h = window_frag3<15 - d>(s.bh);
    if constexpr (BF16X3) {
      const u32x4 b_l = window_frag3<15 - d>(s.bl);
      const bf16x8 A_h = __builtin_bit_cast(bf16x8, s.ah), A_l = __builtin_bit_cast(bf16x8, s.al);
      const bf16x8 B_h = __builtin_bit_cast(bf16x8, b_h), B_l = __builtin_bit_cast(bf16x8, b_l);
      acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A_l, B_h, acc[d], 0, 0, 0);
      acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A_h, B_l, acc[d], 0, 0, 0);
      acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A_h, B_h, acc[d], 0, 0, 0);
    } else {
      const f16x8 A_h = __builtin_bit_cast(f16x8, s.ah), B_h = __builtin_bit_cast(f16x8, b_h);
      acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A_h, B_h, acc[d], 0, 0, 0);
    }
  };
  sfor_tile<0, kTileLags>(step);
}

// All K steps (channels x samples) of one block of kTileLags lags.  Operands
// are loaded kDepth steps ahead (a ring of kDepth buffers) so one wave per
// SIMD keeps the MFMA pipe fed: 2 steps for bf16x3 (48 MFMAs per step), 4 for
// fp16 (16 MFMAs per step, fewer registers per buffer).  The load cursor (the
// step's element offset in the plane row) advances by additions only: with
// one wave per SIMD every scalar instruction takes an issue slot from the
// MFMAs.
template <bool BF16X3>
__device__ __forceinline__ void lag_block(f32x16 (&acc)[kTileLags], const unsigned short* __restrict__ ahi,
                                          const unsigned short* __restrict__ alo,
                                          const unsigned short* __restrict__ bhi,
                                          const unsigned short* __restrict__ blo, int ls,
                                          int n_channels, int l16, int p0, int lb, int h) {
  constexpr int kDepth = BF16X3 ? 2 : 4;
#pragma unroll
  for (int d = 0; d < kTileLags; ++d) acc[d] = f32x16{};
  const int total = n_channels * (l16 / 16);  // >= 1
  // lane bases: A at sample 8h of the step, B window 15 + lb samples earlier
  ahi += p0 + 8 * h;
  bhi += p0 + 8 * h - lb - 15;
  if constexpr (BF16X3) {
    alo += p0 + 8 * h;
    blo += p0 + 8 * h - lb - 15;
  }
  // cursor: element offset of the next step to load, samples of its channel
  // before it, and steps left before it stops at the last one (loads past
  // the end repeat that step: harmless and in bounds)
  int ld_off = 0, ld_n = 0, ld_left = total - 1;
  auto advance = [&]() {
    if (ld_left > 0) {
      --ld_left;
      ld_n += 16;
      const bool wrap = ld_n == l16;
      ld_off += wrap ? ls - l16 + 16 : 16;
      ld_n = wrap ? 0 : ld_n;
    }
  };
  StepData buf[kDepth];
#pragma unroll
  for (int q = 0; q < kDepth; ++q) {
    load_step<BF16X3>(buf[q], ahi, alo, bhi, blo, ld_off);
    advance();
  }
  for (int st = 0; st < total; st += kDepth) {
#pragma unroll
    for (int q = 0; q < kDepth; ++q) {
      if (st + q < total) {
        mfma_step<BF16X3>(acc, buf[q]);
        // scheduling: the operand assembly (v_mov, v_alignbyte) spread
        // evenly between the MFMAs, so the single wave keeps issuing while
        // its MFMAs run (fp16 4.6% faster, bf16x3 0.3%; same instructions)
#pragma unroll
        for (int g = 0; g < (BF16X3 ? 48 : 16); ++g) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, BF16X3 ? 3 : 5, 0);  // then up to this many VALU
        }
      }
      load_step<BF16X3>(buf[q], ahi, alo, bhi, blo, ld_off);
      advance();
    }
  }
}

// Running per-pair state of one wave, in LDS, lane-contiguous so every
// access is bank-conflict free: [wave][pair r][...][lane].  Per side the three
// largest values (pos: p1 >= p2 >= p3; neg: n1 <= n2 <= n3) and the lags of
// the first two as 16-bit offsets from lag_first, packed into one word.
struct LagState {
  float v[4][16][6][64];  // p1 p2 p3 n1 n2 n3
  unsigned l[4][16][2][64];  // (lp1 | lp2 << 16), (ln1 | ln2 << 16) - lag_first
};

// Merge of two descending top-3 lists (values a/b, lags of the first two) into
// the top three of their union; ties of the first place go to the smaller lag
// (the two lists cover disjoint lag blocks).  The negative side calls it with
// negated values.
__device__ __forceinline__ void merge_top3(float& a1, float& a2, float& a3, unsigned& la1, unsigned& la2,
                                           float b1, float b2, float b3, unsigned lb1, unsigned lb2) {
  const bool take_b = b1 > a1 || (b1 == a1 && lb1 < la1);
  // W: the list whose head wins, O: the other
  const float w1 = take_b ? b1 : a1, w2 = take_b ? b2 : a2, w3 = take_b ? b3 : a3;
  const unsigned lw1 = take_b ? lb1 : la1, lw2 = take_b ? lb2 : la2;
  const float o1 = take_b ? a1 : b1, o2 = take_b ? a2 : b2;
  const unsigned lo1 = take_b ? la1 : lb1;
  const bool o_second = o1 > w2;
  a1 = w1;
  la1 = lw1;
  a2 = o_second ? o1 : w2;
  la2 = o_second ? lo1 : lw2;
  a3 = o_second ? fmaxf(w2, o2) : fmaxf(w3, o1);
}

template <bool BF16X3>
__global__ __launch_bounds__(256, 1) void k_lag_tiles(LagPairArgs a) {
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int h = lane >> 5;
  __shared__ LagState st;
  for (int item = blockIdx.x; item < a.n_tiles; item += gridDim.x) {
    const int2 t = a.tiles[item];
    const int i0 = 32 * (t.x + a.tile_row0), j0 = 32 * (t.y + a.tile_col0);
    if (i0 >= a.n_events || j0 >= a.n_events) continue;  // ragged last block (workgroup-uniform)
    // this lane's A row and B column (clamped: rows past N compute values that are never stored)
    const int ia = min(i0 + (lane & 31), a.n_events - 1);
    const int jb = min(j0 + (lane & 31), a.n_events - 1);
    const long long rs = (long long)a.n_channels * a.ls;
    const unsigned short* ahi = a.p_hi + ia * rs;
    const unsigned short* alo = BF16X3 ? a.p_lo + ia * rs : nullptr;
    const unsigned short* bhi = a.p_hi + jb * rs;
    const unsigned short* blo = BF16X3 ? a.p_lo + jb * rs : nullptr;
    __syncthreads();  // the previous tile's merge has read the state
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      st.v[wv][r][0][lane] = 0.f; st.v[wv][r][1][lane] = -3.0e38f; st.v[wv][r][2][lane] = -3.0e38f;
      st.v[wv][r][3][lane] = 0.f; st.v[wv][r][4][lane] = 3.0e38f; st.v[wv][r][5][lane] = 3.0e38f;
      st.l[wv][r][0][lane] = 0u; st.l[wv][r][1][lane] = 0u;
    }
    for (int b = wv; b < a.n_blocks; b += 4) {
      const int lb = a.lag_first + kTileLags * b;
      f32x16 acc[kTileLags];
      lag_block<BF16X3>(acc, ahi, alo, bhi, blo, (int)a.ls, a.n_channels, a.l16, a.p0, lb, h);
      // top-3 values (top-2 lags) per pair over the block's lags, in increasing lag order
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float p1 = st.v[wv][r][0][lane], p2 = st.v[wv][r][1][lane], p3 = st.v[wv][r][2][lane];
        float n1 = st.v[wv][r][3][lane], n2 = st.v[wv][r][4][lane], n3 = st.v[wv][r][5][lane];
        const unsigned wp = st.l[wv][r][0][lane], wn = st.l[wv][r][1][lane];
        unsigned lp1 = wp & 0xffffu, lp2 = wp >> 16, ln1 = wn & 0xffffu, ln2 = wn >> 16;
#pragma unroll
        for (int d = 0; d < kTileLags; ++d) {
          const int lag = lb + d;
          const unsigned off = (unsigned)(kTileLags * b + d);
          const bool in = lag >= a.lag_lo && lag <= a.lag_hi;
          const float v = in ? acc[d][r] : 0.f;
          const bool gp = v > p1;
          const bool sp = !gp && v > p2;
          p3 = (gp || sp) ? p2 : fmaxf(p3, v);
          p2 = gp ? p1 : (sp ? v : p2);
          lp2 = gp ? lp1 : (sp ? off : lp2);
          p1 = gp ? v : p1;
          lp1 = gp ? off : lp1;
          const bool gn = v < n1;
          const bool sn = !gn && v < n2;
          n3 = (gn || sn) ? n2 : fminf(n3, v);
          n2 = gn ? n1 : (sn ? v : n2);
          ln2 = gn ? ln1 : (sn ? off : ln2);
          n1 = gn ? v : n1;
          ln1 = gn ? off : ln1;
        }
        st.v[wv][r][0][lane] = p1; st.v[wv][r][1][lane] = p2; st.v[wv][r][2][lane] = p3;
        st.v[wv][r][3][lane] = n1; st.v[wv][r][4][lane] = n2; st.v[wv][r][5][lane] = n3;
        st.l[wv][r][0][lane] = lp1 | (lp2 << 16);
        st.l[wv][r][1][lane] = ln1 | (ln2 << 16);
      }
    }
    // merge the 4 waves' states (lag blocks interleave, so ties go to the smaller lag)
    __syncthreads();
    if (wv == 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float p1 = st.v[0][r][0][lane], p2 = st.v[0][r][1][lane], p3 = st.v[0][r][2][lane];
        float n1 = -st.v[0][r][3][lane], n2 = -st.v[0][r][4][lane], n3 = -st.v[0][r][5][lane];
        unsigned lp1 = st.l[0][r][0][lane] & 0xffffu, lp2 = st.l[0][r][0][lane] >> 16;
        unsigned ln1 = st.l[0][r][1][lane] & 0xffffu, ln2 = st.l[0][r][1][lane] >> 16;
        for (int w = 1; w < 4; ++w) {
          const unsigned qp = st.l[w][r][0][lane], qn = st.l[w][r][1][lane];
          merge_top3(p1, p2, p3, lp1, lp2, st.v[w][r][0][lane], st.v[w][r][1][lane], st.v[w][r][2][lane],
                     qp & 0xffffu, qp >> 16);
          merge_top3(n1, n2, n3, ln1, ln2, -st.v[w][r][3][lane], -st.v[w][r][4][lane], -st.v[w][r][5][lane],
                     qn & 0xffffu, qn >> 16);
        }
        n1 = -n1; n2 = -n2; n3 = -n3;
        const int i = i0 + mfma_row(lane, r);
        const int j = j0 + (lane & 31);
        if (i < a.n_events && j < a.n_events && j >= i) {
          const long long idx = lag_out_index(a, i, j);
          const bool kp = p1 > a.threshold && p1 > 0.f;
          const bool kn = n1 < -a.threshold && n1 < 0.f;
          const int glp1 = a.lag_first + (int)lp1, gln1 = a.lag_first + (int)ln1;
          a.vpos[idx] = kp ? p1 : 0.f;
          a.lpos[idx] = kp ? glp1 : 0;
          a.vneg[idx] = kn ? n1 : 0.f;
          a.lneg[idx] = kn ? gln1 : 0;
          const bool tp = kp && (p1 - p2 < a.tie_tol || p1 < a.tie_tol);
          const bool tn = kn && (n2 - n1 < a.tie_tol || -n1 < a.tie_tol);
          // a third lag within the band: every in-window lag is a candidate
          const bool wp = tp && (p1 - p3 < a.tie_tol || p1 < a.tie_tol);
          const bool wn = tn && (n3 - n1 < a.tie_tol || -n1 < a.tie_tol);
          if (tp || tn) {
            const unsigned slot = atomicAdd(a.tie_count, 1u);
            if (slot < (unsigned)a.tie_cap) {
              a.ties[2 * slot] = make_int4(i, j, (tp ? 1 : 0) | (tn ? 2 : 0) | (wp ? 4 : 0) | (wn ? 8 : 0), 0);
              a.ties[2 * slot + 1] = make_int4(glp1, a.lag_first + (int)lp2, gln1, a.lag_first + (int)ln2);
            }
          }
        }
      }
    }
  }
}

hipError_t launch_lag_tiles(bool bf16x3, const LagPairArgs& a, hipStream_t st) {
  if (a.n_tiles <= 0) return hipSuccess;
  const int grid = a.n_tiles < (1 << 20) ? a.n_tiles : 1 << 20;
  if (bf16x3)
    hipLaunchKernelGGL(k_lag_tiles<true>, dim3(grid), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(k_lag_tiles<false>, dim3(grid), dim3(256), 0, st, a);
  return hipGetLastError();
}

}  // namespace sxc
