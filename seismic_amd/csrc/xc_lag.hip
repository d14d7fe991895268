// Lag-window form on MFMA (gfx950): the correlation over a bounded window of
// lags as dense products.  (Some windows of few lags run tile by tile instead:
// xc_lag_tile.hip.)
//
// The coefficient c_ij(l) = sum_c sum_n xh_ic[n] xh_jc[n - l]
// (xh = x / (|x| sqrt(C)), linear correlation, zero outside [0, L)) is, with
// n = k + l, sum_k xh_i[k + l] xh_j[k].  For one row event i, 32 column events j
// and a block of kLagBlock (32) consecutive lags it is a 32 x 32 x K product
// with K running over samples and channels:
//   A (32 x 16): row r = lag lb + lag(r), A[r][k] = xh_i[k + lb + lag(r)] (a
//                Hankel matrix with its even rows first: lag(r) = 2 (r % 16) + r / 16)
//   B (16 x 32): column = event j, B[k][j] = xh_j[k]
// on v_mfma_f32_32x32x16_{bf16,f16}.  A depends on k + lb only, so the A operand
// of lag block b at step s is that of block b + 1 one step (32 samples)
// earlier: a wave holds NB blocks' accumulators and a ring of A operands, and a
// step of NB products needs one new A and one B operand, both loaded as they
// are used -- no operand is assembled from others.
//
// Precision forms
//   bf16x3: xh = hi + lo with hi = bf16(xh), lo = bf16(xh - hi); the product
//           is hi*hi + hi*lo + lo*hi with FP32 accumulation (3 MFMAs);
//   fp16:   one FP16 product, FP32 accumulation.
// FP64 is used for the per-trace energy and scale, and for the near-tie
// re-evaluation (k_lag_resolve at the two recorded lags; records with a
// third lag inside the band go to the FFT form's resolver, which finds every
// candidate from the pair's FP32 transform).  Scan rule as in the reference
// (Correlation_in_OMP/correlation_c.cpp:102-136): pos = largest value above
// 0 at its first lag, neg = smallest below 0, threshold to (0, 0).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "xc_lag.h"

namespace sxc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// round-to-nearest-even FP32 -> bf16 bits (NaN kept quiet)
__device__ __forceinline__ unsigned short f32_to_bf16_rne(float f) {
  unsigned u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (unsigned short)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf16_to_f32(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

// ----------------------------------------------------------------------------
// prep: one workgroup per (event, channel) row
// ----------------------------------------------------------------------------
// Column operand of a row: blocked [event / 32][channel][sample / 8][event % 32][8],
// so the 64 lanes of an operand load read 1 KiB in one piece.
template <typename Part>
__device__ __forceinline__ void store_columns(const LagPrepArgs& a, int row, Part&& part) {
  const int ev = row / a.n_channels, c = row - ev * a.n_channels, n8 = a.l16 / 8;
  const long long base = ((long long)(ev / 32) * a.n_channels + c) * n8 * 32 + ev % 32;
  for (int g = threadIdx.x; g < n8; g += 256) {
    u32x4 hv, lv;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      unsigned short h[2], l[2];
      part(8 * g + 2 * w, h[0], l[0]);
      part(8 * g + 2 * w + 1, h[1], l[1]);
      hv[w] = h[0] | (unsigned)h[1] << 16;
      lv[w] = l[0] | (unsigned)l[1] << 16;
    }
    reinterpret_cast<u32x4*>(a.b_hi)[base + 32ll * g] = hv;
    if (a.b_lo) reinterpret_cast<u32x4*>(a.b_lo)[base + 32ll * g] = lv;
  }
}

// What a launch makes: the operands, the row operands alone (LagPrepArgs::energy_in)
// or planes (p_hi).
enum class Prep { kOperands, kRows, kPlanes };
template <Prep kWhat>
__global__ __launch_bounds__(256) void k_lag_prep(LagPrepArgs a) {
  const int row = blockIdx.x;
  if (row == 0 && threadIdx.x == 0) {
    if (a.zero0) *a.zero0 = 0u;
    if (a.zero1) *a.zero1 = 0u;
  }
  if (kWhat == Prep::kOperands && row >= a.n_rows) {  // the last column tile's empty events
    store_columns(a, row, [](int, unsigned short& h, unsigned short& l) { h = l = 0; });
    return;
  }
  const float* x = a.in + (long long)row * a.in_stride;
  __shared__ double red[256];
  double mean = 0.0, E;
  if constexpr (kWhat == Prep::kRows) {
    E = a.energy_in[row];
  } else {
    double s1 = 0.0;
    for (int n = threadIdx.x; n < a.L; n += 256) s1 += (double)(n < a.in_len ? x[n] : 0.f);
    red[threadIdx.x] = s1;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
      if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
      __syncthreads();
    }
    mean = a.demean ? red[0] / (double)a.L : 0.0;
    __syncthreads();
    double s2 = 0.0;
    for (int n = threadIdx.x; n < a.L; n += 256) {
      const float v = n < a.in_len ? x[n] : 0.f;
      const float u = a.demean ? (float)((double)v - mean) : v;
      s2 += (double)u * (double)u;
    }
    red[threadIdx.x] = s2;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
      if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
      __syncthreads();
    }
    E = red[0];
    if (threadIdx.x == 0) {
      a.norms[row] = sqrt(E);
      if (a.energy) a.energy[row] = E;
    }
  }
  const double scale = E > 0.0 ? 1.0 / sqrt(E * (double)a.n_channels) : 0.0;
  // A row with a NaN or infinite sample has no coefficients: NaN throughout, so
  // that every lag of its pairs is NaN whatever samples a range of lags skips,
  // and the pairs come out as (0, lag 0) as in the FFT form.
  const float outside = E <= 1.7e308 ? 0.f : __int_as_float(0x7fc00000);
  auto store_trace = [&] {
    if (!a.traces_out) return;
    float* tr = a.traces_out + (long long)row * a.L;
    for (int n = threadIdx.x; n < a.L; n += 256) {
      const float v = n < a.in_len ? x[n] : 0.f;
      tr[n] = a.demean && n < a.in_len ? (float)((double)v - mean) : v;
    }
  };
  // sample n of the scaled trace as its 16-bit hi and lo parts
  auto part = [&](int n, unsigned short& h, unsigned short& l) {
    float v = outside;
    if (outside == 0.f && n >= 0 && n < a.L && n < a.in_len) {
      const float u = a.demean ? (float)((double)x[n] - mean) : x[n];
      v = (float)((double)u * scale);
    }
    if (a.fp16) {
      h = __builtin_bit_cast(unsigned short, (_Float16)v);
      l = 0;
    } else {
      h = f32_to_bf16_rne(v);
      l = f32_to_bf16_rne(v - bf16_to_f32(h));
    }
  };
  if constexpr (kWhat == Prep::kPlanes) {
    for (int s = threadIdx.x; s < a.ls; s += 256) {
      unsigned short h, l;
      part(s - a.p0, h, l);
      a.p_hi[(long long)row * a.ls + s] = h;
      if (a.p_lo) a.p_lo[(long long)row * a.ls + s] = l;
    }
    store_trace();
    return;
  }
  // row operand: element q of copy 0 is sample q + lag_first, of copy 1 the next
  unsigned* h0 = reinterpret_cast<unsigned*>(a.h_hi + (long long)row * 2 * a.hs);
  unsigned* l0 = a.h_lo ? reinterpret_cast<unsigned*>(a.h_lo + (long long)row * 2 * a.hs) : nullptr;
  for (int q = threadIdx.x; q < a.hs / 2; q += 256) {
    unsigned short h[3], l[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) part(2 * q + u + a.lag_first, h[u], l[u]);
    h0[q] = h[0] | (unsigned)h[1] << 16;
    h0[a.hs / 2 + q] = h[1] | (unsigned)h[2] << 16;
    if (l0) {
      l0[q] = l[0] | (unsigned)l[1] << 16;
      l0[a.hs / 2 + q] = l[1] | (unsigned)l[2] << 16;
    }
  }
  if constexpr (kWhat == Prep::kRows) return;
  store_columns(a, row, part);
  store_trace();
}

// ----------------------------------------------------------------------------
// pair kernel
// ----------------------------------------------------------------------------
// MFMA 32x32x16 operand layout: lane l supplies A[l % 32][8*(l/32) + e] and
// B[8*(l/32) + e][l % 32], e < 8; result register r of lane l holds
// D[8*(r/4) + 4*(l/32) + r%4][l % 32].
//
// Lag within a block of register r: the registers' rows 8 (r/4) + 4 h + r%4 hold
// even lags for r < 8 and the odd ones after them for r >= 8.  Operand loads
// move 64 bytes per cycle when four neighbouring lanes read one 64-byte piece;
// with rows in lag order neighbours alternated between the two copies a row
// operand is stored in (36 instead of about 22 cycles per load: N = 3000,
// L = 2048, +-20:
// fp16 2.48 -> 2.05 ms, bf16x3 3.46 -> 2.98).
__device__ __forceinline__ constexpr int lag_in_block(int h, int r) {
  return 2 * (8 * ((r & 7) >> 2) + 4 * h + (r & 3)) + (r >> 3);
}
// Registers in increasing lag order: order(r) = 2 (r % 8) + r / 8, and back.
__device__ __forceinline__ constexpr int lag_order(int r) { return 2 * (r & 7) + (r >> 3); }
__device__ __forceinline__ constexpr int order_lag(int h, int o) { return lag_in_block(h, (o >> 1) + 8 * (o & 1)); }

// Operands go through buffer resources (scalar base and offset, one lane offset,
// constants as immediates).  Loads that run ahead of the last product reach up to
// kLagAhead elements past an operand.  The range check need not cover the scalar
// offset, so those elements are allocated too (lag_operands): clamping the offsets
// instead cost fp16 0.6% (N = 2001, L = 4096, +-512 12.72 -> 12.80 ms).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_rsrc(const unsigned short* base, long long elems) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)(2 * elems), 0x00020000);
}
__device__ __forceinline__ u32x4 plane_load(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// v_med3 on integers (the compiler forms it from four instructions' worth of
// min and max only when it can see the order of two operands).
__device__ __forceinline__ int med3_i(int a, int b, int c) {
  int d;
  asm("v_med3_i32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
  return d;
}
__device__ __forceinline__ unsigned med3_u(unsigned a, unsigned b, unsigned c) {
  unsigned d;
  asm("v_med3_u32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "v"(c));
  return d;
}

// Running state of a lane's pair on one side, over the lags the lane has seen:
// the extremum (exact) and the three best keys, largest first, with the lag
// blocks of the first two.  A key is a value's bits with the low four replaced
// by 15 - lag_order(r) of its register r, which orders equal values by lag and
// carries the lag along: inserting is one max and two med3 per value,
// with the block noted once per 16 values.  The positive side compares bits as
// signed integers (non-negative floats in order, negative ones below), the
// negative side as unsigned ones (the most negative first, positive ones
// last).  A key differs from its value by less than 16 units in the last place,
// at most kKeySlack for |value| <= 1.  The best key's lag is the extremum's unless
// another key differs from it in the lag bits alone; such a pair is a near tie, which
// FP64 settles, and one beyond the record capacity is searched again (seek_lags).
constexpr float kKeySlack = 2e-6f;
template <typename T>
struct Best3 {
  T e, k1, k2, k3;
  int b1, b2;
};
__device__ __forceinline__ int top(int a, int b) { return a > b ? a : b; }
__device__ __forceinline__ unsigned top(unsigned a, unsigned b) { return a > b ? a : b; }
__device__ __forceinline__ int mid(int a, int b, int c) { return med3_i(a, b, c); }
__device__ __forceinline__ unsigned mid(unsigned a, unsigned b, unsigned c) { return med3_u(a, b, c); }

template <typename T>
__device__ __forceinline__ void insert16(Best3<T>& s, const T (&bits)[16], const T (&key)[16], int block) {
  const T o1 = s.k1, o2 = s.k2;
#pragma unroll
  for (int r = 0; r < 16; r += 2) s.e = top(top(s.e, bits[r]), bits[r + 1]);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    s.k3 = mid(s.k2, s.k3, key[r]);
    s.k2 = mid(s.k1, s.k2, key[r]);
    s.k1 = top(s.k1, key[r]);
  }
  const bool c1 = s.k1 != o1;
  s.b2 = s.k2 == o2 ? s.b2 : ((c1 && s.k2 == o1) ? s.b1 : block);
  s.b1 = c1 ? block : s.b1;
}

// A pair's state on one side with the keys in one (signed) order and the lags
// as offsets from the first: what lanes and waves merge.
struct Side {
  int e, k1, k2, k3, o1, o2;
};
__device__ __forceinline__ int key_row(int key, int h) { return order_lag(h, 15 - (key & 15)); }
__device__ __forceinline__ Side side_of(const Best3<int>& s, int h) {
  return Side{s.e, s.k1, s.k2, s.k3, 32 * s.b1 + key_row(s.k1, h), 32 * s.b2 + key_row(s.k2, h)};
}
__device__ __forceinline__ Side side_of(const Best3<unsigned>& s, int h) {
  constexpr unsigned f = 0x80000000u;  // unsigned order to signed order
  return Side{(int)(s.e ^ f), (int)(s.k1 ^ f), (int)(s.k2 ^ f), (int)(s.k3 ^ f),
              32 * s.b1 + key_row((int)s.k1, h), 32 * s.b2 + key_row((int)s.k2, h)};
}
// Merge of two lists over disjoint lags; equal first keys go to the smaller lag.
__device__ __forceinline__ void merge_side(Side& a, const Side& b) {
  a.e = top(a.e, b.e);
  const bool tb = b.k1 > a.k1 || (b.k1 == a.k1 && b.o1 < a.o1);
  // W: the list whose head wins, O: the other
  const int w1 = tb ? b.k1 : a.k1, w2 = tb ? b.k2 : a.k2, w3 = tb ? b.k3 : a.k3;
  const int lw1 = tb ? b.o1 : a.o1, lw2 = tb ? b.o2 : a.o2;
  const int v1 = tb ? a.k1 : b.k1, v2 = tb ? a.k2 : b.k2, lv1 = tb ? a.o1 : b.o1;
  const bool v_second = v1 > w2;
  a.k1 = w1;
  a.o1 = lw1;
  a.k2 = v_second ? v1 : w2;
  a.o2 = v_second ? lv1 : lw2;
  a.k3 = v_second ? top(w2, v2) : top(w3, v1);
}
__device__ __forceinline__ Side shfl_side(const Side& s, int mask) {
  return Side{__shfl_xor(s.e, mask, 64),  __shfl_xor(s.k1, mask, 64), __shfl_xor(s.k2, mask, 64),
              __shfl_xor(s.k3, mask, 64), __shfl_xor(s.o1, mask, 64), __shfl_xor(s.o2, mask, 64)};
}

template <bool BF16X3>
struct Operand {
  u32x4 hi;
};
template <>
struct Operand<true> {
  u32x4 hi, lo;
};
template <bool BF16X3>
struct PlaneRows {
  __amdgpu_buffer_rsrc_t hi, lo;
  __device__ __forceinline__ Operand<BF16X3> load(int voff, int soff) const {
    Operand<BF16X3> o;
    o.hi = plane_load(hi, voff, soff);
    if constexpr (BF16X3) o.lo = plane_load(lo, voff, soff);
    return o;
  }
};

// Steps the operands of a range are loaded ahead: a step's products take
// 32 NI NBX cycles (three times that for bf16x3) and the SIMD's other wave as
// much, and about 800 cycles cover a load from L2.  RS ring entries and DB
// column operands (a divisor of RS, so that both are addressed at compile time
// in a turn of RS steps) give RS - NBX and DB - 1 steps.
template <bool BF16X3, int NI, int NBX>
struct Depth {
  static constexpr int kSteps = 12 / (NI * NBX * (BF16X3 ? 3 : 1));
  static constexpr int kAhead = kSteps < 2 ? 2 : (kSteps > 6 ? 6 : kSteps);
  static constexpr int pick() {  // the DB with the shortest ring
    int best = kAhead + 1;
    for (int d = kAhead + 1; d <= kAhead + 3; ++d)
      if (ring(d) < ring(best)) best = d;
    return best;
  }
  static constexpr int ring(int d) { return (NBX + kAhead + d - 1) / d * d; }
  static constexpr int DB = pick(), RS = ring(DB);
};

// The products of NBX lag blocks from block b0 on, for NI row events, into
// acc[ni * NB + b]: every channel, the 16-sample chunks [t0, t1) in two passes
// (even, then odd ones): within a pass the lag blocks' A operands are
// consecutive ring entries.
template <bool BF16X3, int NI, int NB, int NBX>
__device__ __forceinline__ void lag_range(f32x16 (&acc)[NI * NB], const PlaneRows<BF16X3> (&rows)[NI],
                                          const PlaneRows<BF16X3>& cols, int vh, int vb, const LagPairArgs& a, int b0,
                                          int t0, int t1) {
  constexpr int DB = Depth<BF16X3, NI, NBX>::DB, RS = Depth<BF16X3, NI, NBX>::RS;
  // loads at the last step: DB - 1 steps (of 1024 elements) on, and RS - 1 ring entries (of 32)
  static_assert(1024 * (DB - 1) <= kLagAhead && 32 * (RS - NBX) <= kLagAhead, "allocated past the operands");
#pragma unroll
  for (int u = 0; u < NI * NB; ++u) acc[u] = f32x16{};
  for (int c = 0; c < a.n_channels; ++c)
    for (int p = 0; p < 2; ++p) {
      const int t = t0 + ((p - t0) & 1);  // even and odd by the chunk's number: the order does not depend on t0
      const int steps = (t1 - t + 1) >> 1;
      if (steps <= 0) continue;  // traces of at most 16 samples have no odd chunk
      int hb = 4 * c * a.hs + 32 * t + 64 * b0;  // bytes: a row is two copies of hs elements
      int bb = 1024 * (c * (a.l16 / 16) + t);
      Operand<BF16X3> ring[NI][RS], col[DB];
#pragma unroll
      for (int v = 0; v < DB - 1; ++v) col[v] = cols.load(vb, bb + 2048 * v);
#pragma unroll
      for (int u = 0; u < RS - 1; ++u)
#pragma unroll
        for (int i = 0; i < NI; ++i) ring[i][u] = rows[i].load(vh + 64 * u, hb);
      for (int s = 0; s < steps; s += RS, hb += 64 * RS, bb += 2048 * RS) {
#pragma unroll
        for (int q = 0; q < RS; ++q) {
          if (s + q >= steps) break;
          col[(q + DB - 1) % DB] = cols.load(vb, bb + 2048 * (q + DB - 1));
#pragma unroll
          for (int i = 0; i < NI; ++i) ring[i][(q + RS - 1) % RS] = rows[i].load(vh + 64 * (q + RS - 1), hb);
          const Operand<BF16X3>& B = col[q % DB];
          // the three products block by block, so that products into one
          // accumulator are NI * NBX apart
          if constexpr (BF16X3) {
            const bf16x8 b_h = __builtin_bit_cast(bf16x8, B.hi), b_l = __builtin_bit_cast(bf16x8, B.lo);
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
              for (int b = 0; b < NBX; ++b)
                acc[i * NB + b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(bf16x8, ring[i][(q + b) % RS].lo), b_h, acc[i * NB + b], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
              for (int b = 0; b < NBX; ++b)
                acc[i * NB + b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(bf16x8, ring[i][(q + b) % RS].hi), b_l, acc[i * NB + b], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
              for (int b = 0; b < NBX; ++b)
                acc[i * NB + b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(bf16x8, ring[i][(q + b) % RS].hi), b_h, acc[i * NB + b], 0, 0, 0);
          } else {
            const f16x8 b_h = __builtin_bit_cast(f16x8, B.hi);
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
              for (int b = 0; b < NBX; ++b)
                acc[i * NB + b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                    __builtin_bit_cast(f16x8, ring[i][(q + b) % RS].hi), b_h, acc[i * NB + b], 0, 0, 0);
          }
        }
      }
    }
}

// A range's values into the pair's state, block by block in increasing lag order.
template <int NI, int NB, int NBX>
__device__ __forceinline__ void scan_range(f32x16 (&acc)[NI * NB], int ni, Best3<int>& pos, Best3<unsigned>& neg,
                                           const LagPairArgs& a, int b0, int h) {
#pragma unroll
  for (int b = 0; b < NBX; ++b) {
    f32x16 v = acc[ni * NB + b];
    if (b == NBX - 1 && b0 + NBX == a.n_blocks) {  // lags beyond the window's last
      const int last = a.lag_hi - a.lag_first - 32 * (b0 + b);
#pragma unroll
      for (int r = 0; r < 16; ++r) v[r] = lag_in_block(h, r) <= last ? v[r] : 0.f;
    }
    int bits[16], key[16];
    unsigned ubits[16], ukey[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      bits[r] = __float_as_int(v[r]);
      key[r] = (bits[r] & ~15) | (15 - lag_order(r));
      ubits[r] = (unsigned)bits[r];
      ukey[r] = (unsigned)key[r];
    }
    insert16(pos, bits, key, b0 + b);
    insert16(neg, ubits, ukey, b0 + b);
  }
}

template <bool BF16X3>
__device__ __forceinline__ PlaneRows<BF16X3> row_operand(const LagPairArgs& a, int i) {
  const long long o = (long long)min(i, a.n_events - 1) * a.n_channels * 2 * a.hs;
  PlaneRows<BF16X3> r;
  r.hi = plane_rsrc(a.h_hi + o, 2ll * a.n_channels * a.hs);
  if constexpr (BF16X3) r.lo = plane_rsrc(a.h_lo + o, 2ll * a.n_channels * a.hs);
  return r;
}
template <bool BF16X3>
__device__ __forceinline__ PlaneRows<BF16X3> column_operand(const LagPairArgs& a, int j0) {
  const long long o = (long long)(j0 / 32) * a.n_channels * a.l16 * 32;
  PlaneRows<BF16X3> c;
  c.hi = plane_rsrc(a.b_hi + o, 32ll * a.n_channels * a.l16);
  if constexpr (BF16X3) c.lo = plane_rsrc(a.b_lo + o, 32ll * a.n_channels * a.l16);
  return c;
}
// Lane offsets in bytes: A row r starts lag(r) samples in, at an even element of the
// copy of its parity; B column r of the chunk's two groups of 8 samples.
__device__ __forceinline__ int row_offset(const LagPairArgs& a, int lane) {
  const int r = lane & 31;
  return 2 * ((r >> 4) * a.hs + 8 * (lane >> 5) + 2 * (r & 15));
}
__device__ __forceinline__ int column_offset(int lane) { return 16 * lane; }

// First lags at which this row has the values p and n, block by block (the bits are
// those of the ranges, whose products differ by zeros alone).  Every lane takes its
// column's values.  Values past the window's last lag come after the first.
template <bool BF16X3>
__device__ __forceinline__ void seek_lags(const LagPairArgs& a, int i, int j0, int lane, float p, float n, int& fp,
                                          int& fn) {
  const int h = lane >> 5;
  const PlaneRows<BF16X3> rows[1] = {row_operand<BF16X3>(a, i)}, cols = column_operand<BF16X3>(a, j0);
  const int vh = row_offset(a, lane), vb = column_offset(lane);
  int lp = a.lag_hi, ln = a.lag_hi;
  for (int b = a.n_blocks - 1; b >= 0; --b) {
    const int l0 = a.lag_first + 32 * b, l1 = min(l0 + 31, a.lag_hi);
    f32x16 acc[1];
    lag_range<BF16X3, 1, 1, 1>(acc, rows, cols, vh, vb, a, b, max(0, -l1) >> 4, (min(a.L, a.L - l0) + 15) >> 4);
#pragma unroll
    for (int o = 15; o >= 0; --o) {
      const float v = acc[0][(o >> 1) + 8 * (o & 1)];
      const int lag = l0 + order_lag(h, o);
      lp = v == p ? lag : lp;
      ln = v == n ? lag : ln;
    }
  }
  fp = min(lp, __shfl_xor(lp, 32, 64));
  fn = min(ln, __shfl_xor(ln, 32, 64));
}

constexpr int kLagWaves = 8;  // per workgroup, two per SIMD
struct LagMerge {
  int v[kLagWaves][12][64];
};

// Bound by the matrix cores at the clock the power limit leaves: 0.82-0.86 busy
// at 1.6-1.8 GHz, 1.6 PFLOP/s of bf16 and 1.3 of fp16 issued (a 16384-cubed
// library matmul reaches 1.31 and 1.25 on the same card); deeper or shallower
// operand rings, one to three steps ahead, change it by less than 1%.  The tile kernel
// (xc_lag_tile.hip: 32 x 32 pairs at one lag, 24-sample column windows
// shifted into 16 operands per step, 3-4 vector instructions per product, one
// wave per SIMD, every lag over all samples) takes N = 1500, C = 3,
// L = 2048, +-512 bf16x3 32.1 ms against 25.3 here, N = 2001, L = 4096, +-512 fp16
// 17.2 against 12.7, and N = 40..491 up to 16 times as long: its unit of work is
// a whole 32 x 32 tile.  Windows of one or two blocks are bound by the operand loads,
// which take the CU's load path about 22 cycles each: N = 2000, C = 3, L = 4096, +-20
// bf16x3 7.48 ms, 0.8 of the rate above (the tile kernel 5.9).
//
// One workgroup per (tile of 32 columns, group of rows of the tile's 32).  Its
// waves take NI consecutive rows each; when a job has too few rows to fill the
// chip (split > 1), `split` waves share a row's lag ranges and merge in LDS.
// Ranges are NB or NB - 1 blocks, a.n_long of the former first.
template <bool BF16X3, int NI, int NB>
__global__ __launch_bounds__(64 * kLagWaves, 2) void k_lag_pairs(LagPairArgs a) {
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5, r32 = lane & 31;
  __shared__ LagMerge mg;
  const int split = a.split, part = wv % split;
  const int rows_per_wg = kLagWaves / split * NI, groups = 32 / rows_per_wg;
  const int n_items = a.n_tiles * groups;
  const int vh = row_offset(a, lane), vb = column_offset(lane);
  // XCD-aware walk: XCD blockIdx % 8 takes its own contiguous eighth of the
  // items, so the tiles of a row of tiles share their rows' operands in its L2
  const int n_xcd = (gridDim.x % 8 == 0) ? 8 : 1;
  const int xcd = blockIdx.x % n_xcd, local = blockIdx.x / n_xcd, n_local = gridDim.x / n_xcd;
  const int seg = (n_items + n_xcd - 1) / n_xcd, seg_end = min(n_items, (xcd + 1) * seg);
  for (int item = xcd * seg + local; item < seg_end; item += n_local) {
    const int2 t = a.tiles[item / groups];
    const int ib = 32 * (t.x + a.tile_row0) + item % groups * rows_per_wg, j0 = 32 * (t.y + a.tile_col0);
    if (ib >= a.n_events || j0 >= a.n_events) continue;  // ragged last block (workgroup-uniform)
    const int i0 = ib + wv / split * NI;  // this wave's first row
    const bool live = i0 < a.n_events;
    PlaneRows<BF16X3> rows[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) rows[i] = row_operand<BF16X3>(a, i0 + i);
    const PlaneRows<BF16X3> cols = column_operand<BF16X3>(a, j0);
    Best3<int> pos[NI];
    Best3<unsigned> neg[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      pos[i] = Best3<int>{0, 0, (int)0x80000000, (int)0x80000000, 0, 0};
      neg[i] = Best3<unsigned>{0x80000000u, 0x80000000u, 0u, 0u, 0, 0};
    }
    if (live)
      for (int rg = part; rg < a.n_ranges; rg += split) {
        const bool is_long = rg < a.n_long;
        const int b0 = is_long ? rg * NB : a.n_long * NB + (rg - a.n_long) * (NB - 1);
        const int nb = is_long ? NB : NB - 1;
        // samples k with 0 <= k < L and 0 <= k + l < L for some lag l of the range
        const int l0 = a.lag_first + 32 * b0, l1 = min(l0 + 32 * nb - 1, a.lag_hi);
        const int t0 = max(0, -l1) >> 4, t1 = (min(a.L, a.L - l0) + 15) >> 4;
        f32x16 acc[NI * NB];
        if (is_long) {
          lag_range<BF16X3, NI, NB, NB>(acc, rows, cols, vh, vb, a, b0, t0, t1);
#pragma unroll
          for (int i = 0; i < NI; ++i) scan_range<NI, NB, NB>(acc, i, pos[i], neg[i], a, b0, h);
        } else if constexpr (NB > 1) {
          lag_range<BF16X3, NI, NB, NB - 1>(acc, rows, cols, vh, vb, a, b0, t0, t1);
#pragma unroll
          for (int i = 0; i < NI; ++i) scan_range<NI, NB, NB - 1>(acc, i, pos[i], neg[i], a, b0, h);
        }
      }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      Side p = side_of(pos[i], h), n = side_of(neg[i], h);
      merge_side(p, shfl_side(p, 32));
      merge_side(n, shfl_side(n, 32));
      if (split > 1) {
        __syncthreads();  // the previous merge has been read
        const int w[12] = {p.e, p.k1, p.k2, p.k3, p.o1, p.o2, n.e, n.k1, n.k2, n.k3, n.o1, n.o2};
#pragma unroll
        for (int q = 0; q < 12; ++q) mg.v[wv][q][lane] = w[q];
        __syncthreads();
        if (part == 0)
          for (int o = 1; o < split; ++o) {
            int u[12];
#pragma unroll
            for (int q = 0; q < 12; ++q) u[q] = mg.v[wv + o][q][lane];
            merge_side(p, Side{u[0], u[1], u[2], u[3], u[4], u[5]});
            merge_side(n, Side{u[6], u[7], u[8], u[9], u[10], u[11]});
          }
      }
      const int ii = i0 + i, j = j0 + r32;
      const bool out = part == 0 && h == 0 && ii < a.n_events && j < a.n_events && j >= ii;
      // values in float: the negative side's magnitudes
      auto mag = [](int k) { return -__uint_as_float((unsigned)k ^ 0x80000000u); };
      const float p1 = __int_as_float(p.e), n1 = -mag(n.e);
      const bool kp = p1 > a.threshold && p1 > 0.f;
      const bool kn = n1 < -a.threshold && n1 < 0.f;
      const int glp1 = a.lag_first + p.o1, gln1 = a.lag_first + n.o1;
      const float tol = a.tie_tol + 2.f * kKeySlack;
      const float q1 = __int_as_float(p.k1), m1 = mag(n.k1);
      // near ties; wide ones (a third lag in the band): every in-window lag is a candidate
      const bool tp = out && kp && (q1 - __int_as_float(p.k2) < tol || q1 < tol);
      const bool tn = out && kn && (m1 - mag(n.k2) < tol || m1 < tol);
      const bool wp = tp && (q1 - __int_as_float(p.k3) < tol || q1 < tol);
      const bool wn = tn && (m1 - mag(n.k3) < tol || m1 < tol);
      if (out) {
        const long long idx = lag_out_index(a, ii, j);
        a.vpos[idx] = kp ? p1 : 0.f;
        a.lpos[idx] = kp ? glp1 : 0;
        a.vneg[idx] = kn ? n1 : 0.f;
        a.lneg[idx] = kn ? gln1 : 0;
      }
      const unsigned long long ties = __ballot(tp || tn);  // one counter update per wave
      if (ties) {
        unsigned base = 0;
        if (lane == 0) base = atomicAdd(a.tie_count, (unsigned)__popcll(ties));
        base = (unsigned)__builtin_amdgcn_readfirstlane((int)base);
        const unsigned slot = base + (unsigned)__popcll(ties & ((1ull << lane) - 1ull));
        if ((tp || tn) && slot < (unsigned)a.tie_cap) {
          a.ties[2 * slot] = make_int4(ii, j, (tp ? 1 : 0) | (tn ? 2 : 0) | (wp ? 4 : 0) | (wn ? 8 : 0), 0);
          a.ties[2 * slot + 1] = make_int4(glp1, a.lag_first + p.o2, gln1, a.lag_first + n.o2);
        }
        // beyond the capacity the extrema keep their own first lags
        const bool lost = (tp || tn) && slot >= (unsigned)a.tie_cap;
        if (__ballot(lost)) {
          int fp, fn;
          seek_lags<BF16X3>(a, ii, j0, lane, p1, n1, fp, fn);
          if (lost) {
            const long long idx = lag_out_index(a, ii, j);
            a.lpos[idx] = kp ? fp : 0;
            a.lneg[idx] = kn ? fn : 0;
          }
        }
      }
    }
  }
}

// ----------------------------------------------------------------------------
// FP64 resolver for the lag-window form: one wave per recorded pair
// ----------------------------------------------------------------------------

// FP64 sums sum_n ti[n] tj[n - lag_q] over the overlap of the two traces in
// [0, L), for NQ lags at once (callers repeat a lag to fill unused slots):
// each ti sample is read once for all of them, the loads of 8 steps of 64
// samples and all NQ lags are issued together before any is used (no
// per-lag branches; one memory round trip per 512 samples: fp16 resolver
// 6.1 -> 5.6 ms at 753k records), and two sets of partial sums per lane
// keep the FP64 FMA chains short.  The results are wave-uniform.
template <int NQ>
__device__ __forceinline__ void lin_corr_f64(const float* __restrict__ ti, const float* __restrict__ tj, int L,
                                             const int (&lag)[4], int lane, double (&out)[4]) {
  constexpr int U = 8;  // 64-sample steps per turn
  double sa[NQ], sb[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) sa[q] = sb[q] = 0.0;
  for (int n0 = lane; n0 < L; n0 += U * 64) {
    float av[U], bv[U][NQ];
    bool ok[U][NQ];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int n = n0 + 64 * k;
      const bool in = n < L;
      av[k] = ti[in ? n : 0];
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int u = n - lag[q];
        ok[k][q] = in && u >= 0 && u < L;
        bv[k][q] = tj[ok[k][q] ? u : 0];
      }
    }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const double a = (double)av[k];
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        double& acc = (k & 1) ? sb[q] : sa[q];
        acc += ok[k][q] ? a * (double)bv[k][q] : 0.0;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    double v = sa[q] + sb[q];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    out[q] = v;
  }
}

// Every lag of [lag_lo, lag_hi] at once, one lag per lane: FP64 sum of
// sg * c_ij(l) over channels (already normalised), and the wave's best by the
// reference scan rule (largest above 0, smallest lag on exact ties).  For the
// records whose third-best FP32 value is also inside the band, when the plan
// has no FFT period to hand them to (no supported P >= L + max |lag|).
__device__ __forceinline__ void sweep_window_f64(const LagResolveArgs& a, int i, int j, double sg, int lane,
                                                 double& best, int& best_lag, bool& have) {
  for (int l0 = a.lag_lo; l0 <= a.lag_hi; l0 += 64) {
    const int lag = l0 + lane;
    double acc = 0.0;
    for (int c = 0; c < a.n_channels; ++c) {
      const double ni = a.norms[(long long)i * a.n_channels + c], nj = a.norms[(long long)j * a.n_channels + c];
      if (!(ni > 0.0 && nj > 0.0)) continue;
      const float* ti = a.traces + ((long long)i * a.n_channels + c) * a.tr_stride;
      const float* tj = a.traces + ((long long)j * a.n_channels + c) * a.tr_stride;
      // sum_n ti[n] tj[n - lag] over 0 <= n < L, 0 <= n - lag < L
      double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
      auto term = [&](int n) -> double {
        const int u = n - lag;
        const bool ok = u >= 0 && u < a.L;
        const float b = tj[ok ? u : 0];
        return ok ? (double)ti[n] * (double)b : 0.0;
      };
      int n = 0;
      for (; n + 3 < a.L; n += 4) {
        s0 += term(n);
        s1 += term(n + 1);
        s2 += term(n + 2);
        s3 += term(n + 3);
      }
      for (; n < a.L; ++n) s0 += term(n);
      acc += ((s0 + s1) + (s2 + s3)) / (ni * nj * (double)a.n_channels);
    }
    acc *= sg;
    // wave argmax of this pass: larger value, then smaller lag
    double v = (lag <= a.lag_hi && acc > 0.0) ? acc : -1.0;
    int lg = lag;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const double ov = __shfl_xor(v, o, 64);
      const int ol = __shfl_xor(lg, o, 64);
      if (ov > v || (ov == v && ol < lg)) { v = ov; lg = ol; }
    }
    if (v > 0.0 && (!have || v > best)) {  // passes run in increasing lag order
      best = v;
      best_lag = lg;
      have = true;
    }
  }
}

__global__ __launch_bounds__(64) void k_lag_resolve(LagResolveArgs a) {
  const int lane = threadIdx.x;
  const unsigned total = min(*a.tie_count, (unsigned)a.tie_cap);
  // XCD-aware walk: XCD x = blockIdx % 8 resolves its own contiguous eighth
  // of the record list (records arrive roughly grouped by tile or row), so
  // the traces a record re-reads are usually still in that XCD's L2
  const unsigned n_xcd = (gridDim.x % 8 == 0) ? 8 : 1;
  const unsigned xcd = blockIdx.x % n_xcd, local = blockIdx.x / n_xcd, n_local = gridDim.x / n_xcd;
  const unsigned seg = (total + n_xcd - 1) / n_xcd;
  const unsigned rec0 = xcd * seg + local, seg_end = min(total, (xcd + 1) * seg);
  for (unsigned rec = rec0; rec < seg_end; rec += n_local) {
    const int4 t0 = a.ties[2 * rec], t1 = a.ties[2 * rec + 1];
    const int i = __builtin_amdgcn_readfirstlane(t0.x), j = __builtin_amdgcn_readfirstlane(t0.y);
    const int sides = __builtin_amdgcn_readfirstlane(t0.z);
    const long long idx = a.out_ld ? (long long)(i - a.out_row0) * a.out_ld + (j - a.out_col0)
                                   : (long long)i * a.n_events - (long long)i * (i - 1) / 2 + (j - i);
    // wide sides: any in-window lag may hold the FP64 winner; the FFT form's
    // resolver finds the candidates from the pair's FP32 transform
    const int wide_sides = (sides >> 2) & sides & 3;
    if (a.wide && wide_sides && lane == 0) {
      const unsigned slot = atomicAdd(a.wide_count, 1u);
      if (slot < (unsigned)a.wide_cap) a.wide[slot] = make_int4(i, j, wide_sides, 0);
    }
    // candidate lags of the sides resolved here (the two recorded ones per
    // side, in the window, without repeats), evaluated in one pass over the
    // traces per channel
    int lag[4] = {0, 0, 0, 0}, q_side[4] = {0, 0, 0, 0};
    int nq = 0;
    bool sweep[2] = {false, false};
    for (int sd = 0; sd < 2; ++sd) {
      if (!(sides & (1 << sd))) continue;
      if (sides & (4 << sd)) {
        sweep[sd] = !a.wide;  // else handed to the FFT form's resolver
        continue;
      }
      const int c0 = __builtin_amdgcn_readfirstlane(sd == 0 ? t1.x : t1.z);
      const int c1 = __builtin_amdgcn_readfirstlane(sd == 0 ? t1.y : t1.w);
      if (c0 >= a.lag_lo && c0 <= a.lag_hi) { lag[nq] = c0; q_side[nq] = sd; ++nq; }
      if (c1 != c0 && c1 >= a.lag_lo && c1 <= a.lag_hi) { lag[nq] = c1; q_side[nq] = sd; ++nq; }
    }
    for (int q = nq; q < 4; ++q) lag[q] = lag[0];  // unused slots repeat a lag
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (nq > 0) {
      for (int c = 0; c < a.n_channels; ++c) {
        const double ni = a.norms[(long long)i * a.n_channels + c], nj = a.norms[(long long)j * a.n_channels + c];
        if (!(ni > 0.0 && nj > 0.0)) continue;
        const float* ti = a.traces + ((long long)i * a.n_channels + c) * a.tr_stride;
        const float* tj = a.traces + ((long long)j * a.n_channels + c) * a.tr_stride;
        double sum[4] = {0.0, 0.0, 0.0, 0.0};
        // one side's two lags (the usual record) in a two-lag pass
        if (nq <= 2) lin_corr_f64<2>(ti, tj, a.L, lag, lane, sum);
        else lin_corr_f64<4>(ti, tj, a.L, lag, lane, sum);
        const double w = ni * nj * (double)a.n_channels;
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] += sum[q] / w;
      }
    }
    for (int sd = 0; sd < 2; ++sd) {
      if (!(sides & (1 << sd))) continue;
      if ((sides & (4 << sd)) && !sweep[sd]) continue;
      const double sg = sd == 0 ? 1.0 : -1.0;
      double best = 0.0;
      int best_lag = 0;
      bool have = false;
      if (sweep[sd]) {
        sweep_window_f64(a, i, j, sg, lane, best, best_lag, have);
      } else {
        // only the two recorded lags can hold the FP64 winner
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (q >= nq || q_side[q] != sd) continue;
          const double v = sg * acc[q];
          if (v > 0.0 && (!have || v > best || (v == best && lag[q] < best_lag))) {
            best = v;
            best_lag = lag[q];
            have = true;
          }
        }
      }
      if (lane == 0) {
        const float v = (float)best;
        if (sd == 0) {
          const bool keep = have && v > a.threshold;
          a.vpos[idx] = keep ? v : 0.f;
          a.lpos[idx] = keep ? best_lag : 0;
        } else {
          const bool keep = have && v > a.threshold;
          a.vneg[idx] = keep ? -v : 0.f;
          a.lneg[idx] = keep ? best_lag : 0;
        }
      }
    }
  }
}

// ----------------------------------------------------------------------------
// block output: FP32 / int32 -> float16 / int16 (round to nearest even)
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_pack_block(PackBlockArgs a) {
  const long long n = (long long)a.rows * a.cols;
  for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += (long long)gridDim.x * 256) {
    const int r = (int)(e / a.cols), c = (int)(e - (long long)r * a.cols);
    const bool below = a.mirror && c < r;
    const long long src = below ? (long long)c * a.in_ld + r : (long long)r * a.in_ld + c;
    const int lag = a.l[src];
    a.coef[e] = __builtin_bit_cast(unsigned short, (_Float16)a.v[src]);
    a.lag[e] = (short)(below ? -lag : lag);
  }
}

// ----------------------------------------------------------------------------
// launchers
// ----------------------------------------------------------------------------
hipError_t launch_lag_prep(const LagPrepArgs& a, hipStream_t st) {
  if (a.n_rows <= 0) return hipSuccess;
  const int events = a.n_rows / a.n_channels;
  const int rows = (events + 31) / 32 * 32 * a.n_channels;  // with the last column tile's empty ones
  if (a.energy_in)
    hipLaunchKernelGGL(k_lag_prep<Prep::kRows>, dim3(a.n_rows), dim3(256), 0, st, a);
  else if (a.p_hi)
    hipLaunchKernelGGL(k_lag_prep<Prep::kPlanes>, dim3(a.n_rows), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL(k_lag_prep<Prep::kOperands>, dim3(rows), dim3(256), 0, st, a);
  return hipGetLastError();
}

template <bool BF16X3, int NI, int NB>
static hipError_t launch_lag_pairs_k(const LagPairArgs& a, hipStream_t st) {
  const int items = a.n_tiles * (32 * a.split / (kLagWaves * NI));
  const int grid = items < (1 << 20) ? (items + 7) / 8 * 8 : 1 << 20;
  hipLaunchKernelGGL((k_lag_pairs<BF16X3, NI, NB>), dim3(grid), dim3(64 * kLagWaves), 0, st, a);
  return hipGetLastError();
}

template <bool BF16X3, int NB>
static hipError_t launch_lag_pairs_nb(int nb, const LagPairArgs& a, hipStream_t st) {
  if constexpr (NB > 1)
    if (nb < NB) return launch_lag_pairs_nb<BF16X3, NB - 1>(nb, a, st);
  // Few blocks make few products per operand load: two rows per wave then share
  // a column operand, where a job has rows enough (turns of the 256 CUs, a
  // two-row turn taking about 1.7 of the others').  N = 3000, L = 2048, one
  // channel, one row per wave -> two: bf16x3 +-10 2.27 -> 1.84 ms, +-20
  // 2.98 -> 2.64; fp16 +-50 2.68 -> 2.52, +-20 2.05 -> 2.04 (four rows 2.15), +-10
  // (one block) 1.94 -> 1.98.
  constexpr int NI = BF16X3 ? (NB <= 3 ? 2 : 1) : (NB >= 2 && NB <= 4 ? 2 : 1);
  if constexpr (NI > 1) {
    const long long wgs = 4ll * a.n_tiles;
    if (a.n_ranges == 1 && 17 * ((wgs / 2 + 255) / 256) <= 10 * ((wgs + 255) / 256))
      return launch_lag_pairs_k<BF16X3, NI, NB>(a, st);
  }
  return launch_lag_pairs_k<BF16X3, 1, NB>(a, st);
}

hipError_t launch_lag_pairs(bool bf16x3, LagPairArgs a, hipStream_t st) {
  if (a.n_tiles <= 0) return hipSuccess;
  // ranges of at most 7 (bf16x3) or 8 blocks (the registers of two waves per
  // SIMD), as even as possible
  const int most = bf16x3 ? 7 : 8;
  a.n_ranges = (a.n_blocks + most - 1) / most;
  const int nb = (a.n_blocks + a.n_ranges - 1) / a.n_ranges;
  a.n_long = a.n_blocks - a.n_ranges * (nb - 1);
  // Waves sharing a row's ranges: a workgroup of 8 takes 8 / split rows, so
  // the 256 CUs take ceil(4 split tiles / 256) turns of ceil(ranges / split)
  // ranges each; the split with the fewest (the smallest of equals) is taken.
  a.split = 1;
  long long best = 0;
  for (int sp = 1; sp <= kLagWaves && sp / 2 < a.n_ranges; sp *= 2) {
    const long long turns = ((long long)a.n_tiles * 4 * sp + 255) / 256 * ((a.n_ranges + sp - 1) / sp);
    if (sp == 1 || turns < best) {
      best = turns;
      a.split = sp;
    }
  }
  return bf16x3 ? launch_lag_pairs_nb<true, 7>(nb, a, st) : launch_lag_pairs_nb<false, 8>(nb, a, st);
}

hipError_t launch_pack_block(const PackBlockArgs& a, hipStream_t st) {
  const long long n = (long long)a.rows * a.cols;
  if (n <= 0) return hipSuccess;
  const long long g = (n + 255) / 256;
  hipLaunchKernelGGL(k_pack_block, dim3((unsigned)(g < 8192 ? g : 8192)), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_lag_resolve(const LagResolveArgs& a, int grid, hipStream_t st) {
  hipLaunchKernelGGL(k_lag_resolve, dim3(grid), dim3(64), 0, st, a);
  return hipGetLastError();
}

}  // namespace sxc
