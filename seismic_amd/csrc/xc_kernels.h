// Kernel argument blocks and launchers for the FP32-FFT form.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace sxc {

struct ForwardArgs {
  const float* in;        // [n_rows][in_stride] float32
  long long in_stride;
  int in_len;             // samples read per row (zero beyond)
  int L;                  // samples entering energy / mean
  int n_rows;             // events * channels
  int n_channels;         // C in scale = 1/sqrt(E*C*P)
  int demean;             // subtract the FP64 mean of the first L samples
  double* norms;          // [n_rows] sqrt(E) in FP64
  float* out_traces;      // optional [n_rows][out_stride] copy of the transformed samples (P per row)
  long long out_stride;
  float2* spec;           // [n_rows][spec_stride] bins 0..M
  long long spec_stride;
  const float2* tw;       // forward twiddle tables (TwLayout)
  const float2* post_tw;  // exp(-2 pi i k / P), k = 0..M
  const int* row_len;     // optional per-event sample counts (rows of one event share it);
                          // when set it replaces in_len and L for that row
  // Reversed-row mode (the reference's second R2C, Correlation_in_OMP/
  // correlation_c.cpp:43-45): the rows are the caller's reversed traces r_j.
  // The energy is not summed here; the scale comes from norms_in (the forward
  // rows' sqrt(E)), and the row is stored as the column spectrum
  // conj(rfft(r_j)[k] * exp(+2 pi i k rev_shift / P)) * scale, so that the
  // pair kernel's Xhat_i conj(col) is X_i R_j rotated by rev_shift = L - 1:
  // its lag-l slot then holds the reference's corr_t[L - 1 + l].
  int reversed;
  int rev_shift;
  const double* norms_in;
  unsigned* zero;         // optional: set to 0 (the near-tie counter of the execute this launch begins)
  // Segment mode (n_seg > 0): every row gives n_seg row spectra and n_seg
  // column spectra of the launch's period P.  Segment s is the samples
  // [s seg_len, (s + 1) seg_len) for the row side and, for the column side, those
  // and the seg_back before and seg_ahead after them, sample n at element
  // (n - s seg_len) mod P (seg_len + seg_back + seg_ahead <= P), all with the
  // whole row's mean and energy.  Row r's spectra: spec and seg_cols, from row
  // r n_seg on.  out_traces takes the row side's samples.
  int n_seg, seg_len, seg_back, seg_ahead;
  float2* seg_cols;
  int seg_sides;          // 0: both sides' spectra, 1: the row side's only (with norms and out_traces), 2: the column side's
};

// Bound of the FP32 rounding of a coefficient (at most 1) that is exactly 0.
constexpr float kScanNoise = 5e-7f;

struct PairArgs {
  const float2* spec;     // row spectra [n_rows][n_channels][spec_stride]
  long long spec_stride;
  const float2* col_spec; // column spectra (null: the row spectra, all-pairs mode)
  int n_events;           // all-pairs: events; rectangular: columns
  int dense_cols;         // 0: packed upper triangle; > 0: out[i * dense_cols + j], all (i, j)
  int pos_only;           // 1: write only vpos / lpos
  int n_channels;
  const int2* work;       // (row i, first column) per work item; null (rectangular mode): item e is row
                          // e % n_rows and column chunk e / n_rows
  int n_work;
  int n_rows;             // rectangular mode without a work list: rows
  int chunk;              // columns per work item
  int n_lds;              // set by launch_pairs: channels of the row held in LDS when not all fit
  int lag_lo, lag_hi;     // scanned lags, inclusive
  float threshold;
  float tie_tol;
  const float2* tw;       // inverse twiddle tables (TwLayoutCT)
  float* vpos;
  int* lpos;
  float* vneg;
  int* lneg;
  int4* ties;             // (i, j, sides, 0)
  unsigned* tie_count;
  int tie_cap;
};

struct ResolveArgs {
  const float2* spec;
  long long spec_stride;
  const float2* col_spec; // column spectra (null: spec); reversed-row mode when rev_traces is set
  const float* rev_traces;// reversed-row mode: [n_events * n_channels][rev_stride] r_j, zero beyond rev_len;
                          // the lag-l value is sum_m x_i[m] r_j[(l + rev_shift - m) mod P]
  long long rev_stride;
  int rev_len;
  int rev_shift;
  int n_spec;             // spectra of an event: n_channels, or as many per segment
  int period;             // of the FP64 sums: lags are circular mod this
  int n_events;
  int n_channels;
  const double* norms;    // [n_events * n_channels]
  const float* traces;    // [n_events * n_channels][tr_stride], zero beyond tr_len
  long long tr_stride;
  int tr_len;
  int lag_lo, lag_hi;
  float threshold;
  float tie_tol;
  const float2* tw;
  float* vpos;
  int* lpos;
  float* vneg;
  int* lneg;
  const int4* ties;
  const unsigned* tie_count;
  const unsigned* tie_begin;  // null: records from 0; else from *tie_begin (launch groups of a blocked call)
  int tie_cap;
  long long out_ld;       // 0: packed triangle output; else dense block rows of this stride
  int out_row0, out_col0; // event index of the block's first row / column
};

// Per-R launchers, one translation unit per R (xc_kernels.hip with -DSXC_R).
template <int R> hipError_t launch_forward_r(const ForwardArgs& a, hipStream_t st);
template <int R> hipError_t launch_pairs_r(bool full, const PairArgs& a, int grid, hipStream_t st);
template <int R> hipError_t launch_resolve_r(const ResolveArgs& a, int grid, hipStream_t st);

// Runtime dispatch over R (xc_dispatch.cpp).
hipError_t launch_forward(int R, const ForwardArgs& a, hipStream_t st);
hipError_t launch_pairs(int R, bool full, const PairArgs& a, int grid, hipStream_t st);
hipError_t launch_resolve(int R, const ResolveArgs& a, int grid, hipStream_t st);
hipError_t launch_fill_u32(unsigned* p, unsigned v, int n, hipStream_t st);
hipError_t launch_copy_f4(float4* dst, const float4* src, long long n, hipStream_t st);
// top-k of each row of a dense [n_rows][n_cols] score matrix, by value
// (descending; equal values by smaller column); rows with fewer than k
// columns pad with (-inf, 0, -1).
hipError_t launch_topk(const float* v, const int* l, int n_rows, int n_cols, int k, float* out_v,
                       int* out_l, int* out_idx, hipStream_t st);
// The same result in two passes for few rows: each row's columns in
// n_slices slices (one workgroup each) into tmp [n_rows][n_slices * k]
// (value, lag, column), then the top-k of those candidates per row.
constexpr int kTopkMaxSlices = 16;
hipError_t launch_topk_split(const float* v, const int* l, int n_rows, int n_cols, int k, int n_slices,
                             float* tmp_v, int* tmp_l, int* tmp_idx, float* out_v, int* out_l, int* out_idx,
                             hipStream_t st);

// Histograms and threshold over packed results computed without a threshold
// (the OMP ABI's histograms count every pair before its threshold).
struct HistArgs {
  float* vpos;
  int* lpos;
  float* vneg;
  int* lneg;
  long long n;            // packed pairs
  int n_classes;
  float delta;            // float(1.0 / n_classes)
  float threshold;
  int* hist_pos;          // [n_classes], accumulated with atomics
  int* hist_neg;
};
hipError_t launch_hist_threshold(const HistArgs& a, hipStream_t st);

// compact twiddle tables + staged row spectra + one transpose buffer per wave
constexpr size_t kLdsBytes = 160 * 1024;  // of a CU
constexpr size_t pair_lds_bytes(int R, int n_channels, int waves) {
  return (size_t)(640 + 8 * R + n_channels * (64 * R + 1) + waves * 576) * 8;
}

// Workgroup shapes of a period in order of preference: W waves, S waves per
// SIMD in all, so 4 S / W workgroups share a CU and its 160 KiB of LDS (tables,
// staged rows and one buffer per wave each).  The first that fits the job's
// channels is used.  Compact twiddle tables throughout (fewer LDS reads per
// pair for a few more multiplies: measured 1-1.3% faster at P <= 4096, 22% at
// P = 6144).
//   S: as many waves as the registers allow without spilling the transform
//   (P = 2048 at S = 6 spills 32 bytes per lane and still gains): short
//   transforms wait on LDS and memory more than they issue.
//   W: several small workgroups per CU rather than one of 16 waves, so that one
//   computes while another waits at the barrier that restages its row.
// N = 1500, full lags, one 16-wave workgroup -> the shape below: P = 1024,
// C = 1..4: 1.07 -> 0.80, 1.25 -> 0.95, 1.46 -> 1.15, 1.70 -> 1.42 ms; P = 2048:
// 1.71 -> 1.46, 2.02 -> 1.77, 2.41 -> 2.21, 2.89 -> 2.70; P = 3072, C = 1..3:
// 2.52 -> 2.29, 3.00 -> 2.74, 3.51 -> 3.40; P = 4096, C = 1, 2: 3.24 -> 2.95,
// 3.97 -> 3.90; one 12-wave workgroup -> 3 of 4: P = 5120, C = 1 4.26 -> 4.20,
// P = 6144 5.11 -> 5.00.  W is a multiple of 4: 6, 10 or 14 waves load the four
// SIMDs unevenly and the next workgroup no longer fits (P = 1024 with 14: 1.12).
// P = 8192 runs 8 waves per CU: its 128 spectrum registers per lane need 256 VGPRs;
// two workgroups of 4 where one channel leaves the LDS for them: N = 1500, C = 1
// 7.14 -> 6.83 ms, +-2730 8.55 -> 7.79, N = 200 233 -> 221 us.
struct PairShape {
  int waves, per_simd;  // W, S; 0: no further shape
};
constexpr PairShape pair_shape(int R, int i) {
  constexpr PairShape k8[] = {{8, 6}, {12, 6}, {8, 4}, {0, 0}, {0, 0}};
  constexpr PairShape k16[] = {{8, 6}, {12, 6}, {8, 4}, {16, 4}, {0, 0}};
  constexpr PairShape k24[] = {{8, 4}, {16, 4}, {12, 3}, {0, 0}, {0, 0}};
  constexpr PairShape k32[] = {{8, 4}, {16, 4}, {12, 3}, {8, 2}, {0, 0}};
  constexpr PairShape k48[] = {{4, 3}, {12, 3}, {8, 2}, {0, 0}, {0, 0}};  // and R = 40
  constexpr PairShape k64[] = {{4, 2}, {8, 2}, {0, 0}, {0, 0}, {0, 0}};
  return R == 8 ? k8[i] : R == 16 ? k16[i] : R == 24 ? k24[i] : R == 32 ? k32[i] : R == 64 ? k64[i] : k48[i];
}
constexpr bool pair_shape_fits(int R, int n_channels, PairShape k) {
  return (size_t)(4 * k.per_simd / k.waves) * pair_lds_bytes(R, n_channels, k.waves) <= kLdsBytes;
}
// The last shape serves the rest too, with as many channels in LDS as it holds
// (with all of them read from memory by every wave, the row's spectra doubled
// the traffic from L2 that bounds such jobs: N = 1500, P = 4096, C = 8 27.6 -> 12.0
// ms, P = 6144, C = 5 20.0 -> 12.0, P = 8192, C = 4 24.9 -> 14.3, C = 8 56 -> 33).
inline PairShape pair_shape_for(int R, int n_channels) {
  int i = 0;
  while (!pair_shape_fits(R, n_channels, pair_shape(R, i)) && pair_shape(R, i + 1).waves > 0) ++i;
  return pair_shape(R, i);
}

// Measured time of the pair kernel at period 128 R with 1 .. 8 channels (ms,
// N = 1500; the mean of the full lag range and +-P/5): what the choice between
// periods compares.
inline double pair_cost(int R, int n_channels) {
  struct Row { int R; double ms[8]; };
  static constexpr Row rows[] = {{8, {0.90, 1.04, 1.26, 1.49, 1.75, 2.15, 2.44, 2.72}},
                                 {16, {1.56, 1.90, 2.27, 2.66, 3.41, 4.03, 4.64, 5.17}},
                                 {24, {2.34, 2.81, 3.35, 4.30, 5.20, 6.11, 6.87, 7.73}},
                                 {32, {3.08, 3.72, 4.72, 5.60, 6.72, 8.40, 9.08, 11.9}},
                                 {40, {4.26, 5.09, 6.06, 7.25, 8.80, 11.4, 14.4, 17.4}},
                                 {48, {4.81, 5.97, 7.09, 8.47, 12.0, 15.6, 18.9, 22.5}},
                                 {64, {7.46, 9.09, 11.2, 14.3, 18.8, 23.7, 28.3, 33.1}}};
  for (const Row& r : rows)
    if (r.R == R) return r.ms[n_channels - 1];
  return 0.0;
}

// Columns per work item: 64 keep one chunk's column spectra in an XCD's L2 over
// its rows, but a small job is then a few workgroups of many serial pairs.  A
// wave's share of the job, in pairs, is about the workgroups' turns on the
// 256 CUs times the columns of an item each wave takes, plus half a pair per
// turn for staging the row; the chunk with the smallest is taken, a smaller one
// only for a gain of 3%.  items(c): work items with chunks of c columns.
// With 64 columns always -> this rule (and the shapes above): N = 200, C = 3,
// P = 2048, +-100 137 -> 102 us; N = 64, C = 3, P = 4096 123 -> 82; one 4096-sample
// query against 4096 x 3 x 2048 catalog events (P = 5120) 99 -> 48 in the pair
// kernel.
template <typename Items>
inline int pair_chunk(int R, int n_channels, Items items) {
  const PairShape k = pair_shape_for(R, n_channels);
  const long long slots = 256 * 4 * k.per_simd / k.waves;
  int best = 64;  // 4 columns only ever pay for workgroups of 4 waves
  double cost = 0.0;
  for (int c : {64, 32, 16, 8, 4}) {
    const double t = (double)((items(c) + slots - 1) / slots) * ((c + k.waves - 1) / k.waves + 0.5);
    if (c == 64 || t < 0.97 * cost) {
      best = c;
      cost = t;
    }
  }
  return best;
}
// Work items (row, column chunk) of the packed triangle, chunk-major: chunk c
// holds min(N, chunk (c + 1)) rows.
inline long long triangle_items(long long n, long long chunk) {
  const long long q = n / chunk, r = n % chunk;
  return chunk * (q * (q + 1) / 2) + (r ? n : 0);
}
// Workgroups of a pair launch: a multiple of 8 (one share per XCD).
inline int pair_grid(int n_work) { return n_work >= 4096 ? 4096 : (n_work + 7) / 8 * 8; }
// Workgroups of a resolver launch over the records of up to n_pairs pairs: one
// wave each, 8192 at most; a small job's grid is kept small, since a launch of
// 8192 that find no record takes 17 us.
inline int resolve_grid(long long n_pairs) {
  const long long few = n_pairs < 256 ? n_pairs : 256, g = n_pairs / 8 > few ? n_pairs / 8 : few;
  return (int)(g >= 8192 ? 8192 : (g + 7) / 8 * 8);
}

}  // namespace sxc
