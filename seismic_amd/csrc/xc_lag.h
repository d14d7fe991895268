// Argument blocks and launchers of the lag-window (MFMA) form.
#pragma once
#include <hip/hip_runtime.h>

namespace sxc {

constexpr int kLagBlock = 32;  // lags per block (one accumulator tile each)
// The widest window a plan takes, in whole blocks of kTileLags from tile_first_lag on (a
// limit of the interface: the product over lags needs none).
constexpr int kLagMaxSpan = 65536;

// Elements past a row's or a column tile's operand that the product's loads may
// reach (their values are not used).
constexpr int kLagAhead = 8192;
// Parts of the operands' allocation, in elements (256-byte aligned): row operands
// of `rows` rows, then column operands of `cols` rows (a multiple of 32 events),
// which with what follows them are the room past the row operands.
struct LagOperands {
  long long h, b;  // elements of each part
};
inline LagOperands lag_operands(long long rows, long long cols, int hs, int l16) {
  auto up = [](long long n) { return (n + 127) / 128 * 128; };
  return {up(rows * 2 * hs), up(cols * l16 + kLagAhead)};
}

// The kernel of tiles of 32 x 32 pairs at one lag (xc_lag_tile.hip) takes whole blocks of
// this many lags.
constexpr int kTileLags = 16;
// First lag of a plan's blocks there: 1 modulo 8, which aligns every window.
inline int tile_first_lag(int lag_lo) {
  int lf = lag_lo;
  while (((lf - 1) % 8 + 8) % 8 != 0) --lf;
  return lf;
}
// Whether a window runs there.  With one or two blocks of 32 lags the product over
// lags is bound by its operand loads where a pair's samples (of all channels) are
// many, and pads up to 31 lags; the tile kernel takes one tile per CU and turn, so a
// job must fill its turns.  N = 2000, product -> tiles: bf16x3, 33..47 lags, C = 3,
// L = 4096 7.48 -> 5.82 ms, L = 1500 2.72 -> 2.21, C = 1, L = 4096 2.46 -> 2.09, L = 1500
// 0.97 of it; 49..63 lags, C = 3, L = 4096 7.49 -> 6.63; 97..105 lags 13.3 -> 12.0; fp16, 1 lag,
// C = 3, L = 4096 4.57 -> 3.55, 3..31 lags 18% faster, 33..47 16%.  The gains below, of 100 where turns are
// full, are those measured at N = 2000 by the pair's samples (from 2500, 4000, 7000
// and 12000 on).  A rule on the plan alone: tiled runs give a plan's bits.
inline bool lag_tiles(bool bf16x3, int n_events, int n_channels, int trace_len, int lag_lo, int lag_hi) {
  const long long samples = (long long)n_channels * ((trace_len + 15) / 16 * 16), T = (n_events + 31LL) / 32;
  const long long tiles = T * (T + 1) / 2, lags = (long long)lag_hi - lag_lo + 1;
  const long long blocks = (lags + kLagBlock - 1) / kLagBlock;
  const long long tile_blocks = (lag_hi - (long long)tile_first_lag(lag_lo) + kTileLags) / kTileLags;
  if (samples < 2500 || tiles < 128 || tile_blocks > 7) return false;
  const int q = samples < 4000 ? 0 : (samples < 7000 ? 1 : (samples < 12000 ? 2 : 3));
  constexpr int x3_1[] = {0, 0, 3, 7}, x3_2a[] = {9, 18, 29, 29}, x3_2b[] = {0, 2, 10, 13}, x3_4[] = {0, 5, 12, 10};
  constexpr int f16_lag[] = {5, 9, 23, 29}, f16_1[] = {0, 5, 13, 19}, f16_2a[] = {0, 5, 10, 16}, f16_2b[] = {0, 0, 2, 5};
  const int* gain = nullptr;
  if (blocks == 1) gain = bf16x3 ? x3_1 : (lags == 1 ? f16_lag : f16_1);
  else if (blocks == 2 && tile_blocks == 3) gain = bf16x3 ? x3_2a : f16_2a;
  else if (blocks == 2 && tile_blocks == 4) gain = bf16x3 ? x3_2b : f16_2b;
  else if (blocks == 4 && tile_blocks == 7 && bf16x3) gain = x3_4;
  if (!gain) return false;
  // shares of the CUs' turns that do work: one tile per workgroup here; there four
  // workgroups per tile, or two (of 1.5 turns) where a wave takes two rows
  const bool two_rows = blocks <= (bf16x3 ? 3 : 4) && (bf16x3 || blocks > 1);
  auto turns = [](long long wgs) { return (double)((wgs + 255) / 256); };
  const double here = (double)tiles / (256.0 * turns(tiles)), one = turns(4 * tiles), two = 1.5 * turns(2 * tiles);
  const double there = (two_rows ? 1.5 * 2.0 : 4.0) * (double)tiles / 256.0 / (two_rows && two < one ? two : one);
  return (100 + gain[q]) * here >= 104.0 * there;
}

struct LagPrepArgs {
  const float* in;          // [n_rows][in_stride]
  long long in_stride;
  int in_len;               // samples present per row (zero beyond)
  int L;                    // trace length used
  int n_rows;
  int n_channels;
  int demean;
  int fp16;                 // 1: FP16 plane only; 0: bf16 hi and lo planes
  int lag_first;            // row operand: element q is sample q + lag_first
  int hs;                   // row operand length (a multiple of 8)
  int l16;                  // trace length rounded up to 16
  unsigned short* h_hi;     // [n_rows][2][hs], the second copy one sample on
  unsigned short* h_lo;     // or null (fp16)
  unsigned short* b_hi;     // column operand [event / 32][channel][sample / 8][event % 32][8]
  unsigned short* b_lo;     // or null
  // in their place, when set: zero-padded planes, sample n at element n + p0 of a row
  unsigned short *p_hi, *p_lo;  // [n_rows][ls]
  int p0, ls;
  unsigned* zero0;          // optional counters to clear
  unsigned* zero1;
  double* norms;            // [n_rows]
  double* energy;           // optional [n_rows]
  // Row operands alone, of traces demeaned before, with the energies an earlier
  // launch left.
  const double* energy_in;
  float* traces_out;        // [n_rows][L] FP32 copy (demeaned) for the FP64 resolver
};

struct LagPairArgs {
  const unsigned short *h_hi, *h_lo, *b_hi, *b_lo;  // operands (LagPrepArgs)
  int hs;
  int n_events, n_channels;
  int L, l16;               // trace length, and rounded up to 16
  int lag_hi;               // last scanned lag
  int lag_first;            // first scanned lag
  int n_blocks;             // blocks of kLagBlock lags
  int n_ranges, n_long, split;  // set by launch_lag_pairs
  // launch_lag_tiles: planes (LagPrepArgs), the first scanned lag and blocks of kTileLags
  // from lag_first on, which is at or before it
  const unsigned short *p_hi, *p_lo;
  long long ls;
  int p0, lag_lo;
  const int2* tiles;        // (row tile, column tile), column >= row
  int n_tiles;
  int tile_row0, tile_col0; // added to every tile entry (block runs)
  long long out_ld;         // 0: packed triangle output; else dense block with this row stride
  int out_row0, out_col0;   // event index of the block's first row / column
  float threshold, tie_tol;
  float* vpos;
  int* lpos;
  float* vneg;
  int* lneg;
  int4* ties;               // 2 int4 per record: (i, j, sides, 0), (lp1, lp2, ln1, ln2); sides bit 0/1:
                            // pos/neg near tie, bit 2/3: a third lag of that side is in the band too
  unsigned* tie_count;
  int tie_cap;
};

struct LagResolveArgs {
  const float* traces;      // [n_events * n_channels][tr_stride]
  long long tr_stride;
  const double* norms;
  int n_events, n_channels, L;
  int lag_lo, lag_hi;
  float threshold;
  const int4* ties;
  const unsigned* tie_count;
  int tie_cap;
  float* vpos;
  int* lpos;
  float* vneg;
  int* lneg;
  long long out_ld;         // as in LagPairArgs
  int out_row0, out_col0;
  // Sides whose band held a third lag ("wide") are appended to this list as
  // (i, j, sides, 0) for the FFT form's resolver when set; swept over the
  // whole window in FP64 here otherwise.  One entry per processed record at
  // most, so a list of tie_cap entries cannot overflow.
  int4* wide;
  unsigned* wide_count;
  int wide_cap;
};

// Place of pair (i, j) in the outputs.
__host__ __device__ __forceinline__ long long lag_out_index(const LagPairArgs& a, int i, int j) {
  return a.out_ld ? (long long)(i - a.out_row0) * a.out_ld + (j - a.out_col0)
                  : (long long)i * a.n_events - (long long)i * (i - 1) / 2 + (j - i);
}

// FP32 value / int32 lag block -> float16 coefficient / int16 lag block
struct PackBlockArgs {
  const float* v;
  const int* l;
  long long in_ld;
  int rows, cols;
  unsigned short* coef;     // float16 bits, [rows][cols]
  short* lag;
  int mirror;               // diagonal block: entries below the diagonal are the
                            // transposed ones above it, lag negated
};

hipError_t launch_lag_prep(const LagPrepArgs& a, hipStream_t st);
hipError_t launch_lag_pairs(bool bf16x3, LagPairArgs a, hipStream_t st);
hipError_t launch_lag_tiles(bool bf16x3, const LagPairArgs& a, hipStream_t st);
hipError_t launch_lag_resolve(const LagResolveArgs& a, int grid, hipStream_t st);
hipError_t launch_pack_block(const PackBlockArgs& a, hipStream_t st);

}  // namespace sxc
