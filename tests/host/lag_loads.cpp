// Every buffer load of the lag-window product, lane by lane on the CPU: inside
// the operands' allocation, whatever the hardware's range check does with the
// scalar offset.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdio.h>
#include <vector>

using ::max;
using ::min;
#include "../../seismic_amd/csrc/xc_lag.hip"

static long g_bad = 0, g_loads = 0;
static long long g_begin, g_end;  // the operands' allocation, as addresses
void on_buffer_load(const BufferRsrc& r, int voff, int soff, int bytes) {
  ++g_loads;
  const long long first = (long long)r.base + voff + soff, last = first + bytes;
  if (voff < 0 || soff < 0 || first < g_begin || last > g_end) ++g_bad;
}

using namespace sxc;

// The loads of a range for the last row event and the last column tile of n events.
template <bool X3, int NI, int NB, int NBX>
static void range(const LagPairArgs& a, int b0) {
  const int l0 = a.lag_first + 32 * b0, l1 = min(l0 + 32 * NBX - 1, a.lag_hi);
  const int t0 = max(0, -l1) >> 4, t1 = (min(a.L, a.L - l0) + 15) >> 4;
  const long long row = (a.n_events - 1) * 2ll * a.n_channels * a.hs;
  const long long tile = (a.n_events - 1) / 32 * 32ll * a.n_channels * a.l16;
  PlaneRows<X3> rows[NI], cols;
  for (int i = 0; i < NI; ++i) {
    rows[i].hi = plane_rsrc(a.h_hi + row, 2ll * a.n_channels * a.hs);
    if constexpr (X3) rows[i].lo = plane_rsrc(a.h_lo + row, 2ll * a.n_channels * a.hs);
  }
  cols.hi = plane_rsrc(a.b_hi + tile, 32ll * a.n_channels * a.l16);
  if constexpr (X3) cols.lo = plane_rsrc(a.b_lo + tile, 32ll * a.n_channels * a.l16);
  for (int lane = 0; lane < 64; ++lane) {
    const int h = lane >> 5, r32 = lane & 31;
    const int vh = 2 * ((r32 >> 4) * a.hs + 8 * h + 2 * (r32 & 15)), vb = 16 * (32 * h + r32);
    f32x16 acc[NI * NB];
    lag_range<X3, NI, NB, NBX>(acc, rows, cols, vh, vb, a, b0, t0, t1);
  }
}

template <bool X3, int NB>
static void ranges(LagPairArgs a, int nb) {
  if constexpr (NB > 1)
    if (nb < NB) return ranges<X3, NB - 1>(a, nb);
  for (int rg = 0; rg < a.n_ranges; ++rg) {
    const bool is_long = rg < a.n_long;
    const int b0 = is_long ? rg * NB : a.n_long * NB + (rg - a.n_long) * (NB - 1);
    if (is_long) {
      range<X3, 1, NB, NB>(a, b0);
      range<X3, 2, NB, NB>(a, b0);
    } else if constexpr (NB > 1) {
      range<X3, 1, NB, NB - 1>(a, b0);
    }
  }
}

int main() {
  const int lens[] = {1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 100, 257, 513};
  int cases = 0;
  for (int L : lens)
    for (int C : {1, 3})
      for (int lo : {-(L - 1), -L / 2, -1, 0, L / 3, L - 1})
        for (int hi : {-(L - 1), -L / 2, 0, 1, L / 3, L - 1}) {
          if (lo > hi || lo <= -L || hi >= L) continue;
          for (bool x3 : {false, true}) {
            // the operands' layout, as a plan of one tile has it
            LagPairArgs a{};
            a.n_events = 32;
            a.n_channels = C;
            a.L = L;
            a.l16 = (L + 15) / 16 * 16;
            a.lag_first = lo;
            a.lag_hi = hi;
            a.n_blocks = (hi - lo + 1 + kLagBlock - 1) / kLagBlock;
            a.hs = a.l16 + kLagBlock * a.n_blocks;
            const LagOperands ops = lag_operands(32ll * C, 32ll * C, a.hs, a.l16);
            const unsigned short* base = reinterpret_cast<const unsigned short*>(1 << 20);
            g_begin = 1 << 20;
            g_end = g_begin + 2 * (ops.h + ops.b) * (x3 ? 2 : 1);
            a.h_hi = base;
            a.b_hi = base + ops.h;
            a.h_lo = base + ops.h + ops.b;
            a.b_lo = base + 2 * ops.h + ops.b;
            const int most = x3 ? 7 : 8;
            a.n_ranges = (a.n_blocks + most - 1) / most;
            const int nb = (a.n_blocks + a.n_ranges - 1) / a.n_ranges;
            a.n_long = a.n_blocks - a.n_ranges * (nb - 1);
            const long before = g_bad;
            if (x3) ranges<true, 7>(a, nb);
            else ranges<false, 8>(a, nb);
            ++cases;
            if (g_bad > before && before == 0)
              printf("first loads outside the operands: L=%d C=%d [%d, %d] %s\n", L, C, lo, hi, x3 ? "bf16x3" : "fp16");
          }
        }
  printf("%d cases, %ld loads, %ld outside the operands\n", cases, g_loads, g_bad);
  return g_bad ? 1 : 0;
}
