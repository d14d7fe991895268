// Plans, host-buffer jobs and tiled runs on a device with little memory left.
// fft: a window far shorter than the traces, in just the memory that whole rows
// need: the plan is made and runs on whole rows; with more it runs on segments.
// lag: less memory than the row operands of all events take: they are held for a
// band of events at a time, and every launch finds its rows' operands.
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <set>
#include <vector>

#include "../../include/seismic_xcorr.h"
#include "standin.h"

static int g_seg;

static int execute(sxc_plan* p, int n, int C, int L) {
  const size_t np = (size_t)n * (n + 1) / 2;
  std::vector<float> x((size_t)n * C * L, 1.f), v(np);
  std::vector<int> l(np);
  g_seg = -1;
  standin::on_forward = [&](int, const sxc::ForwardArgs& a) { return g_seg = a.n_seg, 0; };
  const int rc = sxc_plan_execute(p, x.data(), L, L, v.data(), l.data(), v.data(), l.data(), nullptr);
  standin::on_forward = nullptr;
  return rc;
}

static int fft() {
  const int n = 200, L = 4096, P = 8192;
  sxc_plan_desc d{n, 1, L, P, -50, 50, 0.f, 0.f, 0, SXC_FORM_FFT_F32};
  // spectra, norms, near-tie records, work list and counter, and tables of two periods
  const size_t pairs = (size_t)n * (n + 1) / 2;
  const size_t whole = (size_t)n * (P / 2 + 32) * 8 + n * 8 + pairs * (16 + 8) + 2 * (8192 + 4097 + 2048) * 8;
  sxc_plan* p = nullptr;
  if (sxc_plan_create(&d, &p) || execute(p, n, 1, L) || g_seg < 2) return printf("no segments (%d)\n", g_seg), 1;
  const size_t cut = standin::used();
  sxc_plan_destroy(p);
  if (cut <= whole) return printf("the job does not tell: %zu <= %zu\n", cut, whole), 1;
  standin::limit = whole;
  if (sxc_plan_create(&d, &p)) return printf("create: %s\n", seismic_last_error()), 1;
  if (seismic_last_error()[0]) return printf("error left: %s\n", seismic_last_error()), 1;
  if (execute(p, n, 1, L) || g_seg != 0) return printf("execute: %s, segments %d\n", seismic_last_error(), g_seg), 1;
  sxc_plan_destroy(p);
  standin::limit = 1 << 20;
  if (sxc_plan_create(&d, &p) != SXC_ERR_MEMORY || p) return printf("made in 1 MiB\n"), 1;
  return standin::used() != 0;
}


// Follows the row operands: which event each place of the allocation holds.
struct Rows {
  const double* norms0 = nullptr;             // of event 0 (the first launch)
  std::map<const unsigned short*, int> held;  // place -> event
  std::set<std::pair<int, int>> pairs;        // tiles run
  int launches = 0, bad = 0;
  void watch() {
    standin::on_lag_prep = [this](const sxc::LagPrepArgs& a) {
      if (!a.energy_in && !norms0) norms0 = a.norms;
      const int e0 = (int)(a.norms - norms0) / a.n_channels;
      for (int e = 0; e < a.n_rows / a.n_channels; ++e) {
        const unsigned short* at = a.h_hi + (size_t)e * a.n_channels * 2 * a.hs;
        held[at] = e0 + e;
        bad += !standin::size_of(at + (size_t)a.n_channels * 2 * a.hs - 1);
      }
      return 0;
    };
    standin::on_lag_pairs = [this](bool, const sxc::LagPairArgs& a) {
      ++launches;
      for (int t = 0; t < a.n_tiles; ++t) {
        const int ti = a.tiles[t].x + a.tile_row0, tj = a.tiles[t].y + a.tile_col0;
        if (32 * ti >= a.n_events || 32 * tj >= a.n_events) continue;
        bad += !pairs.insert({ti, tj}).second;
        for (int i = 32 * ti; i < std::min(32 * ti + 32, a.n_events); ++i) {
          auto it = held.find((const unsigned short*)((size_t)a.h_hi + (size_t)i * a.n_channels * 4 * a.hs));
          bad += it == held.end() || it->second != i;
        }
      }
      return 0;
    };
  }
  bool all(int n) {
    const int T = (n + 31) / 32;
    const bool ok = !bad && (int)pairs.size() == T * (T + 1) / 2;
    if (!ok) printf("%d bad, %zu of %d tiles\n", bad, pairs.size(), T * (T + 1) / 2);
    pairs.clear();
    return ok;
  }
};

static int lag() {
  const int n = 203, C = 2, L = 1000, w = 40, block = 96;
  const size_t np = (size_t)n * (n + 1) / 2;
  std::vector<float> x((size_t)n * C * L, 1.f), v(np);
  std::vector<int> l(np);
  for (int form : {SXC_FORM_LAG_BF16X3, SXC_FORM_LAG_FP16}) {
    sxc_plan_desc d{n, C, L, 0, -w, w, 0.f, 0.f, 1, form};
    // 0: a plan, 1: a host-buffer job, 2: a tiled run; with all the memory, then with
    // what zero-padded planes of l16 + 2 (w + 16) samples in place of the operands take
    for (int what = 0; what < 3; ++what) {
      size_t full = 0;
      for (int low = 0; low < 2; ++low) {
        // and one band of 32 events, energies and the room past the operands
        const size_t sample = C * 2 * (form == SXC_FORM_LAG_BF16X3 ? 2 : 1);  // bytes of every event
        const size_t l16 = 1008, hs = l16 + 32 * 3, operands = n * sample * (2 * hs + l16);
        standin::limit = low ? full - operands + n * sample * (l16 + 2 * (w + 16)) + 32 * sample * 2 * hs + (1 << 16)
                             : (size_t)1 << 40;
        Rows r;
        r.watch();
        sxc_plan* p = nullptr;
        sxc_tiled* t = nullptr;
        int rc = 0;
        if (what == 0) {
          rc = sxc_plan_create(&d, &p);
          full = rc || low ? full : standin::used();
          for (int k = 0; k < 2 && !rc; ++k) {
            rc = sxc_plan_execute(p, x.data(), L, L, v.data(), l.data(), v.data(), l.data(), nullptr);
            if (!rc && !r.all(n)) rc = -100;
          }
          sxc_plan_destroy(p);
        } else if (what == 1) {
          setenv("SEISMIC_XCORR_CACHE_MB", "0", 1);
          standin::on_resolve = [&](int, const sxc::ResolveArgs&) {
            full = low ? full : standin::used();
            return 0;
          };
          rc = sxc_allpairs_host(&d, x.data(), L, L, v.data(), l.data(), v.data(), l.data());
          if (!rc && !r.all(n)) rc = -100;
        } else {
          rc = sxc_tiled_create(&d, block, 1, &t);
          full = rc || low ? full : standin::used();
          for (int k = 0; k < 2 && !rc; ++k) {
            sxc_block_info b{};
            rc = sxc_tiled_start(t, x.data(), L, L);
            while (!rc && !(rc = sxc_tiled_next(t, &b, nullptr, nullptr, nullptr, nullptr, 0)) && b.index >= 0) {}
            if (!rc && !r.all(n)) rc = -100;
          }
          sxc_tiled_destroy(t);
        }
        if (rc || standin::used())
          return printf("form %d, case %d, low %d: %d (%s), %zu bytes left\n", form, what, low, rc, seismic_last_error(),
                        standin::used()), 1;
        if (low && standin::limit >= full) return printf("the limit does not tell\n"), 1;
        printf("form %d case %d low %d: %d launches, limit %zu of %zu\n", form, what, low, r.launches, standin::limit, full);
      }
    }
  }
  return 0;
}

// Whole rows or segments, by the size of the job.
static int rule() {
  struct Case { int n, C, L, P, w, n_seg; };
  for (const Case& c : {Case{64, 1, 4096, 8192, 1000, 0}, {200, 1, 4096, 8192, 1000, 0}, {500, 1, 4096, 8192, 1000, 2},
                        {64, 2, 2048, 4096, 200, 2}, {200, 2, 2048, 4096, 200, 0}, {1000, 2, 2048, 4096, 200, 2},
                        {64, 1, 4096, 8192, 50, 5}, {200, 1, 4096, 8192, 50, 5}}) {
    sxc_plan_desc d{c.n, c.C, c.L, c.P, -c.w, c.w, 0.f, 0.f, 0, SXC_FORM_FFT_F32};
    sxc_plan* p = nullptr;
    if (sxc_plan_create(&d, &p) || execute(p, c.n, c.C, c.L) || g_seg != c.n_seg)
      return printf("N=%d C=%d L=%d +-%d: %d segments\n", c.n, c.C, c.L, c.w, g_seg), 1;
    sxc_plan_destroy(p);
  }
  return 0;
}

int main(int argc, char** argv) {
  const int rc = !strcmp(argv[1], "fft") ? fft() : !strcmp(argv[1], "rule") ? rule() : lag();
  if (!rc) printf("ok\n");
  return rc;
}
