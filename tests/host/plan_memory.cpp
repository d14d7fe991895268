// Plans on a device with little memory left.  Argument "fft": a window far
// shorter than the traces, in just the memory that whole rows need: the plan is made
// and runs on whole rows; with more it runs on segments.
#include <stdio.h>
#include <string.h>

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

int main(int argc, char** argv) {
  const int rc = !strcmp(argv[1], "fft") ? fft() : 2;
  if (!rc) printf("ok\n");
  return rc;
}
