// The drop-in call with a window far shorter than the traces runs its reversed
// rows at the caller's period: no spectra, tables or column chunks for another.
#include <stdio.h>

#include <vector>

#include "../../include/seismic_xcorr.h"
#include "standin.h"

extern "C" void sxc_reference_call(float*, float*, int, int, int, int, float, float*, int*, float*, int*);

int main() {
  for (int n : {40, 200, 1100}) {
    const int L = 4000, P = 8192, shift = 50;
    const size_t np = (size_t)n * (n + 1) / 2, row = (size_t)n * P;
    std::vector<float> x(row, 1.f), v(np);
    std::vector<int> l(np);
    int chunk = 0, bad = 0;
    const int want = sxc::pair_chunk(P / 128, 1, [&](int c) { return sxc::triangle_items(n, c); });
    standin::on_pairs = [&](int R, bool, const sxc::PairArgs& a) { return chunk = a.chunk, bad += R != P / 128, 0; };
    const size_t before = standin::used();
    sxc_reference_call(x.data(), x.data(), n, L, shift, P, 0.f, v.data(), l.data(), v.data(), l.data());
    if (seismic_last_error()[0]) return printf("N=%d: %s\n", n, seismic_last_error()), 1;
    // the job, kept for the next call: input and reversed rows, outputs, both spectra,
    // norms, records, work lists, and the tables of one period
    const size_t need = 2 * row * 4 + np * 16 + 2 * (size_t)n * (P / 2 + 32) * 8 + n * 8 + np * 16 +
                        2 * 8 * (size_t)sxc::triangle_items(n, want) + (8192 + 4097 + 2048) * 8;
    const size_t got = standin::used() - before;
    if (bad || chunk != want || got > need)
      return printf("N=%d: chunk %d (want %d), %d launches elsewhere, %zu bytes (%zu)\n", n, chunk, want, bad, got, need), 1;
  }
  printf("ok\n");
  return 0;
}
