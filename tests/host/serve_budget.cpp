// A memory budget of one batch's buffers, item by item, makes a one-slot server.
#include <stdio.h>

#include <vector>

#include "../../include/seismic_xcorr.h"
#include "standin.h"

int main() {
  for (int B : {1, 2, 5, 31, 64, 100})
    for (int n : {1, 64, 200}) {
      sxc_server_desc d{};
      d.n_catalog = n;
      d.n_channels = 2;
      d.catalog_len = 300;
      d.max_query_len = 301;
      d.top_k = 1;
      d.max_batch_events = B;
      d.n_slots = 2;
      // traces, lengths, spectra, norms, scores and lags, top-k lists and slices,
      // and 64 columns of a catalog per work item
      const unsigned long long b = B, C = 2, chunks = (n + 63) / 64;
      d.mem_budget = b * C * 301 * 4 + b * 4 + b * C * (1024 / 2 + 32) * 8 + b * C * 8 + b * n * 8 + b * 12 +
                     b * sxc::kTopkMaxSlices * 12 + b * chunks * 8 + 64;
      std::vector<float> cat((size_t)n * 2 * 300, 1.f);
      sxc_server* s = nullptr;
      if (sxc_server_create(&d, cat.data(), &s)) return printf("B=%d n=%d: %s\n", B, n, seismic_last_error()), 1;
      sxc_server_destroy(s);
    }
  printf("ok\n");
  return 0;
}
