// A batch whose launches fail: every request of it returns the error, on each
// slot's first batch too, and the server goes on.
#include <stdio.h>

#include <atomic>
#include <vector>

#include "../../include/seismic_xcorr.h"
#include "standin.h"

int main() {
  sxc_server_desc d{};
  d.n_catalog = 64;
  d.n_channels = 1;
  d.catalog_len = 256;
  d.max_query_len = 256;
  d.top_k = 4;
  d.max_batch_events = 8;
  d.n_slots = 2;
  std::vector<float> cat(64 * 256, 1.f);
  sxc_server* s = nullptr;
  if (sxc_server_create(&d, cat.data(), &s)) return printf("create failed: %s\n", seismic_last_error()), 1;
  std::atomic<bool> fail{true};
  for (int stage = 0; stage < 3; ++stage) {
    if (stage == 0) standin::on_forward = [&](int, const sxc::ForwardArgs&) { return fail ? 1 : 0; };
    if (stage == 1) {
      standin::on_forward = nullptr;
      standin::on_pairs = [&](int, bool, const sxc::PairArgs&) { return fail ? 1 : 0; };
    }
    if (stage == 2) fail = false;
    std::vector<long long> ids;
    const int len[8] = {256, 200, 100, 256, 1, 2, 3, 4};
    for (int k = 0; k < 20; ++k) {
      long long id = 0;
      if (sxc_server_submit(s, cat.data(), 256, len, 8, &id)) return printf("submit failed\n"), 1;
      ids.push_back(id);
    }
    std::vector<sxc_match> out(8 * 4);
    for (long long id : ids) {
      const int rc = sxc_server_wait(s, id, out.data(), nullptr);
      if (rc != (fail ? SXC_ERR_HIP : SXC_OK)) return printf("stage %d: status %d\n", stage, rc), 1;
    }
  }
  sxc_server_destroy(s);
  printf("ok, %zu bytes left\n", standin::used());
  return standin::used() ? 1 : 0;
}
