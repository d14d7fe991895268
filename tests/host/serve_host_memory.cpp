// A server whose warm request buffers cannot be allocated serves without them.
#include <stdio.h>
#include <stdlib.h>

#include <new>
#include <vector>

#include "../../include/seismic_xcorr.h"
#include "standin.h"

static bool g_short = false;
void* operator new(size_t n) {
  if (g_short && n > (1u << 20)) throw std::bad_alloc();
  void* p = malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

int main() {
  sxc_server_desc d{};
  d.n_catalog = 16;
  d.n_channels = 1;
  d.catalog_len = 512;
  d.max_query_len = 512;
  d.top_k = 2;
  d.max_batch_events = 1024;  // 2 MiB a batch, 8 buffers
  d.n_slots = 2;
  std::vector<float> cat(16 * 512, 1.f);
  sxc_server* s = nullptr;
  g_short = true;
  if (sxc_server_create(&d, cat.data(), &s)) return printf("create: %s\n", seismic_last_error()), 1;
  const int len[3] = {512, 100, 7};
  std::vector<sxc_match> out(3 * 2);
  for (int k = 0; k < 20; ++k) {
    long long id = 0;
    if (sxc_server_submit(s, cat.data(), 512, len, 3, &id) || sxc_server_wait(s, id, out.data(), nullptr))
      return printf("request: %s\n", seismic_last_error()), 1;
  }
  sxc_server_destroy(s);
  printf("ok\n");
  return 0;
}
