// The tile kernel's operand loads on the CPU: planes laid out as a plan's, against
// pages that cannot be read on either side; every lane's blocks of lags.
#include <hip/hip_runtime.h>

#include <stdio.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>

using ::max;
using ::min;
#define __builtin_amdgcn_alignbyte(hi, lo, n) ((hi) ^ (lo))
#define __builtin_amdgcn_sched_group_barrier(...) ((void)0)
#include "../../seismic_amd/csrc/xc_lag_tile.hip"

void on_buffer_load(const BufferRsrc&, int, int, int) {}
using namespace sxc;

int main() {
  const size_t page = sysconf(_SC_PAGESIZE);
  int cases = 0;
  for (int L : {1, 15, 16, 17, 33, 64, 100, 513, 1000})
    for (int C : {1, 3})
      for (int lo = -(L - 1); lo < L; lo += std::max(1, L / 37))
        for (int span : {0, 1, 15, 30, 47, 104}) {
          const int hi = std::min(lo + span, L - 1), l16 = (L + 15) / 16 * 16;
          // the layout of sxc_lag_plan_create_band
          const int first = tile_first_lag(lo), blocks = (hi - first + 1 + kTileLags - 1) / kTileLags;
          const int p0 = std::max(0, (first + kTileLags * blocks - 1 + 7) / 8 * 8);
          const int ls = (std::max(p0 + l16, p0 + l16 - first + 9) + 7) / 8 * 8;
          const size_t bytes = 2ul * 2 * C * ls, span_bytes = (bytes + page - 1) / page * page;
          char* m = (char*)mmap(nullptr, span_bytes + 2 * page, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
          mprotect(m + page, span_bytes, PROT_READ | PROT_WRITE);
          // two events' planes, once against the page after them, once against the one before
          for (char* at : {m + page + span_bytes - bytes, m + page})
            for (int row = 0; row < 2; ++row)
              for (int b = 0; b < blocks; ++b)
                for (int h = 0; h < 2; ++h) {
                  const unsigned short* r = (const unsigned short*)at + (size_t)row * C * ls;
                  f32x16 acc[kTileLags];
                  lag_block<true>(acc, r, r, r, r, ls, C, l16, p0, first + kTileLags * b, h);
                  lag_block<false>(acc, r, nullptr, r, nullptr, ls, C, l16, p0, first + kTileLags * b, h);
                  if (((size_t)(r + p0 + 8 * h - (first + kTileLags * b) - 15) & 15) != ((size_t)at & 15))
                    return printf("unaligned window: L=%d [%d, %d]\n", L, lo, hi), 1;
                }
          munmap(m, span_bytes + 2 * page);
          ++cases;
        }
  printf("%d cases\n", cases);
  return 0;
}
