// The lag-window scan's running state (insert16, side_of, merge_side) on the CPU,
// over values many of which share all but their last four bits: the extremum
// against a plain scan, and the best key's lag, which is its first one unless
// other values share those bits.
#include <hip/hip_runtime.h>

#include <random>
#include <stdio.h>

using ::max;
using ::min;
template <typename T>
static void host_med3(T& d, T a, T b, T c) {
  d = max(min(a, b), min(max(a, b), c));
}
#define asm(...) host_med3(d, a, b, c)  // v_med3 in the functions of that name
#include "../../seismic_amd/csrc/xc_lag.hip"
#undef asm

void on_buffer_load(const BufferRsrc&, int, int, int) {}
using namespace sxc;

int main() {
  std::mt19937 rng(1);
  long sides = 0, close_ones = 0, wrong = 0;
  for (int it = 0; it < 200000; ++it) {
    const int n = 1 + rng() % 6, kind = it % 4;
    float value[6 * 32];
    for (float& v : value) {
      const unsigned q = rng();
      if (kind == 0) v = ((int)(q % 2001) - 1000) * 1e-3f;
      if (kind == 1) v = __int_as_float(0x3f300000 + q % 24) * (q >> 29 ? 1.f : -1.f);
      if (kind == 2) v = q % 5 ? (q >> 8) % 100 * -0.01f : __int_as_float(0x3f300000 + (int)((q >> 8) % 40) - 20);
      if (kind == 3) v = q % 9 ? (q % 3 ? 0.f : 1e-7f) : -__int_as_float(0x3f7ffff0 + (q >> 8) % 20);
    }
    Side s[2][2];
    for (int h = 0; h < 2; ++h) {  // a lane of either half
      Best3<int> pos{0, 0, (int)0x80000000, (int)0x80000000, 0, 0};
      Best3<unsigned> neg{0x80000000u, 0x80000000u, 0u, 0u, 0, 0};
      for (int b = 0; b < n; ++b) {
        int bits[16], key[16];
        unsigned ubits[16], ukey[16];
        for (int r = 0; r < 16; ++r) {
          ubits[r] = bits[r] = __float_as_int(value[32 * b + lag_in_block(h, r)]);
          ukey[r] = key[r] = (bits[r] & ~15) | (15 - lag_order(r));
        }
        insert16(pos, bits, key, b);
        insert16(neg, ubits, ukey, b);
      }
      s[0][h] = side_of(pos, h);
      s[1][h] = side_of(neg, h);
    }
    for (int sd = 0; sd < 2; ++sd) {
      merge_side(s[sd][0], s[sd][1]);
      float best = 0.f;
      int at = -1, sharing = 0;
      for (int l = 0; l < 32 * n; ++l) {
        const float v = sd ? -value[l] : value[l];
        if (v > best) best = v, at = l;
      }
      auto shares = [&](float v) { return (__float_as_uint(v) ^ __float_as_uint(best)) < 16u; };
      for (int l = 0; l < 32 * n; ++l) sharing += shares(sd ? -value[l] : value[l]);
      const int k = s[sd][0].o1;
      const float got = sd ? __uint_as_float((unsigned)s[sd][0].e) : __int_as_float(s[sd][0].e);
      ++sides;
      close_ones += sharing > 1;
      const bool ok = got == best && (sharing > 1 ? shares(sd ? -value[k] : value[k]) : k == at);
      if (at >= 0 && !ok && wrong++ < 5)
        printf("kind %d side %d: %.9g at %d, should be %.9g at %d\n", kind, sd, got, k, best, at);
    }
  }
  printf("%ld sides, %ld with close keys, %ld wrong\n", sides, close_ones, wrong);
  return wrong || close_ones < sides / 4;
}
