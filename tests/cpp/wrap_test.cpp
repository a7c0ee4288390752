// Checks wrap.hpp against 64-bit arithmetic: every margin a pass has, axes from one
// node to the longest an int32 node index allows.  Prints "ok".
#include "../../m3lb_amd/csrc/wrap.hpp"

#include <cstdint>
#include <cstdio>

int main() {
  const int sizes[] = {1,         2,         3,         5,         8,          9,
                       10,        63,        64,        65,        1000,       715827882,
                       715827883, 800000000, 1 << 30,   1500000000, 2147483600};
  long long checked = 0;
  for (int s : sizes) {
    for (int m = 0; m <= 66; ++m) {
      const int64_t at[] = {-m, -m / 2, -1, 0, s / 2, int64_t(s) - 1, s, int64_t(s) - 1 + m};
      for (int64_t v : at) {
        if (v < -m || v > int64_t(s) - 1 + m || v > INT32_MAX) continue;
        const int64_t want = ((v % s) + s) % s;
        if (m3lb::wrapped(int(v), s) != want) {
          std::printf("v %lld s %d: %d, want %lld\n", (long long)v, s, m3lb::wrapped(int(v), s),
                      (long long)want);
          return 1;
        }
        ++checked;
      }
    }
    for (int v = -200; v < 200; ++v) {
      const int64_t want = ((int64_t(v) % s) + s) % s;
      if (m3lb::wrapped(v, s) != want) {
        std::printf("v %d s %d\n", v, s);
        return 1;
      }
    }
  }
  std::printf(checked > 1000 ? "ok\n" : "too few\n");
  return 0;
}
