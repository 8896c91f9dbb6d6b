// CPU check of the rules in heliopause_amd/csrc/hp_mid_policy.h on an MI355X's
// 256 CUs.
#include <cstdio>
#include <cstdlib>

#include "hp_mid_policy.h"

namespace {

hp::MidShape shape(long long rows, int k, bool q4, bool q6, bool f16) {
  return hp::MidShape{(rows + 15) / 16, k / 256, q4, q6, f16, 256};
}

int failures = 0;
void check(bool ok, const char *what) {
  if (!ok) {
    std::printf("FAIL %s\n", what);
    failures++;
  }
}

// The grid of a class-pair launch stays below 2^32 threads, whatever is taken.
void grids() {
  for (long long rows = 1; rows < (1ll << 31) / 64; rows = rows * 2 + 1)
    for (size_t cols = 1; cols <= 65535; cols = cols * 2 + 1)
      for (int t = 1; t < 4; t++) {
        const hp::MidShape l = shape(rows, 256, t & 1, t & 2, true);
        if (!hp::mid_takes(l, cols) || hp::mid_row_waves(l)) continue;
        const double threads = double((l.segs + 7) / 8 * 8) * double((cols + 15) / 16) * 512;
        check(threads < 4294967296.0, "grid");
      }
  check(!hp::mid_takes(shape(8192 * 16, 256, true, true, true), 65535), "131072 mixed rows, 65535 columns");
  check(hp::mid_takes(shape(262144, 2560, false, true, false), 65535), "one type: row waves");
}

}  // namespace

int main() {
  grids();
  if (failures) return 1;
  std::printf("mid policy ok\n");
  return 0;
}
