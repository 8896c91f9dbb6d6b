// CPU check of the rules in heliopause_amd/csrc/hp_mid_policy.h on an MI355X's
// 256 CUs.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "hp_mid_policy.h"

namespace {

hp::MidShape shape(long long rows, int k, bool q4, bool q6, bool f16) {
  hp::MidShape l{};
  l.segs = (rows + 15) / 16;
  l.nb = k / 256;
  l.q4 = q4;
  l.q6 = q6;
  l.f16 = f16;
  l.cus = 256;
  return l;
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

// Two to four columns: single-operand launches keep kquant_mfma; full-range
// Q6_K from four blocks, at two columns with full rounds only; gate/up by type
// and row length; small launches never.
void few_columns() {
  for (size_t cols = 2; cols <= 4; cols++) {
    for (int k : {256, 1024, 2560, 3840}) {
      check(!hp::mid_takes(shape(262144, k, true, false, true), cols), "Q4_K head");
      check(!hp::mid_takes(shape(262144, k, false, true, true), cols), "narrow Q6_K head");
      check(hp::mid_takes(shape(262144, k, false, true, false), cols) == (k >= 1024), "full-range head");
      check(!hp::mid_takes(shape(65520, k, false, true, false), cols), "fewer than 16 segments a CU");
    }
    check(hp::mid_takes(shape(100000, 2560, false, true, false), cols) == (cols > 2), "last round nearly empty");
    check(hp::mid_takes(shape(131072, 2560, true, true, false), cols) == (cols > 2), "mixed types, full-range");
    check(!hp::mid_takes(shape(131072, 1024, true, true, false), cols), "mixed types, short rows");
    check(!hp::mid_takes(shape(131072, 2560, true, true, true), cols), "mixed types, narrow");
    for (int k : {256, 1024, 2560, 3840})
      for (bool q4 : {true, false}) {
        hp::MidShape l = shape(2 * 40960, k, q4, !q4, q4);
        l.pair = true;
        check(hp::mid_takes(l, cols) == (cols == 4 || (cols == 3 && (!q4 || k >= 2560)) || k >= (q4 ? 3840 : 2560)),
              "gate/up");
      }
  }
  check(!hp::mid_takes(shape(262144, 2560, false, true, false), 1), "one column");
}

// Five to eight columns of short rows in single f16 operands: kquant_mfma,
// unless the activation tiles come without a launch of their own.
void short_rows() {
  for (size_t cols = 5; cols <= 9; cols++) {
    const bool to8 = cols <= 8;
    for (long long rows : {1, 16, 2560, 10240, 32752}) {
      hp::MidShape l = shape(rows, 256, true, false, true);
      check(hp::mid_takes(l, cols) == !to8, "one block");
      l.folded = true;
      check(hp::mid_takes(l, cols), "one block, folded");
      check(hp::mid_takes(shape(rows, 256, false, true, false), cols), "one block, full-range");
      check(hp::mid_takes(shape(rows, 2560, true, true, true), cols), "ten blocks");
    }
    check(hp::mid_takes(shape(32768, 256, true, false, true), cols), "one block, many rows");
    check(hp::mid_takes(shape(32768, 256, false, true, true), cols) == !to8, "one block, many rows of Q6_K");
    check(hp::mid_takes(shape(8192, 512, false, true, true), cols) == !to8, "Q6_K row waves, two blocks");
    check(hp::mid_takes(shape(8192, 768, false, true, true), cols) == (cols != 5), "Q6_K row waves, three blocks");
    check(hp::mid_takes(shape(8160, 512, false, true, true), cols), "Q6_K class pairs, two blocks");
    check(hp::mid_takes(shape(8192, 512, true, false, true), cols), "Q4_K row waves, two blocks");
    check(hp::mid_takes(shape(65536, 1536, true, true, true), cols) == !to8, "mixed, six blocks");
    check(hp::mid_takes(shape(16384, 1024, true, true, true), cols), "mixed, four blocks");
    hp::MidShape l = shape(32768, 256, true, true, false);
    check(hp::mid_takes(l, cols), "mixed, one block, full-range");
    l.pair = true;
    check(hp::mid_takes(l, cols), "mixed gate/up, one block, full-range");
    l.f16 = true;
    check(hp::mid_takes(l, cols) == !to8, "mixed gate/up, one block");
    check(!hp::mid_takes(shape(131072, 256, true, true, false), cols), "mixed, one block, many rows");
  }
}

// Many columns of host calls: the bit-exact prefill kernel for short rows of
// enough work and for long rows of class pairs, never below 64 columns.
void many_columns() {
  for (int nb = 1; nb <= 40; nb++)
    for (long long rows : {16, 2560, 8176})
      for (size_t cols = 1; cols < 64; cols++)
        check(!hp::prefill_takes(shape(rows, 256 * nb, true, false, true), cols), "below 64");
  for (size_t cols = 30; cols < 64; cols++) {
    check(hp::prefill_takes(shape(8192, 512, true, true, true), cols) == (cols > 32), "mixed types, short rows");
    check(!hp::prefill_takes(shape(8192, 1024, true, true, true), cols), "mixed types, four blocks");
  }
  check(!hp::prefill_takes(shape(2560, 256, true, false, true), 256), "one block, 40960");
  check(hp::prefill_takes(shape(2560, 256, true, false, true), 512), "one block, 81920");
  check(!hp::prefill_takes(shape(2560, 512, false, true, true), 512), "two blocks, 81920");
  check(hp::prefill_takes(shape(2560, 512, false, true, true), 768), "two blocks, 122880");
  check(!hp::prefill_takes(shape(5120, 1024, true, false, true), 4096), "four blocks");
  check(hp::prefill_takes(shape(2560, 10240, false, true, true), 1024), "40 blocks");
  check(!hp::prefill_takes(shape(2560, 10240, false, true, true), 1023), "40 blocks, fewer columns");
  check(hp::prefill_takes(shape(3072, 2560, true, true, true), 1536), "10 blocks, mixed");
  check(!hp::prefill_takes(shape(2560, 10240, false, true, false), 4096), "full-range");
  check(!hp::prefill_takes(shape(8192, 10240, false, true, true), 4096), "row waves");
}

}  // namespace

int main() {
  grids();
  few_columns();
  short_rows();
  many_columns();
  if (failures) return 1;
  std::printf("mid policy ok\n");
  return 0;
}
