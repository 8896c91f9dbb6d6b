// hp_mid_policy.h -- which projection launches the mid kernels
// (kquant_mid.hip) take: rules on sizes and types alone.
//
// Host-only C++ without HIP, so that the rules can be run on the CPU.
#ifndef HP_MID_POLICY_H
#define HP_MID_POLICY_H

#include <stddef.h>

namespace hp {

// What a launch's weights are.
struct MidShape {
  long long segs;  // 16-row segments of all weights
  int nb;          // blocks of a row
  bool q4, q6;     // some weight is Q4_K, Q6_K
  bool f16;        // every weight is exact in single f16 operands (no full-range Q6_K scales)
  bool pair;       // gate and up with their GeGLU
  bool folded;     // the launch before writes the activation tiles
  int cus;
};

// From five columns on: against the vector-ALU kernels (full-range Q6_K) and
// kquant_mfma, five columns of Q/K/V 15.5 -> 10.4 us, O 17.4 -> 9.7, down 35.0
// -> 18.9, the FFN 64.1 -> 38.3.  Fewer columns stay on the kernels whose
// launches quantise their own input: at three Q/K/V 9.5 against 10.4 us here,
// O 7.5 against 9.7, down 17.3 against 19.0, the FFN 35.9 against 37.3; at two
// 8.3, 6.3, 13.1 and 28.3 against 10.5, 9.6, 18.9 and 37.2.  At four the line
// is not where each launch would have it: O 8.1 against 9.7, but Q/K/V 11.3
// against 10.4, down 21.2 against 18.9, the FFN 42.9 against 37.9.  From two
// columns on for some launches of 16 segments a CU.
constexpr size_t kMidMinCols = 5;
constexpr int kMidLargeSegs = 16;  // 16-row segments per CU

// Row waves (a wave per segment) or else class pairs.
inline bool mid_row_waves(const MidShape &l) { return l.q4 != l.q6 && l.segs >= 2ll * l.cus; }

// Class pairs launch a workgroup of up to 512 threads per segment (counted in
// eights) and 16 columns; a grid holds fewer than 2^32 threads.  Row waves
// launch at most a workgroup per CU.
inline bool mid_grid_fits(const MidShape &l, size_t cols) {
  const unsigned long long groups = (cols + 15) / 16;
  return mid_row_waves(l) || (unsigned long long)((l.segs + 7) / 8 * 8) * groups < (1ull << 32) / 512;
}

// Row waves' items of eight segments, one workgroup a CU: the last round of
// items at least leaves no more than a fifth of the launch's CU time idle.
inline bool mid_rounds_full(const MidShape &l) {
  const long long items = (l.segs + 7) / 8, rounds = (items + l.cus - 1) / l.cus;
  return 5 * items >= 4 * rounds * l.cus;
}

// Two to four columns of a launch of 16 segments a CU (heads; gate/up of
// 32768 rows).  Times are this kernel's over the other's, measured at 65536 to
// 262144 rows (gate/up: 32768 to 65536) of 1, 4, 10 and 15 blocks.
inline bool mid_takes_few(const MidShape &l, size_t cols) {
  if (cols < 2 || l.segs < (long long)kMidLargeSegs * l.cus) return false;
  // mixed types, class pairs: full-range Q6_K from 10 blocks 0.70 to 0.87 at
  // three and four columns; else 0.87 to 1.58
  if (!mid_row_waves(l)) return !l.f16 && l.nb >= 10 && cols > 2;
  if (l.pair) {
    // the wide kernel with GeGLU: four columns 0.35 to 0.97; three 0.54 to
    // 1.03 for Q6_K, 0.63 to 0.72 for Q4_K from 10 blocks (fewer: up to
    // 1.22); two 0.67 to 0.86 for Q6_K from 10 blocks (fewer: up to 1.18),
    // 0.76 to 0.96 for Q4_K from 15 (10 blocks: up to 1.15)
    if (cols == 4) return true;
    if (cols == 3) return !l.q4 || l.nb >= 10;
    return l.nb >= (l.q4 ? 15 : 10);
  }
  // kquant_mfma, one launch and one operand a weight: 0.93 to 1.46, Q6_K 1.03 and more
  if (l.f16) return false;
  // the vector-ALU kernels, weights read once for the columns they hold: from
  // four blocks 0.56 to 0.90 at three and four columns, 0.80 to 1.02 at two
  // (last round nearly empty: 1.05); one block up to 1.48
  return l.nb >= 4 && (cols > 2 || mid_rounds_full(l));
}

// Five to eight columns for which kquant_mfma's one launch (single-operand
// weights) is faster than a launch that writes activation tiles and this
// kernel: short rows.  Times are this kernel's over that one's.
inline bool mfma_takes(const MidShape &l, size_t cols) {
  if (!l.f16 || l.pair || l.folded || cols > 8) return false;
  if (l.q4 && l.q6 && l.segs >= 2ll * l.cus) {
    // class pairs for want of one type: 8192 rows of 1 and 2 blocks 1.20,
    // 1.07, of 3 blocks 0.98; 16384 of 3 blocks 1.05 to 1.21, of 4 0.98;
    // 32768 to 131072 of 4 to 6 blocks 1.05 to 1.32, of 10 blocks 0.97
    return l.nb <= (l.segs >= 8ll * l.cus ? 6 : l.segs >= 4ll * l.cus ? 3 : 2);
  }
  // many rows: Q4_K 32768 of one block 0.95, 65536 0.78; Q6_K 32768 1.05, 65536 0.86
  if (l.segs >= (l.q4 ? 8ll : 16ll) * l.cus) return false;
  // one block 1.02 to 1.16
  if (l.nb == 1) return true;
  // row waves of Q6_K: two blocks 1.05 to 1.14, three 1.05 to 1.11 at five
  // columns and 0.92 to 0.95 at six to eight; four 0.9 and less
  return l.q6 && mid_row_waves(l) && (l.nb == 2 || (l.nb == 3 && cols == 5));
}

// Hundreds of columns (host-pointer calls, which keep to bit-exact kernels) of
// class-pair launches in single f16 operands, for which the bit-exact prefill
// kernel with its 64-column tiles is faster: a class pair reads a column's
// activation tiles once per 16-row segment, and over short rows the exchange
// of the chains costs as much as the blocks.  Times are this kernel's over that
// one's, measured at 16 to 500 segments.
inline bool prefill_takes(const MidShape &l, size_t cols) {
  if (!l.f16 || mid_row_waves(l)) return false;  // row waves 0.41 to 0.74
  // class pairs for want of one type, short rows: 8192 to 131072 rows of one
  // and two blocks 0.99 to 1.26 from 40 columns, 0.69 to 0.93 at 32
  if (l.segs >= 2ll * l.cus && l.nb <= 2 && cols > 32) return true;
  const long long work = l.segs * (long long)cols;
  // one block 0.92 to 1.01 up to 65536 segment columns, 1.08 to 1.71 from
  // 81920; 16 segments 1.08 at 1536 columns, 1.25 at 2048
  if (l.nb == 1) return work >= 80000 || cols >= 2048;
  // two blocks 0.97 to 1.0 at 81920, 1.04 to 1.34 from 122880
  if (l.nb == 2) return work >= 120000;
  // four blocks 0.77 to 0.95.  Long rows, whose activation tiles pass the L2
  // (128 segments and more): 15 to 40 blocks 0.81 to 1.02 at 768 columns, 1.05
  // to 1.21 at 1024; 10 blocks 0.96 to 0.99 at 1024, 0.97 to 1.09 from 1536;
  // 16 segments 0.5 to 1.1; gate/up 0.5 to 0.95
  if (l.pair || l.segs < 128) return false;
  return cols >= 1536 ? l.nb >= 10 : cols >= 1024 && l.nb >= 15;
}

// Rows of one block in both types (class pairs of one block: the exchange of
// the chains is most of the launch), many of them: 131072 rows 1.13 to 1.23 up
// to 12 columns, 0.9 to 1.0 at 16; gate/up of 16384 in single f16 operands 1.39
// to eight columns, 0.84 from nine.  Fewer rows 0.5 to 0.98.
inline bool one_block_mixed(const MidShape &l, size_t cols) {
  if (!l.q4 || !l.q6 || l.nb != 1) return false;
  return l.pair ? l.f16 && cols <= 8 && l.segs >= 8ll * l.cus : cols < 16 && l.segs >= 32ll * l.cus;
}

inline bool mid_takes(const MidShape &l, size_t cols) {
  if (!mid_grid_fits(l, cols) || one_block_mixed(l, cols)) return false;
  return cols >= kMidMinCols ? !mfma_takes(l, cols) : mid_takes_few(l, cols);
}

}  // namespace hp

#endif
