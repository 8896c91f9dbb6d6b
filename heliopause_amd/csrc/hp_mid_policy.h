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
  int cus;
};

// From five columns on (measured against the vector-ALU and kquant_mfma
// kernels: five columns of Q/K/V 14.3 -> 9.5 us, of the FFN 61.8 -> 36.0; at
// four O 6.9 -> 9.1, Q/K/V 9.8 -> 9.8, with the launch that writes the
// activation tiles), and from two on for launches of 16 segments a CU (the
// head, two columns 176 -> 155 us, three 223 -> 164; heads of 2000 segments
// the same either way).
constexpr size_t kMidMinCols = 5;
constexpr size_t kMidMinColsLarge = 2;
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

inline bool mid_takes(const MidShape &l, size_t cols) {
  const size_t least = l.segs >= (long long)kMidLargeSegs * l.cus ? kMidMinColsLarge : kMidMinCols;
  return cols >= least && mid_grid_fits(l, cols);
}

}  // namespace hp

#endif
