// Where the KN loop in one launch (kn_loop.hip) is taken.  Host arithmetic only.
#pragma once

namespace isvd {

constexpr int kLoopRows = 16;     // rows of the state and of M per workgroup
constexpr int kLoopBlocks = 128;  // workgroups at most

// FP64 (elem = 8 bytes) up to 64 columns: three l x l matrices in LDS.  FP32 up to 80: at 96 the
// chain's products in one workgroup take longer than those spread over 18 (80 against 75 us an
// iteration, Nl = 2016).  The workgroups wait for each other, so all must be resident at once: LDS
// leaves room for one per CU at the larger l, and a device or partition with fewer CUs than workgroups
// takes the separate launches.
inline bool kn_loop_fits(int elem, long long l, long long Nl, int cus) {
  const long long blocks = (Nl + kLoopRows - 1) / kLoopRows;
  return l >= 1 && l <= (elem == 8 ? 64 : 80) && Nl >= l && blocks <= kLoopBlocks && blocks <= cus;
}

}  // namespace isvd
