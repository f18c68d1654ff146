// rat_table.h -- layout of the node tables of the rational approximation of
// x^(-1/2) on [1, 2^b] (ratnodes.h), shared by the kernels that read them and
// gen_ratnodes.cpp, which computes them when the library is built.
#pragma once

namespace lk {

// rows b = 1 .. kRatBuckets - 1: nodes tab[b * kRatLd + j], weights
// tab[b * kRatLd + kRatLd / 2 + j], j < n[b].  The coarse table holds the
// fewest nodes within kRatCoarseTol, at most kRatCoarseMost: enough up to 2^26,
// 1.7e-12 relative at 2^27 growing to 1.2e-7 at 2^47.  The fine one, within
// kRatFineTol and at most kRatFineMost, is within 6e-16 up to 2^42 (its
// tolerance is looked at in 200 points), 2e-15 to 3e-14 from 2^43 on.
constexpr int kRatBuckets = 48;
constexpr int kRatLd = 128;
constexpr int kRatCoarseMost = 31, kRatFineMost = 62;
constexpr double kRatCoarseTol = 1e-12, kRatFineTol = 5e-16;

}  // namespace lk
