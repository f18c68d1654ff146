// gen_ratnodes.cpp -- writes ratnodes_table.h: the node tables as constants.
// Run by the build: they took 13 ms (coarse) and 35 ms (fine, in extended
// precision) of the first analysis of a process, on grids whose analysis
// takes 0.2.
//
// kRatTab: the coarse table's rows 0 .. kRatBuckets - 1, then the fine one's;
// kRatN: their node counts.  Where no count meets the tolerance, the most.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <vector>

#include "rat_table.h"
#include "ratnodes.h"

using namespace lk;

int main() {
  std::vector<double> tab((size_t)2 * kRatBuckets * kRatLd, 0.0);
  std::vector<int> n((size_t)2 * kRatBuckets, 0);
  for (int b = 1; b < kRatBuckets; ++b) {
    const double kappa = std::ldexp(1.0, b);
    double* s = tab.data() + (size_t)b * kRatLd;
    double* w = s + kRatLd / 2;
    int m = rat::choose(kappa, kRatCoarseTol, kRatCoarseMost, s, w,
                        std::min(kRatCoarseMost, rat::fewest(kappa, kRatCoarseTol)));
    if (m < 0) rat::nodes(kappa, m = kRatCoarseMost, s, w);
    n[(size_t)b] = m;
    s += (size_t)kRatBuckets * kRatLd;
    w += (size_t)kRatBuckets * kRatLd;
    m = rat::choose_fine(kappa, kRatFineTol, kRatFineMost, s, w);
    n[(size_t)(kRatBuckets + b)] = m < 0 ? kRatFineMost : m;   // s and w hold them then
  }
  std::printf("// written by gen_ratnodes.cpp, to be read after rat_table.h\n#pragma once\n\n"
              "namespace lk {\n\nstatic const double kRatTab[2 * kRatBuckets * kRatLd] = {\n");
  for (size_t i = 0; i < tab.size(); ++i)
    if (tab[i] == 0.0) std::printf("0,%s", i % 16 == 15 ? "\n" : "");
    else std::printf("%a,%s", tab[i], i % 4 == 3 ? "\n" : "");
  std::printf("};\nstatic const int kRatN[2 * kRatBuckets] = {\n");
  for (size_t i = 0; i < n.size(); ++i) std::printf("%d,%s", n[i], i % 16 == 15 ? "\n" : "");
  std::printf("};\n\n}  // namespace lk\n");
  return std::ferror(stdout) || std::fflush(stdout) ? 1 : 0;
}
