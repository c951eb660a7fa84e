// prune_lists.hpp -- work lists of band-limited transforms: the blocks of
// each pass that hold a line inside the band.  Host code without a device.
//
// The host predicate carries a relative margin over the kernels' exactly
// rounded one, so every block the kernels would use is listed (a listed
// block with no needed line only writes zeros that no later pass reads).
#pragma once

#include <vector>

namespace trvg {

// Blocks of nl consecutive lines (the last may hold fewer of the nlines) of
// which in(line) wants one.
template <class In>
std::vector<int> blocks_with(long long nlines, int nl, In in) {
  std::vector<int> blocks;
  for (long long b0 = 0; b0 < nlines; b0 += nl) {
    const long long b1 = b0 + nl < nlines ? b0 + nl : nlines;
    bool any = false;
    for (long long l = b0; l < b1 && !any; l++) any = in(l);
    if (any) blocks.push_back(int(b0 / nl));
  }
  return blocks;
}

// z-first passes: z lines (i, j) inside the radius and y slabs i.
struct PruneLists {
  std::vector<int> zblocks, yblocks;
  double d_lines = 0., slabs = 0.;   // needed z lines and y slabs
};

// x-first passes: x lines (j, k) inside the radius and y lines of such k.
struct PruneListsXF {
  std::vector<int> xblocks, yblocks;
  double x_lines = 0., y_lines = 0.;   // needed x lines, written y lines
};

// Squared wavenumbers of an axis.
inline std::vector<double> axis_k2(int n, double dk) {
  std::vector<double> k2(n);
  for (int i = 0; i < n; i++) {
    const double k = (i < n / 2 ? i : i - n) * dk;
    k2[i] = k * k;
  }
  return k2;
}

// Lines (a, b) of two axes inside the radius (with the margin), b fastest,
// and their exact count.
inline std::vector<char> lines_in(const std::vector<double>& a2, const std::vector<double>& b2,
                                  double kcut2, double& count) {
  const double kc = kcut2 * (1. + 1.e-12);
  std::vector<char> in;
  in.reserve(a2.size() * b2.size());
  for (double a : a2)
    for (double b : b2) {
      in.push_back(a + b < kc);
      count += a + b < kcut2;
    }
  return in;
}

inline PruneLists make_prune_lists(const int n[3], const double dk[3], double kcut2, int nl_z,
                                   int nl_y) {
  PruneLists pl;
  const std::vector<double> x2 = axis_k2(n[0], dk[0]), y2 = axis_k2(n[1], dk[1]);
  const std::vector<char> line_in = lines_in(x2, y2, kcut2, pl.d_lines);
  const std::vector<char> slab_in = lines_in(x2, {0.}, kcut2, pl.slabs);
  pl.zblocks = blocks_with((long long)n[0] * n[1], nl_z, [&](long long l) { return line_in[l]; });
  pl.yblocks = blocks_with((long long)n[0] * n[2], nl_y,
                           [&](long long l) { return slab_in[l / n[2]]; });
  return pl;
}

inline PruneListsXF make_prune_lists_xfirst(const int n[3], const double dk[3], double kcut2,
                                            int nl_x, int nl_y) {
  PruneListsXF pl;
  const std::vector<double> y2 = axis_k2(n[1], dk[1]), z2 = axis_k2(n[2], dk[2]);
  const std::vector<char> line_in = lines_in(y2, z2, kcut2, pl.x_lines);
  double nkz = 0.;
  const std::vector<char> kz_in = lines_in(z2, {0.}, kcut2, nkz);
  pl.y_lines = nkz * n[0];
  pl.xblocks = blocks_with((long long)n[1] * n[2], nl_x, [&](long long l) { return line_in[l]; });
  pl.yblocks = blocks_with((long long)n[0] * n[2], nl_y,
                           [&](long long l) { return kz_in[l % n[2]]; });
  return pl;
}

}  // namespace trvg
