"""Work lists of band-limited transforms (prune_lists.hpp): the blocks that
hold a wanted line, on meshes whose line count is and is not a multiple of a
block's.  The program is built with the library's checked vectors, so a read
past a list aborts it."""

import subprocess

import pytest

import conftest as cf

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include "prune_lists.hpp"
using namespace trvg;
static double k2(int i, int n, double dk) {
  const double k = (i < n / 2 ? i : i - n) * dk;
  return k * k;
}
static void same(const std::vector<int>& got, const std::set<int>& want) {
  if (std::vector<int>(want.begin(), want.end()) != got) { std::puts("differ"); std::exit(1); }
}
int main(int argc, char** argv) {
  const int n[3] = {std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3])};
  const double dk[3] = {1., 0.9, 1.1};
  for (int nl : {1, 2, 3, 8, 11, 14, 17, 256})
    for (double kc : {0., 0.5, 1.5, 0.4371 * n[0], 1e30}) {
      const double c2 = kc * kc;
      std::set<int> z, y, xx, xy;
      double lines = 0., slabs = 0.;
      for (int i = 0; i < n[0]; i++) {
        slabs += k2(i, n[0], dk[0]) < c2;
        for (int j = 0; j < n[1]; j++)
          if (k2(i, n[0], dk[0]) + k2(j, n[1], dk[1]) < c2) { z.insert((i * n[1] + j) / nl); lines++; }
        for (int k = 0; k < n[2]; k++) {
          if (k2(i, n[0], dk[0]) < c2) y.insert((i * n[2] + k) / nl);
          if (k2(k, n[2], dk[2]) < c2) xy.insert((i * n[2] + k) / nl);
        }
      }
      for (int j = 0; j < n[1]; j++)
        for (int k = 0; k < n[2]; k++)
          if (k2(j, n[1], dk[1]) + k2(k, n[2], dk[2]) < c2) xx.insert((j * n[2] + k) / nl);
      const PruneLists a = make_prune_lists(n, dk, c2, nl, nl);
      const PruneListsXF b = make_prune_lists_xfirst(n, dk, c2, nl, nl);
      same(a.zblocks, z);
      same(a.yblocks, y);
      same(b.xblocks, xx);
      same(b.yblocks, xy);
      if (a.d_lines != lines || a.slabs != slabs) return 1;
    }
  return 0;
}
"""


@pytest.fixture(scope='module')
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp('lists')
    (d / 'main.cpp').write_text(PROGRAM)
    subprocess.run(['g++', '-std=c++17', '-O1', '-D_GLIBCXX_ASSERTIONS',
                    '-I', str(cf.ROOT / 'triumvirate_amd' / 'csrc'),
                    str(d / 'main.cpp'), '-o', str(d / 'main')], check=True)
    return d / 'main'


@pytest.mark.parametrize('mesh', [(16, 16, 16), (14, 12, 18), (8, 10, 26),
                                  (144, 120, 18), (64, 8, 32)])
def test_listed_blocks_hold_a_wanted_line(program, mesh):
    subprocess.run([str(program), *map(str, mesh)], check=True, timeout=60)
