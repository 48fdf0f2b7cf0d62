// The launch-shape rules of csrc/hpsi_shape.hpp behind a line protocol, for
// tests/test_hpsi_shape_rules.py: one request per input line, one answer per
// output line.
//   resolve n1 n2 n3 md size nb nonlocal analytic nseg  ry ty zlen chunk bt rx psplit
//     -> ry ty zlen chunk bt rx psplit fits
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>

#include "hpsi_shape.hpp"

using namespace rsg;

namespace {

bool fits(const HpsiGrid &g, const HpsiShape &sh, size_t s) {
  return sh.rx == 2 ? pair_fits(g.n1, g.n2, g.md, sh.ry, sh.ty, s) : row_tile(g.n1, g.md, sh.ry, sh.ty, s).fits;
}

HpsiGrid read_grid(std::istream &in, size_t &s, int &nb) {
  HpsiGrid g;
  in >> g.n1 >> g.n2 >> g.n3 >> g.md >> s >> nb >> g.nonlocal >> g.analytic >> g.nseg;
  g.N = int64_t(g.n1) * g.n2 * g.n3;
  return g;
}

}  // namespace

int main() {
  std::string line, what;
  while (std::getline(std::cin, line)) {
    std::istringstream in(line);
    in >> what;
    size_t s = 0;
    int nb = 0;
    const HpsiGrid g = read_grid(in, s, nb);
    HpsiShape a;
    in >> a.ry >> a.ty >> a.zlen >> a.chunk >> a.bt >> a.rx >> a.psplit;
    if (!in || what != "resolve") return 2;
    const HpsiShape sh = resolve_shape(g, a, s, nb);
    std::printf("%d %d %d %d %d %d %d %d\n", sh.ry, sh.ty, sh.zlen, sh.chunk, sh.bt, sh.rx, sh.psplit,
                int(fits(g, sh, s)));
  }
  return 0;
}
