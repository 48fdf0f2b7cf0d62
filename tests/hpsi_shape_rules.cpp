// The launch-shape rules of csrc/hpsi_shape.hpp behind a line protocol, for
// tests/test_hpsi_shape_rules.py: one request per input line, one answer per
// output line.
//   resolve n1 n2 n3 md size nb nonlocal analytic nseg  ry ty zlen chunk bt rx psplit max_chunk
//     -> ry ty zlen chunk bt rx psplit fits
//   search n1 n2 n3 md size nb nonlocal analytic nseg  ry rx psplit chunk ty cold
//     the autotuner's search with a clock that prefers these values (0: no
//     preference; cold 1: the first timing takes twice as long, 3: every third
//     half as long) -> the count
//     of timed shapes, the best shape, and each shape timed, in order:
//     ry ty zlen chunk bt order rx proj plds psplit
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

void print(const HpsiShape &h) {
  std::printf(" %d %d %d %d %d %d %d %d %d %d", h.ry, h.ty, h.zlen, h.chunk, h.bt, h.order, h.rx, h.proj, h.plds,
              h.psplit);
}

int search(std::istream &in) {
  size_t s = 0;
  int nb = 0;
  const HpsiGrid g = read_grid(in, s, nb);
  HpsiShape want, best;
  int cold = 0;
  in >> want.ry >> want.rx >> want.psplit >> want.chunk >> want.ty >> cold;
  std::vector<HpsiShape> seen;
  float t = 0.f;
  const int rc = search_shape(
      g, s, nb,
      [&](const HpsiShape &h, float &ms) {
        if (!fits(g, h, s)) return -1;
        seen.push_back(h);
        ms = 100.f;
        for (auto f : {&HpsiShape::ry, &HpsiShape::rx, &HpsiShape::psplit, &HpsiShape::chunk, &HpsiShape::ty})
          if (want.*f && h.*f == want.*f) ms -= 10.f;
        if (cold == 1 && seen.size() == 1) ms *= 2.f;
        if (cold == 3 && seen.size() % 3 == 0) ms *= 0.5f;
        return 0;
      },
      [] { return true; }, best, t);
  std::printf("%d", int(seen.size()));
  print(best);
  for (const HpsiShape &h : seen) print(h);
  std::printf("\n");
  return rc;
}

}  // namespace

int main() {
  std::string line, what;
  while (std::getline(std::cin, line)) {
    std::istringstream in(line);
    in >> what;
    if (what == "search") {
      if (search(in) || !in) return 2;
      continue;
    }
    size_t s = 0;
    int nb = 0;
    HpsiGrid g = read_grid(in, s, nb);
    HpsiShape a;
    in >> a.ry >> a.ty >> a.zlen >> a.chunk >> a.bt >> a.rx >> a.psplit >> g.max_chunk;
    if (!in || what != "resolve") return 2;
    const HpsiShape sh = resolve_shape(g, a, s, nb);
    std::printf("%d %d %d %d %d %d %d %d\n", sh.ry, sh.ty, sh.zlen, sh.chunk, sh.bt, sh.rx, sh.psplit,
                int(fits(g, sh, s)));
  }
  return 0;
}
