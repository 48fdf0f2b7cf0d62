// The K-split rules of csrc/gram_rules.hpp behind a line protocol, for
// tests/test_gram_rules.py.  One context per run; per input line:
//   tune N nb kc_same kc_pair   keep tuned splits, no answer
//   chunk N nb form             -> points per chunk
//   cand N nb form              -> the candidates
//   own nb form                 -> 1 where the library's kernel runs
#include <cstdio>
#include <iostream>
#include <sstream>
#include <string>

#include "gram_rules.hpp"

int main() {
  std::vector<rsg::GramSplit> tuned;
  std::string line, what;
  while (std::getline(std::cin, line)) {
    std::istringstream in(line);
    in >> what;
    long long N = 0, a = 0, b = 0;
    int nb = 0;
    if (what == "own") {
      in >> nb >> a;
      std::printf("%d\n", int(rsg::gram_own(nb, int(a))));
      continue;
    }
    in >> N >> nb >> a;
    if (what == "tune") {
      in >> b;
      rsg::gram_keep(tuned, nb, N, a, b);
    } else if (what == "chunk") {
      std::printf("%lld\n", static_cast<long long>(rsg::gram_chunk(tuned, nb, N, int(a))));
    } else if (what == "cand") {
      for (int64_t c : rsg::gram_candidates(nb, N, int(a))) std::printf("%lld ", static_cast<long long>(c));
      std::printf("\n");
    } else {
      return 2;
    }
    if (!in) return 2;
  }
  return 0;
}
