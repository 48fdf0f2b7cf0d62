// gram_rules.hpp -- which kernel forms a Gram product U^T X (N x nb by
// N x nb, K = N) and in how many chunks of points: host code only, with no
// HIP call, so that the rules can be checked without a GPU.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace rsg {

// The products differ in their kernel, so each has its own split.
enum GramForm {
  kGramSame = 0,  // U^T U, FP64 (Gram-Schmidt)
  kGramPair = 1,  // U^T X of two blocks, FP64 (subspace_diag)
  kGramF32 = 2,   // U^T X of two FP32 blocks: SGEMMs over the chunks
};

// A split chosen by the autotuner: points per chunk, 0 = one GEMM over all of K.
struct GramSplit {
  int64_t N, nb;
  int form;
  int64_t kc;
};

// Bands per tile side of k_gram: 32 or 48, whichever pads less (48 reads
// less per product and takes ties).
inline int gram_tile(int nb) { return (nb + 47) / 48 * 48 <= (nb + 31) / 32 * 32 ? 48 : 32; }

// Where k_gram runs (us per product, against rocBLAS batched over chunks of
// points and the sum of their results): 36^3, 20 bands 13 (35), 48^3, 40
// bands 25 (52), 58^3, 77 bands 75 (184), U^T U of 72^3, 160 bands 335
// (492).  rocBLAS's tiles are 128 bands a side, so it is the faster from 97
// to 128 bands (72^3, 128: 209 against 253) and for the product of two
// different blocks above (160 bands: 492 against 584).
inline bool gram_own(int nb, int form) {
  return form != kGramF32 && (nb <= 96 || (form == kGramSame && nb > 128 && nb <= 192));
}

// Points per chunk where nothing was tuned:
// - k_gram: a block per CU, of 512 points or more (36^3, 20 bands: 13 us
//   with 91 blocks, 22 with 32, 67 with 8);
// - rocBLAS, which runs this K = N >> nb shape on a handful of output tiles:
//   at most 256 chunks of 1024 points or more up to 192 bands, one GEMM
//   above.
inline int64_t gram_default(int nb, int64_t N, int form) {
  if (!gram_own(nb, form)) return nb > 192 || N < 4096 ? 0 : std::max<int64_t>(1024, (N + 255) / 256);
  const int64_t nt = (nb + gram_tile(nb) - 1) / gram_tile(nb);
  const int64_t tiles = form == kGramSame ? nt * (nt + 1) / 2 : nt * nt;
  const int64_t nch = std::max<int64_t>(1, 256 / tiles);
  return std::max<int64_t>(512, (N + nch - 1) / nch);
}

inline int64_t gram_chunk(const std::vector<GramSplit> &tuned, int nb, int64_t N, int form) {
  for (const GramSplit &e : tuned)
    if (e.N == N && e.nb == nb && e.form == form) return e.kc;
  return gram_default(nb, N, form);
}

// What the autotuner times for a form: one GEMM, 8 to 512 chunks of at least
// 512 points, and the split used when nothing was tuned.
inline std::vector<int64_t> gram_candidates(int nb, int64_t N, int form) {
  std::vector<int64_t> c{0};
  for (int n = 8; n <= 512; n *= 2)
    if (N / n >= 512) c.push_back((N + n - 1) / n);
  const int64_t kc = gram_default(nb, N, form);
  if (kc > 0 && kc < N && std::find(c.begin(), c.end(), kc) == c.end()) c.push_back(kc);
  return c;
}

// Where both FP64 products run the same rocBLAS calls, one timing serves both.
inline bool gram_pair_timed(int nb) { return gram_own(nb, kGramSame) || gram_own(nb, kGramPair); }

// Keep the tuned splits of the FP64 products.  The FP32 product runs rocBLAS
// at every size: it takes the split of the two-block product where that was
// timed on rocBLAS too, and its own default where k_gram was timed.
inline void gram_keep(std::vector<GramSplit> &tuned, int nb, int64_t N, int64_t kc_same, int64_t kc_pair) {
  const auto put = [&](int form, int64_t kc) {
    for (GramSplit &e : tuned)
      if (e.N == N && e.nb == nb && e.form == form) {
        e.kc = kc;
        return;
      }
    tuned.push_back({N, nb, form, kc});
  };
  put(kGramSame, kc_same);
  put(kGramPair, kc_pair);
  if (!gram_own(nb, kGramPair)) put(kGramF32, kc_pair);
}

}  // namespace rsg
