// hpsi_shape.hpp -- launch shapes of the H psi kernels: host code only, with
// no HIP call, so that the rules can be checked without a GPU.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <tuple>
#include <vector>

namespace rsg {

// Launch shape of the hpsi kernels for one grid and precision.  A zero ry,
// ty, zlen, chunk, bt, rx or psplit is derived per call (resolve_shape).
struct HpsiShape {
  int ry = 0;     // rows per thread (y register blocking)
  int ty = 0;     // rows per workgroup tile
  int zlen = 0;   // z-planes per workgroup
  int chunk = 0;  // bands per chunk (gather -> scatter -> stencil)
  int bt = 0;     // bands per scatter thread / 4 * bt bands per apply wave
  int order = 0;  // analytic projectors: 0 = nonlocal writes, stencil adds; 1 = stencil writes, nonlocal adds
  int rx = 0;     // x-points per stencil thread: 1, or 2 (pair kernel: FP32, Md 6, even n1, ty | n2)
  int proj = 0;   // analytic projections: 0 = per sphere segment (k_proj_m), 1 = by row tiles (k_proj_rows)
  int plds = 0;   // KiB of LDS reserved per segment-projection wave (fewer waves in flight: a smaller L2 set)
  int psplit = 0; // segment projections: pieces per segment (1, 2, 4, 8), each its own wave and partial slot
};
// pieces per segment where none are asked for
constexpr int kAutoPieces = 4;

// What the rules see of a call's grid and nonlocal operator.
struct HpsiGrid {
  int n1 = 0, n2 = 0, n3 = 0, md = 0;
  int64_t N = 0;
  bool nonlocal = false;  // a nonlocal part runs beside the stencil
  bool analytic = false;  // ... in the analytic form
  int nseg = 0;           // sphere segments of the analytic form
  int max_chunk = 0;      // bands whose projections a caller's scratch holds, 0 = any number
};

constexpr size_t kMaxDynLds = 64 * 1024;
constexpr int kCus = 256;      // compute units
constexpr int64_t kSmallCall = int64_t(1) << 20;  // points times bands below which a stencil thread takes one row
constexpr int kRunStart = 10;  // planes' worth of time a z-run's ring fill takes

inline int round64(int v) { return (v + 63) / 64 * 64; }

// Workgroup of the one-point kernel for ty tile rows: full x-rows while 512
// threads cover them, else (FP64, two rows a thread) the rows in nx equal
// parts, whose columns beside the part are halo too.
struct RowTile {
  int nx, xw, threads, halo;  // halo elements per plane
  size_t lds;
  bool fits;
};
inline RowTile row_tile(int n1, int md, int ry, int ty, size_t s) {
  RowTile r{1, n1, 0, 0, 0, false};
  if (ry < 1 || ty < ry || ty % ry || ty / ry > 512 || n1 > 512) return r;
  const int G = ty / ry;
  while (r.xw * G > 512) ++r.nx, r.xw = (n1 + r.nx - 1) / r.nx;
  const bool parts = r.nx > 1;
  r.threads = round64(r.xw * G);
  r.halo = 2 * md * (parts ? r.xw + ty : n1);
  r.lds = (2 * size_t(ty + 2 * md) * (parts ? r.xw + 2 * md : n1) + 64) * s;
  r.fits = r.lds <= kMaxDynLds &&
           (parts ? s == sizeof(double) && ry == 2 && r.halo <= 2 * r.threads : r.halo <= 4 * r.threads);
  return r;
}

// Tile rows for rows in parts: 16 to 20, with the least padding (8 to 14
// rows leave more halo, 24 and more make the parts narrow: 144^3, 300 bands
// 11.8 ms with 12 rows, 10.8 with 16, 11.9 with 24, 13.7 with 32).
inline int pick_ty_parts(int n1, int n2, int md, size_t s) {
  int best_ty = 0;
  double best = 1e300;
  for (int ty = 16; ty <= 20; ty += 2) {
    const RowTile r = row_tile(n1, md, 2, ty, s);
    if (!r.fits || r.nx == 1) continue;
    const double cost = double(r.nx) * r.xw / n1 * double((n2 + ty - 1) / ty * ty) / n2;
    if (cost < best) {
      best = cost;
      best_ty = ty;
    }
  }
  return best_ty;
}

// Tile rows per workgroup for ry rows per thread: balance idle lanes, the
// partial last tile and the halo rows each plane re-reads.  FP64 with two
// rows a thread spills beyond two halo elements per thread (75^3, 60 bands:
// H psi 592 to 657 us there, 403 with 12 rows and 1.8): only if nothing
// else fits.
inline int pick_ty(int n1, int n2, int md, int ry, size_t s) {
  int best_ty = 0;
  double best = 1e300;
  for (int G = 1; n1 * G <= 512; ++G) {
    const int ty = G * ry;
    if (ty > ((n2 + ry - 1) / ry) * ry) break;
    if ((2 * size_t(ty + 2 * md) * n1 + 64) * s > kMaxDynLds) break;
    const int th = n1 * G;
    if (2 * md * n1 > 4 * round64(th)) continue;
    const int tiles = (n2 + ty - 1) / ty;
    const double cost = double(round64(th)) / th * double(tiles * ty) / n2 *
                        (1.0 + 0.5 * 2.0 * md / ty) * (th < 128 ? 2.0 : 1.0) *
                        (s == sizeof(double) && ry == 2 && 2 * md * n1 > 2 * round64(th) ? 4.0 : 1.0);
    if (cost < best) {
      best = cost;
      best_ty = ty;
    }
  }
  return best_ty;
}

// Pair kernel (two x-points per thread): tile rows for ry rows per
// thread among the divisors of n2, same cost model as pick_ty.
constexpr int kPairMd = 6;

inline bool pair_fits(int n1, int n2, int md, int ry, int ty, size_t s) {
  if (md != kPairMd || n1 % 2 || n1 < 2 * md || ty <= 0 || ty % ry || n2 % ty) return false;
  const int th = round64((n1 / 2) * (ty / ry));
  const size_t lds = (2 * size_t(ty + 2 * md) * (n1 + 2 * md) + 128) * s;
  return th <= 512 && lds <= kMaxDynLds && 2 * md * (n1 / 2) <= 4 * th;
}

inline int pick_ty_pair(int n1, int n2, int md, int ry, size_t s) {
  int best_ty = 0;
  double best = 1e300;
  for (int ty = ry; ty <= n2; ty += ry) {
    if (!pair_fits(n1, n2, md, ry, ty, s)) continue;
    const int th = (n1 / 2) * (ty / ry);
    const double cost = double(round64(th)) / th * (1.0 + 0.5 * 2.0 * md / ty) * (th < 128 ? 2.0 : 1.0);
    if (cost < best) {
      best = cost;
      best_ty = ty;
    }
  }
  return best_ty;
}

// Complete a launch shape: fields left at zero are derived from the grid,
// the precision and the number of bands of the call.  Where the lines lie
// (us per H psi call, analytic projectors):
// - rows per thread: two share their y-window, but in FP64 with more than
//   two halo elements per thread the registers no longer hold the prefetch
//   (108^3, 480 bands: 11740 with two full rows, 7060 with one; 72^3, 160
//   bands, two halo elements: 604 with two, 660 with one); there the rows go
//   in parts where n1 is even (k_stencil's figures), and full rows stay for
//   an odd n1, whose parts start misaligned (99^3, 240 bands: 3782 with full
//   rows, 4001 with parts; 111 x 107 x 101: 4638 and 4762).  Parts of 16 and
//   more rows pay while they pad few of them: up to 1.4 padded rows (96 x 23
//   x 60, 226 bands, 1.39: 917 in parts, 958 with one row; 108 x 13 x 72, 296
//   bands, 1.23: 924 and 972), not above (108 x 22 x 72, 175 bands, 1.45: 929
//   and 888; 144 x 9 x 72, 321 bands, 1.78: 1212 and 1119).  Full rows, two a
//   thread, pad up to 1.3 (75 x 38 x 70, 150 bands, 1.26: 424 with two, 447
//   with one); above, one row a thread where its tile stages no more than two
//   halo elements a thread (78 x 27 x 60, 100 and 250 bands, 1.33: 203 and
//   386 with one, 231 and 397 with two, 250 and 445 in parts; 72 x 18 x 72,
//   100 bands: 307, 361, 401), else still two (84 x 25 x 60, 250 bands, 1.44:
//   847 with two, 919 with one, 943 in parts);
//   a call of few points is a chain of latencies, shorter with one row a
//   thread: the line at 2^20 points times bands lies where the two cross or
//   are level on most grids (36^3, 20 bands 30.9 with one row, 33.6 with two,
//   48 bands 52.1 and 53.3; 40^3, 12 bands 30.8 and 31.3, 40 bands 55.8 and
//   51.4; 72^3, 1 band 56.2 and 58.5, 10 bands 81.4 and 78.6; 48^3 is an
//   exception, 9 bands 36.2 and 32.4);
// - FP32 takes the pair kernel where it fits (72^3, 160 bands: 330 against
//   395; 108^3, 480 bands: 3800 against 4400);
// - the analytic form runs all bands at once (72^3, 160 bands FP64 in
//   chunks of 22: 1160, of 80: 709, whole: 618), its partial projections
//   within 1 GiB;
// - four pieces per segment (72^3 FP64, whole: 660 with one, 618 with four;
//   36^3, 20 bands: 52 and 41);
// - bands per apply wave: the least padding, then the most bands (160
//   bands: 80 a wave 604, 32 a wave 620);
// - z-runs: a run of zlen planes costs zlen + kRunStart planes' time (ring
//   fill; 40^3, 27 bands: stencil 44, 27, 18 us in runs of 40, 20, 10), and
//   the blocks go in rounds of as many as the CUs hold at once; the number
//   of runs with the least rounds x run cost is taken (40^3, 27 bands: 216
//   blocks 48.5, 270 blocks, so two rounds, 59.0; 24^3, 12 bands: one run
//   34, six 26).
// A shape with ty == 0 says that no kernel takes the grid's rows (the caller
// refuses the call): full rows end at 170 points with md 6, where three tile
// rows are the least that stage their halo and the most that 512 threads
// cover, and only the FP64 kernel takes rows in parts.
inline HpsiShape resolve_shape(const HpsiGrid &gr, const HpsiShape &in, size_t s, int nb) {
  HpsiShape sh = in;
  const int n1 = gr.n1, n2 = gr.n2, n3 = gr.n3;
  const bool auto_ry = sh.ry < 1 || sh.ry > 2;
  const auto one_fits = [&](int ry) { return row_tile(n1, gr.md, ry, sh.ty, s).fits; };
  const auto two_fits = [&](int ry) { return pair_fits(n1, n2, gr.md, ry, sh.ty, s); };
  // tile rows that the caller gives stay where a kernel takes them, with the
  // rows and points a thread that fit them
  const bool one = auto_ry ? one_fits(2) || one_fits(1) : one_fits(sh.ry);
  const bool two = auto_ry ? two_fits(2) || two_fits(1) : two_fits(sh.ry);
  if (sh.rx == 0) sh.rx = s == sizeof(float) && (two || !one) ? 2 : 1;
  if (sh.rx == 2 && s == sizeof(float)) {  // pair kernel: FP32 only; else the one-point kernel
    if (auto_ry) sh.ry = two && !two_fits(2) ? 1 : 2;
    if (!two) {
      int ty = pick_ty_pair(n1, n2, gr.md, sh.ry, s);
      if (ty == 0 && auto_ry) ty = pick_ty_pair(n1, n2, gr.md, sh.ry = 1, s);
      if (ty == 0) sh.rx = 1;
      else sh.ty = ty;
    }
  } else {
    sh.rx = 1;
  }
  if (sh.rx == 1 && auto_ry) {
    sh.ry = one && !one_fits(2) ? 1 : 2;
    if (s == sizeof(double) && sh.ry == 2) {
      const int ty = one ? sh.ty : pick_ty(n1, n2, gr.md, 2, s);
      const RowTile rt = row_tile(n1, gr.md, 2, ty, s);
      const bool slow = ty == 0 || (rt.nx == 1 && rt.halo > 2 * rt.threads);  // full rows whose halo spills
      if (one) {
        if ((slow || gr.N * int64_t(nb) < kSmallCall) && one_fits(1)) sh.ry = 1;
      } else if (slow) {
        const int part = ty && n1 % 2 == 0 ? pick_ty_parts(n1, n2, gr.md, s) : 0;
        if (part && (n2 + part - 1) / part * part <= 1.4 * n2) sh.ty = part;
        else sh.ry = 1;
      } else if ((n2 + ty - 1) / ty * ty > 1.3 * n2) {
        const RowTile r1 = row_tile(n1, gr.md, 1, pick_ty(n1, n2, gr.md, 1, s), s);
        if (r1.fits && r1.halo <= 2 * r1.threads) sh.ry = 1;
      } else if (gr.N * int64_t(nb) < kSmallCall) {
        sh.ry = 1;
      }
    }
  }
  const auto ty_bad = [&]() { return !one_fits(sh.ry); };
  if (sh.rx == 1 && ty_bad()) {
    sh.ty = pick_ty(n1, n2, gr.md, sh.ry, s);
    if (sh.ty == 0) {
      sh.ry = 1;
      sh.ty = pick_ty(n1, n2, gr.md, 1, s);
    }
    if (sh.ty == 0 && s == sizeof(double)) {  // rows too long for whole ones, of any parity
      sh.ry = 2;
      sh.ty = pick_ty_parts(n1, n2, gr.md, s);
    }
  }
  if (sh.ty == 0) return sh;  // no tile fits
  if (sh.psplit != 1 && sh.psplit != 2 && sh.psplit != 4 && sh.psplit != 8) sh.psplit = kAutoPieces;
  if (sh.chunk <= 0) {
    sh.chunk = nb;
    if (gr.analytic) {
      const size_t per_band = size_t(std::max(1, gr.nseg)) * sh.psplit * 4 * s;
      sh.chunk = int(std::min<size_t>(size_t(nb), std::max<size_t>(1, (size_t(1) << 30) / per_band)));
      const int nch = (nb + sh.chunk - 1) / sh.chunk;
      sh.chunk = (nb + nch - 1) / nch;  // chunks of equal size
    } else if (gr.nonlocal) {
      // table form: psi + H psi of one chunk within ~128 MB of Infinity Cache
      sh.chunk = int(std::max<size_t>(1, (size_t(64) << 20) / (size_t(gr.N) * s)));
    }
  }
  sh.chunk = std::max(1, std::min(sh.chunk, nb));
  if (gr.max_chunk > 0 && sh.chunk > gr.max_chunk) {  // before z-runs and apply waves, which follow from it
    const int nch = (nb + gr.max_chunk - 1) / gr.max_chunk;
    sh.chunk = (nb + nch - 1) / nch;
  }
  if (sh.zlen <= 0) {
    int tiles = (n2 + sh.ty - 1) / sh.ty, waves, per_cu;
    if (sh.rx == 2) {
      waves = round64((n1 / 2) * (sh.ty / sh.ry)) / 64;
      per_cu = sh.ry == 1 ? 12 : 8;
    } else {
      const RowTile rt = row_tile(n1, gr.md, sh.ry, sh.ty, s);
      tiles *= rt.nx;
      waves = std::max(1, rt.threads / 64);
      per_cu = sh.ry == 1 && rt.halo <= 2 * rt.threads ? 12 : 8;
    }
    const int64_t slots = int64_t(kCus) * std::max(1, per_cu / std::max(1, waves)), blocks = int64_t(tiles) * sh.chunk;
    int64_t best = 0;
    for (int zr = 1; zr <= std::max(1, n3 / 4); ++zr) {
      const int zl = (n3 + zr - 1) / zr;
      const int64_t cost = (blocks * ((n3 + zl - 1) / zl) + slots - 1) / slots * (zl + kRunStart);
      if (!best || cost < best) {
        best = cost;
        sh.zlen = zl;
      }
      if (blocks * zr >= 8 * slots) break;
    }
  }
  sh.zlen = std::max(1, std::min(sh.zlen, n3));
  if (sh.bt != 4 && sh.bt != 8 && sh.bt != 16 && sh.bt != 20 && sh.bt != 32) {
    sh.bt = 8;
    if (gr.analytic) {
      int best = 0;
      for (int bt : {20, 16, 8, 4}) {
        const int pad = (sh.chunk + 4 * bt - 1) / (4 * bt) * (4 * bt);
        if (!best || pad < best) {
          best = pad;
          sh.bt = bt;
        }
      }
    }
  }
  if (sh.order != 0 && sh.order != 1) sh.order = 0;
  if (sh.proj < 0 || sh.proj > 2) sh.proj = 0;
  if (sh.plds < 0 || sh.plds > 64) sh.plds = 0;
  return sh;
}

inline std::tuple<int, int, int, int, int, int, int, int, int, int> shape_key(const HpsiShape &h) {
  return {h.ry, h.ty, h.zlen, h.chunk, h.bt, h.order, h.rx, h.proj, h.plds, h.psplit};
}

// Coordinate search over the launch shape for nb bands of s-byte values, from
// the derived shape on.  time(shape, ms) gives 0, or an error code that ends
// the search, or a negative value where the shape does not fit;
// rows_ready() makes the row tiles of the second projection form and says
// whether there are any.  best and tbest receive the fastest shape and its
// time.  No shape is tried twice but the derived one: its first timing may
// run at the clocks of an idle GPU (72^3, 160 bands FP64 in a new process:
// one row a thread, 682 us a call, was kept over the derived 596), so it is
// timed again after the first candidates.  A candidate that beats the best
// is timed again beside it and has to win again: otherwise one timing of 20
// candidates that is 1 percent low moves the shape (72^3, 160 bands: 64
// bands per apply wave, 604, for 80, 598).
//
// Each field's whole range is timed, also where the derived shape already
// holds the value that is fastest on large grids: 36^3, 20 bands FP32 run
// 28 us with one point and one row a thread, 37 with the pair kernel.
template <typename Time, typename Rows>
int search_shape(const HpsiGrid &gr, size_t s, int nb, Time time, Rows rows_ready, HpsiShape &best, float &tbest) {
  const int n2 = gr.n2;
  std::vector<HpsiShape> timed;
  best = resolve_shape(gr, HpsiShape(), s, nb);
  int rc = time(best, tbest);
  if (rc) return rc;
  timed.push_back(best);
  auto consider = [&](const HpsiShape &in) {
    if (rc) return;
    const HpsiShape cand = resolve_shape(gr, in, s, nb);
    if (cand.ty == 0) return;
    for (const HpsiShape &h : timed)
      if (shape_key(h) == shape_key(cand)) return;
    timed.push_back(cand);
    float t = 0.f, again = 0.f;
    const int r = time(cand, t);
    if (r < 0) return;  // does not fit this grid
    rc = r;
    if (rc || t >= tbest) return;
    // both once more: a difference of the timer's noise is no reason to move
    if ((rc = time(best, again))) return;
    tbest = std::min(tbest, again);
    if ((rc = time(cand, again))) return;
    if (again < tbest) {
      tbest = again;
      best = cand;
    }
  };
  for (int rx = 1; rx <= (s == sizeof(float) ? 2 : 1); ++rx)
    for (int ry = 1; ry <= 2; ++ry) {
      HpsiShape c = best;
      c.rx = rx;
      c.ry = ry;
      c.ty = 0;
      c.zlen = 0;
      consider(c);
    }
  if (!rc) {
    float t = 0.f;
    rc = time(timed.front(), t);
    if (rc) return rc;
    if (t < tbest) {
      tbest = t;
      best = timed.front();
    }
  }
  if (best.rx == 2) {  // neighbouring divisors of n2
    int lo = 0, hi = 0;
    for (int t = best.ty - best.ry; t > 0 && !lo; t -= best.ry)
      if (pair_fits(gr.n1, n2, gr.md, best.ry, t, s)) lo = t;
    for (int t = best.ty + best.ry; t <= n2 && !hi; t += best.ry)
      if (pair_fits(gr.n1, n2, gr.md, best.ry, t, s)) hi = t;
    for (int t : {lo, hi}) {
      HpsiShape c = best;
      c.ty = t;
      c.zlen = 0;
      if (t > 0) consider(c);
    }
  } else {
    for (int f : {-2, -1, 1, 2}) {
      HpsiShape c = best;
      c.ty = best.ty + f * best.ry;
      c.zlen = 0;
      if (c.ty > 0) consider(c);
    }
  }
  if (gr.nonlocal) {
    for (int f : {2, 4}) {
      HpsiShape c = best;
      c.chunk = std::min(nb, best.chunk * f);
      c.zlen = 0;
      consider(c);
    }
    HpsiShape ch = best;
    ch.chunk = std::max(1, best.chunk / 2);
    ch.zlen = 0;
    consider(ch);
    for (int bt : {4, 8, 16, 20, 32}) {
      HpsiShape c = best;
      c.bt = bt;
      consider(c);
    }
    if (gr.analytic) {
      HpsiShape c = best;
      c.order = 1 - best.order;
      consider(c);
      if (rows_ready()) {
        HpsiShape pj = best;
        pj.proj = best.proj == 1 ? 0 : 1;
        consider(pj);
      }
      {  // segment projections with 64 bands per wave
        HpsiShape pj = best;
        pj.proj = best.proj == 2 ? 0 : 2;
        consider(pj);
      }
      if (best.proj != 1)  // fewer segment waves in flight per CU
        for (int kib : {4, 8, 16, 32}) {
          HpsiShape pl = best;
          pl.plds = kib;
          consider(pl);
        }
      if (best.proj != 1)  // segments in pieces: chords shared by two spheres read close in time
        for (int np : {1, 2, 4, 8}) {
          HpsiShape ps = best;
          ps.psplit = np;
          consider(ps);
        }
      for (int f : {4, 8}) {  // smaller chunks keep psi and H psi in the Infinity Cache
        HpsiShape d = best;
        d.chunk = std::max(1, nb / f);
        d.zlen = 0;
        consider(d);
      }
    }
  }
  for (int zf : {2, 4}) {
    HpsiShape c = best;
    c.zlen = std::max(1, best.zlen / zf);
    consider(c);
  }
  {
    HpsiShape c = best;
    c.zlen = gr.n3;
    consider(c);
  }
  return rc;
}

}  // namespace rsg
