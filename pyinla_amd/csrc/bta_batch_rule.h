// How the problems of a batched factorization share the device: an estimate of a
// block step's time, and the number of problems side by side that it finds
// fastest.  Plain host code.
#pragma once
#include <algorithm>
#include <cmath>
#include <vector>

namespace bta {

// A problem as the rule sees it: blocks, and 64-wide tile columns of one.
struct BatchShape {
  int n, nT;
};

// One workgroup per CU (else two): its chain and helpers do not share a CU, but
// there are half as many helpers.  Measured on MI355X, us per block step of equal
// problems, one / two:
//   nT = 4    5 problems 69 / 70,  9 74 / 70, 12 84 / 72, 18 93 / 77
//   nT = 8    4 129 / 130,  8 150 / 161,  9 153 / 144, 14 219 / 187, 18 324 / 216
//   nT = 13   4 219 / 245,  6 283 / 290,  9 421 / 360
//   nT = 19   2 300 / 334,  3 391 / 374,  4 506 / 459
//   nT = 25   1 360 / 391,  2 532 / 537,  3 820 / 697
//   nT = 32   1 546 / 554,  2 1080 / 950;  nT = 40  1 928 / 888
// so one is the better where its helpers, at 3.3 us per nT^3 and problem, take no
// longer than a chain of 15.2 us per tile column, and a problem has 28 of them or
// more (fewer fall behind the chain; nT = 2 needs 14: 41 / 45 with 10 problems).
inline bool step_fits_one(const std::vector<int>& nT, int cus) {
  const int np = (int)nT.size(), h = cus / np - 1, longest = *std::max_element(nT.begin(), nT.end());
  double work = 0.0;
  for (const int t : nT) work += (double)t * t * t;
  return h >= std::min(28, 7 * longest) && 3.3 * work <= 15.2 * longest * h * np;
}

// A block step in us, launch included.  The longest chain takes 13.9 us per tile
// column.  The helpers' work is nT^3 for each problem: 3.4 us of one helper that
// has its CU to itself, 7.0 of one that shares it (two per problem, with its chain's
// own slots four, are busy for the chain alone), and up to 9 once the exchange buffers
// of the problems side by side ((2 nT + 1) nT tiles of 32 KB each) outgrow half of the
// 256 MB last-level cache.  The two overlap but for the waits at the start and the
// end of a panel, for which the root of the squares stands.  Within 25 % of 160
// measured steps, 1 to 20 equal problems of nT = 2 .. 40; us at nT = 32, measured /
// estimated: 1 problem 547 / 632, 2 953 / 1030, 3 1459 / 1594, 6 3681 / 3428, 18
// 12766 / 11909.
inline double step_time(const std::vector<int>& nT, int cus, int cap) {
  double work = 0.0, bytes = 0.0;
  for (const int t : nT) {
    work += (double)t * t * t;
    bytes += 32768.0 * (2 * t + 1) * t;
  }
  const int np = (int)nT.size();
  const double chain = 13.9 * *std::max_element(nT.begin(), nT.end()) + 12.0;
  double helpers;
  if (step_fits_one(nT, cus)) helpers = 3.4 * work / std::max(1, cus - np);
  else helpers = 7.0 * (1.0 + 0.3 * std::max(0.0, 1.0 - 130e6 / bytes)) * work / std::max(1, cap - 4 * np);
  return std::hypot(chain, helpers);
}

// Problems per wave, at most `most`: the number whose waves take the least by the
// estimate; ps longest first.  Finite-difference stencil of 18 problems, nt = 16,
// in ms as waves of 6, 9, 18: b = 120 5.5, 4.9, 4.4; b = 480 11.0, 9.8, 8.4; b =
// 840 21.7, 20.0, 21.6.  18 problems of b = 2040: 8.6 ms per block step as waves of
// 2, 8.8 of 3, 11.0 of 6, 12.8 in one.
inline int pick_lanes(const std::vector<BatchShape>& ps, int most, int cus, int cap) {
  const int np = (int)ps.size();
  int best = 1;
  double best_t = 0.0;
  for (int nl = 1; nl <= std::min(np, most) && cap / nl - 1 >= 1; ++nl) {
    double t = 0.0;
    for (int w0 = 0; w0 < np; w0 += nl)
      for (int i = 0; i < ps[w0].n;) {
        std::vector<int> nts;
        int until = 1 << 30;
        for (int q = w0; q < std::min(np, w0 + nl); ++q)
          if (i < ps[q].n) {
            nts.push_back(ps[q].nT);
            until = std::min(until, ps[q].n);
          }
        t += (until - i) * step_time(nts, cus, cap);
        i = until;
      }
    if (nl == 1 || t < best_t) {
      best = nl;
      best_t = t;
    }
  }
  return best;
}

}  // namespace bta
