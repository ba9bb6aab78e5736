// Host rules that pick a kernel's shape from the sizes of a call.  Plain C++ with no HIP in it: the
// rules are checked on the CPU over many sizes (tests/test_rules.py).
#pragma once
#include <stdint.h>

#include <algorithm>

namespace dmla {

// ---- on-the-fly forward: query rows per workgroup --------------------------------------------
struct OtfShape {
  int rows;
  double fixed_us;    // a workgroup of n key tiles takes fixed_us + n (tile_us + busy_us x), x the share
  double tile_us;     // of CUs with a workgroup
  double busy_us;
};
// Measured at 340 sizes (B * H of 8..512, 16..8192 rows and keys): the estimate below is within 4 % of each
// shape's time on average.
constexpr OtfShape kOtfShapes[] = {{512, 6.0, 2.75, 0.4}, {256, 3.7, 1.7, 0.3}, {128, 4.6, 1.25, 0.2}};
constexpr double kOtfTileBytes = 2 * 64 * 128 * 2;   // the raw K and V rows of a 64-key tile
constexpr double kOtfCacheBytes = 256e6;             // K and V past this come from HBM again for each row tile
constexpr double kOtfHbmBytesPerUs = 4.2e6;          // at this rate

// Key tiles (64 keys) of row tile qt of `rows` query rows.
inline int64_t otf_key_tiles(int rows, int64_t qt, int64_t Sq, int64_t Sk, int causal) {
  const int64_t last = std::min(Sq, (qt + 1) * rows);
  const int64_t kend = causal ? std::min(Sk, last + Sk - Sq) : Sk;
  return (std::max<int64_t>(kend, 0) + 63) / 64;
}

// Time of a call with the given shape.  One workgroup fits a CU, and row tiles start in order, the one
// with the most keys first, so a grid just past a multiple of the CU count runs another full round where
// the workgroups are equally long (non-causal, or a chunk of a long context).  Up to eight workgroups per
// CU the schedule is followed: workgroups of one row tile (of several where B * H < 8) go to the CUs
// that are free first.  Past that it is the mean load, or whole rounds: some CU runs j + 1 workgroups
// at least as long as the (j CUs)-th.
inline double otf_estimate_us(const OtfShape& s, int cus, int64_t BH, int64_t Sq, int64_t Sk, int causal) {
  constexpr int kMaxCus = 512;
  cus = std::min(std::max(cus, 1), kMaxCus);
  const int64_t nq = (Sq + s.rows - 1) / s.rows;
  const double n = (double)nq * (double)BH;
  const double tile_us = s.tile_us + s.busy_us * std::min(1.0, n / cus);
  auto len = [&](int64_t qt) { return s.fixed_us + tile_us * (double)otf_key_tiles(s.rows, qt, Sq, Sk, causal); };
  // the average row tile (at most 64 stand for all of them)
  const int64_t step = (nq + 63) / 64;
  double total = 0;
  int64_t samples = 0;
  for (int64_t qt = nq - 1; qt >= 0; qt -= step, ++samples) total += len(qt);
  const double mean = total / (double)samples;
  double us = n * mean / cus;
  if (n <= 8.0 * cus) {
    struct { double t; int64_t cus; } free_at[kMaxCus];   // CUs free from t on, earliest first
    int nf = 1;
    free_at[0] = {0.0, cus};
    const int64_t group = (8 + BH - 1) / BH;
    for (int64_t qt = nq - 1; qt >= 0; qt -= group) {
      int64_t left = BH * std::min(group, qt + 1);
      const double w = len(qt);
      while (left > 0) {
        const int64_t m = std::min(free_at[0].cus, left);
        const double t = free_at[0].t + w;
        left -= m;
        free_at[0].cus -= m;
        int i = free_at[0].cus == 0 ? 1 : 0, j = 0;   // drop the entry that is used up
        for (; i < nf && free_at[i].t < t; ++i) free_at[j++] = free_at[i];
        if (i == j) {                                 // nothing dropped: make room
          for (int k = nf; k > i; --k) free_at[k] = free_at[k - 1];
          ++nf;
        }
        free_at[j] = {t, m};
      }
    }
    us = free_at[nf - 1].t;
  } else {
    for (int64_t j = 0; j < 64 && (double)j * cus < n; ++j) us = std::max(us, (double)(j + 1) * len(nq - 1 - j * cus / BH));
  }
  if ((double)BH * (double)Sk * 512.0 > kOtfCacheBytes)
    us = std::max(us, n * (mean - s.fixed_us) / tile_us * kOtfTileBytes / kOtfHbmBytesPerUs);
  return us;
}

// Query rows per workgroup: larger tiles cost less per row (the projection is shared by more of
// them), smaller ones occupy more CUs and end sooner.  The smallest estimate wins, the larger tile on a tie.
// Measured with 512 / 256 / 128 rows: 1 x 32 x 500 causal 34.4 / 20.4 / 16.9 us, 2 x 32 x 4096 causal
// 234 / 291 / 401; non-causal 1 x 32 x 2100 109 / 133 / 150 and 1 x 32 x 1100 58 / 38 / 57 (288 workgroups
// of 128 rows on 256 CUs).  Counting rounds as fractions took the 256 rows at 1 x 32 x 2100 and the 128 at
// 1 x 32 x 1100: over 340 sizes it was up to 1.5x off the best shape and 1.3x slower than 512 rows; this
// estimate is 1.06x off at most and 0.2 % on average.
inline int otf_rows(int cus, int64_t BH, int64_t Sq, int64_t Sk, int causal) {
  int best = 0;
  double best_us = 0;
  for (const OtfShape& s : kOtfShapes) {
    const double us = otf_estimate_us(s, cus, BH, Sq, Sk, causal);
    if (best == 0 || us < best_us) {
      best = s.rows;
      best_us = us;
    }
  }
  return best;
}

}  // namespace dmla
