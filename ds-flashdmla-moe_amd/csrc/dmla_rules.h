// Host rules that pick a kernel's shape from the sizes of a call.  Plain C++ with no HIP in it: the
// rules are checked on the CPU over many sizes (tests/test_rules.py).
#pragma once
#include <stdint.h>

#include <algorithm>
#include <cmath>

namespace dmla {

// ---- on-the-fly forward: query rows per workgroup --------------------------------------------
struct OtfShape {
  int rows;
  double fixed_us;    // a workgroup of n key tiles takes fixed_us + n (tile_us + busy_us x), x the share
  double tile_us;     // of CUs with a workgroup
  double busy_us;
};
// Measured at 510 sizes (B * H of 8..512, 16..8192 rows and keys): the estimate below is within 4 % of each
// shape's time on average.
constexpr OtfShape kOtfShapes[] = {{512, 6.0, 2.75, 0.4}, {256, 3.7, 1.7, 0.3}, {128, 4.6, 1.25, 0.2}};
constexpr double kOtfTileBytes = 2 * 64 * 128 * 2;   // the raw K and V rows of a 64-key tile
// K and V of more than kOtfCacheBytes come from HBM again, at kOtfHbmBytesPerUs, for each set of row
// tiles of a head that run at once.
constexpr double kOtfCacheBytes = 256e6;
constexpr double kOtfHbmBytesPerUs = 4.8e6;

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
  if ((double)BH * (double)Sk * 512.0 > kOtfCacheBytes) {
    const double together = std::max(1.0, std::min((double)nq, cus / (double)BH));
    const double hbm_us = n * (mean - s.fixed_us) / tile_us * kOtfTileBytes / together / kOtfHbmBytesPerUs;
    us = std::sqrt(us * us + hbm_us * hbm_us);   // neither hides the other whole
  }
  return us;
}

// Query rows per workgroup: larger tiles cost less per row (the projection is shared by more of
// them), smaller ones occupy more CUs and end sooner.  The smallest estimate wins, the larger tile on a
// tie; 512 rows keep 5 %, about what the estimates are off.
// Measured with 512 / 256 / 128 rows: 1 x 32 x 500 causal 34.4 / 20.4 / 16.9 us, 2 x 32 x 4096 causal
// 234 / 291 / 401; non-causal 1 x 32 x 2100 109 / 133 / 150 and 1 x 32 x 1100 58 / 38 / 57 (288 workgroups
// of 128 rows on 256 CUs).  Counting rounds as fractions took the 256 rows at 1 x 32 x 2100 and the 128 at
// 1 x 32 x 1100: over 510 sizes it was up to 1.5x off the best shape and 1.3x slower than 512 rows; this
// choice is 4.5 % off at most, 0.2 % on average, and at most 2.6 % slower than 512 rows.
inline int otf_rows(int cus, int64_t BH, int64_t Sq, int64_t Sk, int causal) {
  int best = 0;
  double best_us = 0;
  for (const OtfShape& s : kOtfShapes) {
    const double us = (s.rows == 512 ? 0.95 : 1.0) * otf_estimate_us(s, cus, BH, Sq, Sk, causal);
    if (best == 0 || us < best_us) {
      best = s.rows;
      best_us = us;
    }
  }
  return best;
}

// ---- cache-latent prefill: key ranges split over workgroups -----------------------------------
constexpr int kPrefillRows = 64, kPrefillKeys = 32;   // rows of a row tile, keys of a key tile
constexpr int kPrefillMaxParts = 32;                  // key ranges of a row tile

struct PrefillSplit {
  int n_layers;                           // most parts of a row tile; 1: no split
  int first_rt[kPrefillMaxParts];         // layer j holds part j of the row tiles from first_rt[j] on
  int layer_base[kPrefillMaxParts + 1];   // row tiles (of one batch element) in the layers before j
  int64_t workgroups() const { return layer_base[n_layers]; }   // per batch element
  // Partials, per batch element: the row tiles with one part (those before first_rt[1]) write none.
  int64_t slots() const { return n_layers > 1 ? layer_base[n_layers] - first_rt[1] : 0; }
};

inline int64_t prefill_key_tiles(int64_t H, int64_t Sq, int64_t Sk, int causal, int64_t rt) {
  const int64_t last_pos = (std::min<int64_t>((rt + 1) * kPrefillRows, H * Sq) - 1) / H;
  const int64_t kend = causal ? std::min(Sk, last_pos + 1 + (Sk - Sq)) : Sk;
  return (std::max<int64_t>(kend, 0) + kPrefillKeys - 1) / kPrefillKeys;
}

// Whether and how to split the key ranges of a prefill.  A workgroup of n key tiles takes about
// kFixedUs + n kTileUs (measured: prologue and epilogue, and the tile loop), a merge kMergeUs,
// kMergePartUs per part of a row and 4 KB of traffic per row and part at ~4 TB/s.  Unsplit, some CU
// runs j + 1 workgroups at least as long as the (j CUs)-th longest.  Only calls with at most four
// row tiles per CU are considered: past that the grid balances itself.  Measured sides (16 heads,
// causal): 512 of 8192 positions 201 us unsplit, 135 in two parts, 156 in three; 4 of 8000 192 us
// unsplit, 32 in 16 parts; 1024 of 1024 (row tiles of 1 to 32 tiles, one per CU) 32 us unsplit, 43
// with the longest cut in two.  A split has at most kSplitWgsPerCu workgroups per CU, which caps the
// workspace at 16 x 132 KB per CU (539 MB on 256 CUs; 5 x 5 heads, 2047 of 137187 positions took 842 MB in
// 6400 workgroups).  More of them hardly even anything out: by the estimate the bound costs nothing up
// to 8192 keys, and that call takes 13.9 ms in 4000 against 14.1 in 6400, 15.6 in 1600 and 18.1 unsplit.
constexpr double kFixedUs = 5.5, kTileUs = 0.85, kMergeUs = 4.0, kMergePartUs = 0.4;
constexpr int64_t kSplitWgsPerCu = 16;
inline PrefillSplit prefill_split(int64_t cus, int64_t B, int64_t H, int64_t Sq, int64_t Sk, int causal) {
  PrefillSplit sp = {};
  const int64_t n_rt = (H * Sq + kPrefillRows - 1) / kPrefillRows;
  sp.n_layers = 1;
  sp.layer_base[1] = (int)n_rt;
  if (n_rt * B > 4 * cus) return sp;
  auto tiles = [&](int64_t rt) { return prefill_key_tiles(H, Sq, Sk, causal, rt); };
  const int64_t nmax = tiles(n_rt - 1);
  // At most 64 row tiles stand for all of them, their tiles counted once: a call makes this plan twice,
  // for the workspace query and for the launch (512 of 8192 positions: 7.1 -> 2.4 us on one host).
  const int64_t step = (n_rt + 63) / 64;
  int n_at[64], samples = 0;
  double total = 0;
  for (int64_t rt = n_rt - 1; rt >= 0; rt -= step) total += n_at[samples++] = (int)tiles(rt);
  const double mean = total / samples;
  double best = 0;
  for (int64_t j = 0; j * cus < n_rt * B; ++j)
    best = std::max(best, (double)(j + 1) * (kFixedUs + kTileUs * (double)tiles(n_rt - 1 - j * cus / B)));
  best = 0.92 * std::max(best, (double)(n_rt * B) * (kFixedUs + kTileUs * mean) / (double)cus);
  int64_t best_t = 0;
  static constexpr int kTry[] = {2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32};
  for (int s : kTry) {
    const int t = (int)((nmax + s - 1) / s);
    if (t < 4) break;
    int parts = 0, merged = 0;
    for (int i = 0; i < samples; ++i) {
      const int np = n_at[i] <= t ? 1 : (n_at[i] + t - 1) / t;
      parts += np;
      if (np > 1) merged += np;
    }
    const double scale = (double)n_rt * (double)B / samples;
    const double wgs = parts * scale;
    if (wgs > (double)(kSplitWgsPerCu * cus)) break;
    const double rounds = std::max(1.0, std::ceil(wgs / (double)cus - 0.01));
    const double part_us = kFixedUs + kTileUs * mean * samples / parts;
    const double us = std::max(kFixedUs + kTileUs * (double)t, rounds * part_us) + kMergeUs + kMergePartUs * (double)s +
                      merged * scale * kPrefillRows * 4096.0 / 4e6;
    if (us < best) { best = us; best_t = t; }
  }
  if (best_t == 0) return sp;
  const int64_t most = kSplitWgsPerCu * cus / B;   // workgroups per batch element
  do {
    sp.n_layers = (int)std::min<int64_t>((nmax + best_t - 1) / best_t, kPrefillMaxParts);
    int64_t base = 0;
    for (int j = 0; j < sp.n_layers; ++j) {
      int64_t lo = 0, hi = n_rt;   // first row tile with more than j parts: tiles > j best_t (all have part 0)
      while (j > 0 && lo < hi) {
        const int64_t mid = (lo + hi) / 2;
        if (tiles(mid) > j * best_t) hi = mid; else lo = mid + 1;
      }
      sp.first_rt[j] = (int)lo;
      sp.layer_base[j] = (int)base;
      base += n_rt - lo;
    }
    sp.layer_base[sp.n_layers] = (int)base;
    best_t += (best_t + 15) / 16;
  } while (sp.workgroups() > most && sp.n_layers > 1);   // where the samples stood for too few parts
  return sp;
}

}  // namespace dmla
