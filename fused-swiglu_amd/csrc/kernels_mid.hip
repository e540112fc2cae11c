// Plans of the producer / consumer kernel (mid_kernel.h): which tile, pieces and K parts a call takes, by an estimate of their times.
#include <math.h>
#include <stdio.h>

#include "mid_kernel.h"

namespace fsw {

namespace {

constexpr int kNumTiles = sizeof(kMidTiles) / sizeof(kMidTiles[0]);
struct TileSet {
  bool v[kNumTiles];
  bool operator[](int i) const { return v[i]; }
};
// whether there is a tile of as many weight rows and 32 activation rows fewer
const TileSet kNarrower = [] {
  TileSet s;
  for (int i = 0; i < kNumTiles; ++i) {
    s.v[i] = false;
    for (int u = 0; u < kNumTiles; ++u) s.v[i] |= kMidTiles[u].fp == kMidTiles[i].fp && kMidTiles[u].fq == kMidTiles[i].fq - 1;
  }
  return s;
}();

// Estimated time, us, of one launch (and the summing kernel of a split one). The coefficients were fitted to 2300 timings of 230 problems
// (gate/up and down, 1 .. 900 rows, d 1024 .. 8192, aligned and ragged rows, weights from memory) while weight and activation lines shared a
// ring and were asked for in turn. For the kernel as it is: 4.9 % rms and no bias over 1039 chosen plans of up to 1100 rows, worst where they
// hold 129 .. 256 rows of a down projection (aligned 13 % rms, 8 % too low on average) or more than 256 (5 and 8 % too high, aligned and
// ragged); the gate/up tile it picks is 1.0 % slower than the best whole one on average (110 problems of 20 .. 700 rows; worst 1.155: 7392 x
// 1472 208 rows 13.5 on 64 x 128, 11.7 on 96 x 96). It knows neither the depth of the rings nor pairs. A K tile of 64 costs the copies of its
// weight and activation rows (0.00256 us = 128 bytes at 50 bytes per ns, which 0.672 and 0.464 scale) or the LDS reads and MFMAs, whichever
// is more, plus a part of the other; a part that fills the chip shares HBM; a second round overlaps with the first where it is partly filled.
double mid_time(int np, int nq, int k, bool ragged, const MidTile& t, int step, int splits) {
  const int tq = (nq + 32 * t.fq - 1) / (32 * t.fq);
  const long long tp = (np + step - 1) / step;
  const long long wgs = tp * tq * splits;
  const int kt = ((k + 63) / 64 + splits - 1) / splits;
  const int rows = nq < 32 * t.fq ? nq : 32 * t.fq;
  double copy = (0.672 * step + 0.464 * rows) * 0.00256;
  if (wgs >= 200) copy += 0.153 * 0.00256 * step / tq;
  const double mul = 0.0227 * (t.fp + t.fq) + 0.01178 * t.fp * t.fq;
  const double tile = (copy > mul ? copy + 0.397 * mul : mul + 0.397 * copy) + 0.05;
  const double rounds = wgs <= 256 ? 1.0 : 0.787 * (double)((wgs + 255) / 256) + 0.213 * (double)wgs / 256.0;
  double us = rounds * (kt + 2.36 + (ragged ? 1.0 : 0.0)) * tile;
  const double hbm = 2.0 * np * (double)k / 7.305e6;
  us = us * us;
  us = sqrt(sqrt(us * us + hbm * hbm * hbm * hbm)) + 3.12;
  if (splits > 1) us += 1.19 + 0.078 * splits + 8.0 * splits * (double)nq * np / 4.53e6;
  return us;
}

}  // namespace

static MidPlan find_plan(bool gated, int np, int nq, int k, bool ragged, int splits, int max_splits) {
  MidPlan best = {-1, 0, 1, 0.0};
  const int q32 = (nq + 31) / 32;
  for (int tile = 0; tile < kNumTiles; ++tile) {
    const MidTile& t = kMidTiles[tile];
    const int tq = (q32 + t.fq - 1) / t.fq;
    if (t.fq > 1 && (q32 + t.fq - 2) / (t.fq - 1) == tq) {
      // a narrower tile needs no more columns of tiles: this one holds padding only
      if (kNarrower[tile]) continue;
    }
    const int full = 32 * t.fp;
    const long long tp = (np + full - 1) / full;
    int steps[2] = {full, 0};
    const long long rounds = (tp * tq + 255) / 256;
    // As many pieces as whole rounds hold. Aligned 128-row tiles of up to 64 activation rows stay whole where they leave less than an
    // eighth of a round empty: the pieces' wasted MFMA and LDS work costs what those compute units give, and K is then walked from the same
    // start (mid_kernel's `rot`) for all these row counts. us, pieces -> whole: 28672 x 4096 (224 tiles) 16 rows 37.1 -> 36.5, 48 rows 38.4
    // -> 37.9; 28928 x 5568 (226) 11 rows 53.3 -> 51.2; 29056 x 5760 (227) 40 rows 53.7 -> 55.0. With fewer tiles, 27648 x 5120 (216), 16
    // rows 45.2 whole, 43.9 in pieces, 48 rows 51.4 and 49.7.
    const bool whole = !ragged && nq <= 64 && t.fp == 4 && 8 * tp >= 7 * 256 * rounds;
    if (gated && tp * tq <= 1024 && !whole) {
      const long long pieces = rounds * 256 / tq;
      const int step = (int)(((np + pieces - 1) / pieces + 7) / 8 * 8);
      if (step < full && step > full - 32) steps[1] = step;
    }
    for (int s = 0; s < 2 && steps[s] > 0; ++s) {
      const long long tps = (np + steps[s] - 1) / steps[s];
      int sps[3] = {1, 0, 0};
      if (splits > 0) {
        sps[0] = splits;
      } else {
        const int deep = k / 256 < 16 ? k / 256 : 16;
        for (int r = 1; r <= 2; ++r) {
          long long sp = 256LL * r / (tps * tq);
          if (sp > deep) sp = deep;
          if (sp > max_splits) sp = max_splits;
          if (sp > 1 && 4.0 * sp * (double)nq * np <= 256e6 && (r == 1 || sp != sps[1])) sps[r] = (int)sp;
        }
      }
      for (int i = 0; i < 3; ++i) {
        if (sps[i] < 1) continue;
        // Three activation lines and rows that are no whole lines: the shift takes one line of the ring, so every step waits for the activation
        // line that it asked for, which short parts of K do not make up for. Down, 193 .. 256 rows, against the plans of tiles with four lines
        // and more: parts of fewer than 24 lines 1.03 of their time (151 problems, 0.93 .. 1.15; 10840 -> 2728 195 rows 27.6 us on 96 x 224 in
        // 8 parts, 31.8 on 128 x 224 in 11), longer ones 0.93 (189, 0.78 .. 1.03; 24560 -> 6288 193 rows 99 and 77). Whole K is faster, too: 160
        // gate/up problems of 65 .. 1024 rows 0.86 (0.70 .. 1.09; 25776 x 3664 199 rows 62.5 and 50.3, 57104 x 7176 204 rows 214 and 197).
        if (ragged && t.na < 4 && sps[i] > 1 && (k + 63) / 64 < 24 * sps[i]) continue;
        double us = mid_time(np, nq, k, ragged, t, steps[s], sps[i]);
        // The estimate flatters fewer parts on lower tiles, which fetch every activation row for fewer weight rows (11008 -> 4096,
        // 200 rows: four parts on 64 x 224 38.4 us, eight on 128 x 224 34.5; 14336 -> 4096, 256 rows 48.8 and 45.6).
        if (splits == 0 && !gated && nq > 64 && tq == 1 && t.fp == 4) us *= 0.92;
        if (best.tile < 0 || us < best.us) best = {tile, steps[s], sps[i], us};
      }
    }
  }
  return best;
}

// A search takes a few microseconds of host time and one call asks for its plans several times (workspace query, launch), so each
// thread keeps the last few plans by the sizes they follow from.
MidPlan mid_plan(bool gated, int np, int nq, int k, bool ragged, int splits, int max_splits) {
  struct Entry {
    int np, nq, k, rest;
    MidPlan plan;
  };
  static thread_local Entry memo[32];  // zero-initialised: np 0 is never asked for
  const int rest = (gated ? 1 : 0) | (ragged ? 2 : 0) | splits << 2 | max_splits << 8;
  const unsigned h = (((unsigned)np * 31u + (unsigned)nq) * 31u + (unsigned)k) * 31u + (unsigned)rest;
  Entry& e = memo[(h ^ (h >> 7) ^ (h >> 15)) % 32];
  if (e.np != np || e.nq != nq || e.k != k || e.rest != rest)
    e = {np, nq, k, rest, find_plan(gated, np, nq, k, ragged, splits, max_splits)};
  return e.plan;
}

// static storage: "mid_<weight rows>x<activation rows>"
const char* mid_name(const MidPlan& p) {
  static char names[kNumTiles][16];
  static const bool done = [] {
    for (int i = 0; i < kNumTiles; ++i) snprintf(names[i], sizeof(names[i]), "mid_%dx%d", kMidTiles[i].fp * 32, kMidTiles[i].fq * 32);
    return true;
  }();
  (void)done;
  return p.tile >= 0 ? names[p.tile] : "none";
}

int mid_tile_count() { return kNumTiles; }
int mid_tile_rows(int tile) { return 32 * kMidTiles[tile].fp; }
int mid_tile_cols(int tile) { return 32 * kMidTiles[tile].fq; }
int mid_tile_index(int bp, int bq) {
  for (int i = 0; i < kNumTiles; ++i)
    if (kMidTiles[i].fp * 32 == bp && kMidTiles[i].fq * 32 == bq) return i;
  return -1;
}

hipError_t launch_mid(int dtype, bool gated, const MidPlan& p, const GemmArgs& a, hipStream_t stream) {
  if (p.tile < 0 || p.tile >= kNumTiles || p.step <= 0 || p.step > 32 * kMidTiles[p.tile].fp || p.step % 8 != 0)
    return hipErrorInvalidValue;
  if (a.np <= 0 || a.nq <= 0) return hipSuccess;
  const int ph = mid_ragged(a) ? 1 : 0;
  const hipError_t e = dtype == 0 ? (gated ? launch_mid_bf16_gateup(p, a, ph, stream) : launch_mid_bf16_down(p, a, ph, stream))
                                  : (gated ? launch_mid_fp16_gateup(p, a, ph, stream) : launch_mid_fp16_down(p, a, ph, stream));
  if (e != hipSuccess || a.splits <= 1) return e;
  return launch_splitk_reduce(dtype, a, stream);
}

}  // namespace fsw
