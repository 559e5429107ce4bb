// mmp_plan.h -- launch plans as plain host arithmetic: no HIP, so that the
// rules can be compiled and tested without a device.
#pragma once

namespace mmpi {

// Scratch memory of the library (mmpi::scratch), one block per slot.
// SCRATCH_REDUCE_PARTIALS holds tagged words or zeros and nothing else: a
// reader takes a word as this call's partial by the tag in its high half
// alone, so a raw value there could pass for one.  Partials without tags have
// SCRATCH_REDUCE_PLAIN.
enum { SCRATCH_REDUCE_PARTIALS = 0, SCRATCH_REDUCE_TICKETS = 1,
       SCRATCH_SCAN_FLAGS = 2, SCRATCH_SCAN_VALUES = 3,
       SCRATCH_SCAN_COUNTER = 4, SCRATCH_REDUCE_PLAIN = 5, SCRATCH_NSLOTS = 6 };

// HIP counts at most 2^32 - 1 work-items per grid dimension.
inline bool grid_fits(long long blocks, int threads) { return blocks <= 0xffffffffLL / threads; }

// Strided layouts: the split of the reduced axis that leaves the CUs most
// evenly loaded, up to `per_cu` workgroups each and at least `least` steps of rows
// (`steps`: rows over the rows a workgroup's lanes lie on side by side) to a
// split.  Workgroups of a launch of this size all run together, so what
// counts is that each CU gets as many: 40 column blocks x 6 splits (240
// workgroups on 256 CUs) sum 10,000 x 10,001 float32 in 69 us, x 7 (280)
// in 91.  Measured on 16384^2 float32 over axis 0: the column-vector sum runs
// best with one workgroup per CU (256: 6.2 TB/s; 128: 5.3, 512: 5.8, 1024:
// 5.4, 2048: 5.3), the arg kernel with four (argmax 4.76 TB/s; 512: 3.2,
// 2048: 4.45).
constexpr int kColVecPerCu = 1, kColPerCu = 4;
inline int col_splits(long long col_blocks, long long steps, int per_cu, long long cus,
                      int least = 64) {
  long long most = steps / least;
  if (most > 1024) most = 1024;
  // enough workgroups already without splitting, or too few rows to split
  if (col_blocks >= 4 * cus * per_cu || most <= 1) return 1;
  // up to per_cu per CU; where the column blocks alone are about that many, a
  // few more of a long axis, which fill the CUs better (a short one's partials
  // cost more than that: float32 300 x 300 x 300 over the middle axis, 600
  // blocks, 23.3 us whole and 25.4 in halves)
  long long top = (cus * per_cu + col_blocks - 1) / col_blocks;
  if (top < 4 && steps >= 1024) top = 4;
  if (top > most) top = most;
  int best = 1;
  double best_fill = 0.0;
  for (long long s = top; s >= 1; --s) {
    const long long wgs = col_blocks * s, per = (wgs + cus - 1) / cus;
    // the CUs' even share of the busiest one's load, less a little for every
    // workgroup on it beyond the wanted number
    double fill = (double)wgs / (double)(per * cus);
    if (per > per_cu) fill -= 0.02 * (double)(per - per_cu);
    if (per < per_cu) fill *= 0.5 + 0.5 * (double)per / per_cu;
    if (fill > best_fill + 1e-9) {
      best_fill = fill;
      best = (int)s;
    }
  }
  return best;
}

// A reduction over the middle axis of (outer, len, inner): `cw` columns a
// workgroup, 2^lanes threads (of a wave, or for arg-reductions of the
// workgroup) side by side on a row, `ncb` column blocks, the axis in `splits`.
struct ColPlan {
  int lanes;
  int cw;
  long long ncb;
  int splits;
};
// Sums and extremes: a lane on `vec` adjacent columns, or on one where the
// rows are shorter than that.  A CU with one workgroup has a wave per SIMD: too
// few where the arithmetic is what an element costs.  So `heavy` ones
// (comparisons and NaN rules) get two, and four of eight columns a lane, which
// also split from half the rows on; and many one-byte elements two (10,000 x
// 10,001 39 -> 28 us for a mean, 20 MB and less 10 -> 13).
// Maximum over axis 0, one workgroup a CU before and now (the comparisons also
// became one expression): float32 10,000 x 10,001 112 -> 70 us, 300,000 x 333 154
// -> 82, 8 x 4000 x 1001 over the middle axis 36 -> 25; float16 99 -> 38, 133 ->
// 39, 41 -> 17.
inline ColPlan reduce_cols_plan(long long outer, long long len, long long inner, int vec, bool heavy,
                                int elem, long long cus) {
  const int vi = inner >= vec ? vec : 1;
  ColPlan p{0, 0, 0, 1};
  while (p.lanes < 6 && ((long long)vi << p.lanes) < inner) ++p.lanes;
  p.cw = vi << p.lanes;
  p.ncb = (inner + p.cw - 1) / p.cw;
  const bool hard = heavy && vi > 1;
  const int per_cu = hard                                              ? (vi >= 8 ? 4 : 2)
                     : elem == 1 && outer * len * inner >= (64LL << 20) ? 2
                                                                        : kColVecPerCu;
  p.splits = col_splits(outer * p.ncb, len >> (6 - p.lanes), per_cu, cus, hard && vi >= 8 ? 32 : 64);
  return p;
}
// Arg-reductions: a thread per column.
inline ColPlan argreduce_cols_plan(long long outer, long long len, long long inner, long long cus) {
  ColPlan p{0, 0, 0, 1};
  while (p.lanes < 8 && (1LL << p.lanes) < inner) ++p.lanes;
  p.cw = 1 << p.lanes;
  p.ncb = (inner + p.cw - 1) / p.cw;
  p.splits = col_splits(outer * p.ncb, len >> (8 - p.lanes), kColPerCu, cus);
  return p;
}

// Axes so short that a workgroup of the plans above spends its time bringing
// lanes and waves together: a thread per `vec` columns that walks the axis by
// itself.  Up to `rows` of them always (us, plans above / a thread per columns;
// sum, maximum, argmax over the middle axis): float32 60,000 x 16 x 9 90 / 8.5,
// 91 / 8.9, 90 / 7.9; 625 x 16 x 1000 9.4 / 9.1, 9.9 / 9.5, 8.6 / 8.7; float16
// 1 x 16 x 1,250,001 12.1 / 9.5, 13.7 / 12.4, 11.9 / 11.8; 1 x 32 x 625,001 9.8 /
// 9.5, 12.9 / 18, 10 / 12.1; sums of 4 and 8 bytes at 64 rows: float32 1 x
// 156,251 11.2 / 9.2, 78 x 1000 9.4 / 9, 3125 x 50 8.6 / 8.6, float64 1 x 78,125
// 11 / 9.  Further on only where rows are shorter than a
// workgroup and workgroups so many that starting them is the time: float32
// 17,361 x 64 x 9 28 / 8.5, 30 / 17, 40 / 10.8, but 3125 x 64 x 50 8.6 / 8.6, 10 /
// 17, 10.4 / 9.9; `heavy` (extremes of floats) by half as much.
inline bool short_axis(long long outer, long long len, long long inner, int vec, int rows, bool heavy) {
  const long long vecs = inner >= vec ? (inner + vec - 1) / vec : inner;
  if (outer * vecs > 0xffffff00LL) return false;  // threads of one grid
  return len <= rows || (inner < 256 && len <= (heavy ? 64 : 128) && outer >= (heavy ? 128 : 64) * len);
}

// Partials of a strided reduction: few are combined by the last workgroup to
// arrive; more are left as they are, (outer, split, column), for a second
// kernel whose many workgroups read them side by side.  One workgroup alone
// reading 256 partials a column took longer than the reduction of a
// 2,000,000 x 50 matrix (float32 sum over axis 0 98 us, against 76 with the
// second kernel), and 25 a column cost a 10,000 x 10,001 argmax 20 us more;
// but 31 of a 2000 x 300 matrix are done sooner than a second launch (8.6 us
// against 11.7).
inline bool second_kernel(int splits, long long bytes) {
  return splits > 64 || (splits > 16 && bytes >= (32LL << 20));
}

// Where the partials of a strided reduction lie.
inline int partials_slot(bool second) {
  return second ? SCRATCH_REDUCE_PLAIN : SCRATCH_REDUCE_PARTIALS;
}

// Tile and K split of the general kernels.  With few output tiles most
// CUs would idle, so the tile is made smaller or the K range cut as well; a
// split pays for its partial products (written once, read once).  The choice
// is the cheapest by this estimate, in microseconds: rounds of workgroups
// over the CUs (two 128, four 64 or eight 32 wide tiles fit one), each a
// start-up plus its slabs, at the matrix cores' rate for the workgroups that
// share a CU but no faster than one alone hides its loads; and the partials
// at 6 TB/s plus a launch.  A single product (batch 1) of at most 16,384
// outputs over a K of 16,384 or more that may be split is always cut into
// ranges of at most 2048 (up to K = 134,215,680; the grid has 65,535 of them),
// whose sums meet in float64: float32 sums of 10^7 terms then stay within 5e-8
// of exact (2e-6 with ranges of 6000).  A product that may not (the stream is
// captured, or there is no memory for the partials) sums its K in one chain, so
// its last places differ.
// A slab of a 32 wide float64 tile loads twice as much for its arithmetic as one
// of a 64 wide tile; where eight of them fill every CU and more wait, that is
// what bounds them, and the slab counts for a third more.  Us with 32 / 64 / 128
// wide tiles: 300 products of 200^3 204 / 157 / 161, 1000 of them 648 / 516 / 495, of
// 160^3 306 / 238 / 382, 200 of 224^3 167 / 118 / 134; but 1500 x 700 x 900, 1034
// tiles of 32, 62 / 73 / 81.
// Measured over tiles and splits of 30 products, the choice is the fastest or
// within a tenth of it but for float64 4000 x 70 x 3000, 66 us where four ranges take
// 58.  float32 1000^3 28 us (32 wide, unsplit; 64 wide 30, in four 36), 2049^3
// 198 (64 wide; 32 wide 200), 4000 x 70 x 3000 37 (32 wide in two; in four 35);
// float64 500 x 500 x 100,000 0.85 ms (128 wide in 32; 64 wide in 16 0.81;
// unsplit 15.8).
// A tile whose workgroups are more than a grid holds is no choice (from 2^29
// rows of one column on 32 wide ones are).
struct GemmPlan {
  int tile;    // 128, 64 or 32; 0: none fits a grid
  int splits;  // K ranges
  int kspan;   // 128-byte slabs of K in each but the last
  double us;
};
inline double rounds_us(double wgs, double per_cu, double slabs, double start, double shared,
                        double alone, double cus) {
  const double full = __builtin_floor(wgs / (cus * per_cu)), rest = wgs - full * cus * per_cu;
  const double share = __builtin_ceil(rest / cus);
  const double step = shared * share > alone ? shared * share : alone;
  return full * (start + slabs * shared * per_cu) + (rest > 0 ? start + slabs * step : 0.0);
}
inline GemmPlan gemm_plan(long long batch, int M, int N, int K, int elem, bool may_split,
                          double cus) {
  const int nk = (int)(((long long)K * elem + 127) / 128);
  GemmPlan best{0, 1, nk, 1e30};
  const bool long_sum = may_split && batch == 1 && (double)M * N <= 16384 && K >= 16384;
  const int s0 = !long_sum ? 1 : K < 2048 * 65535 ? (K + 2047) / 2048 : 65535;  // grid limit
  for (int tile = 128; tile >= 32; tile /= 2) {
    const long long one = (((long long)M + tile - 1) / tile) * (((long long)N + tile - 1) / tile);
    if (!grid_fits(one, 256)) break;  // nor do smaller tiles
    const double tiles = (double)one * (double)batch;
    const double per_cu = tile == 128 ? 2 : tile == 64 ? 4 : 8;
    const bool crowded = elem == 8 && tiles > cus * per_cu;  // (of 32 wide ones)
    const double start = tile == 128 ? 6.0 : tile == 64 ? 3.0 : 1.5;  // and the result's stores
    // a slab of one workgroup: of several sharing a CU, and alone on it (the
    // 16-bit matrix rate leaves a slab to its loads and LDS traffic)
    const double shared = elem == 2 ? (tile == 128 ? 0.85 : tile == 64 ? 0.4 : 0.18)
                                    : (tile == 128 ? 1.85 : tile == 64 ? 0.5 : crowded ? 0.2 : 0.15);
    const double alone = elem == 2 ? (tile == 128 ? 1.05 : tile == 64 ? 0.55 : 0.35)
                                   : (tile == 128 ? 2.2 : tile == 64 ? 0.65 : 0.25);
    for (int s = s0; s <= 65535; s *= 2) {
      const double wgs = tiles * s;
      if (s > s0 && (!may_split || nk / s < 4 || wgs > 2 * cus * per_cu)) break;
      double t = rounds_us(wgs, per_cu, (nk + s - 1) / s, start, shared, alone, cus);
      if (s > 1) t += 4.0 + 2e-6 * s * (double)batch * M * N * (elem == 2 ? 4 : elem) / 6.0;
      if (t < best.us * 0.98) best = GemmPlan{tile, s, 0, t};
    }
  }
  best.kspan = (nk + best.splits - 1) / best.splits;
  best.splits = (nk + best.kspan - 1) / best.kspan;
  return best;
}

// Rows from which unaligned ones, each longer than a tile, are scanned by a
// workgroup each instead of in tiles that look back.  What a row's waves walk
// is paid in latency, so fewer rows need more bytes a step.  40,000,000
// elements, us in tiles / by rows at 260, 416, 900 and 2000 rows: float32 157 /
// 119, 152 / 90, 153 / 76, 191 / 73; int32 to int64 209 / 164, 208 / 129, 205 /
// 113, 272 / 116; float64 209 / 200, 206 / 158, 221 / 148, 224 / 141; int64 166 /
// 200, 162 / 159, 191 / 147, 187 / 141; float16 97 / 122, 87 / 77, 93 / 65, 130 /
// 55; int16 to int64 104 / 171, 107 / 133, 100 / 119, 133 / 121.
inline long long scan_by_rows_least(int in_size, int out_size) {
  if (in_size <= 2 && out_size == 8) return 2000;
  return in_size == 4 ? 256 : 400;
}

// Whether a scan down `inner` columns whose rows are not whole aligned vectors
// takes 16-byte vectors (with a pass of its own for the chunks' carries) or a
// column per thread.  Vectors pay where the carries are what a thread per column
// spends its time on, and for the largest inputs; 2-byte elements, whose eight
// running sums a lane are too long a chain, and 8-byte ones, never.  By column /
// by vectors, us: float32 10,000 x 33 44 / 19, 30,000 x 1001 101 / 73, 100,000 x
// 333 125 / 89, 10,000 x 5001 135 / 123, 256 x 100,001 57 / 52, but 1000 x 1001 11 / 15, 3000 x 3001 25 /
// 26.5, 256 x 65,537 35.5 / 40.5, 1,000,000 x 33 375 / 498 (the axis is cut 256
// times at most); int32 to int64 10,000 x 333 50 / 27, 100,000 x 33 97 / 73, but
// 3000 x 1001 23 / 26, 100,000 x 5 53 / 59; float16 10,000 x 1001 53 / 82.
inline bool scan_cols_by_vector(long long len, long long inner, int in_size, int out_size) {
  if (in_size != 4 || inner < 4 || len > (1 << 18)) return false;
  if (out_size > 4) return len >= 8192 && inner >= 32 && inner <= 4096;
  return len >= 8192 || (len >= 3000 && inner <= 2048) || (len >= 256 && len * inner >= 24'000'000);
}

// Substitution with n unknowns: the kernel that solves blocks of 32 (8
// right-hand sides a workgroup, a wave each), with `waves` waves a workgroup,
// or 0: the one with a barrier per unknown and 32 right-hand sides a workgroup.
// The block kernel's chain is 32 steps a block whatever n is, so few unknowns,
// and many right-hand sides of them, are quicker by the other.  Us, by unknown /
// by block; float64: 1 x (16, 1 right-hand side) 11 / 13, (32, 1) 20 / 14, (32, 4)
// 20 / 22, (64, 8) 51 / 63, (128, 8) 139 / 123, (64, 40) 109 / 64; 2000 x (32, 1)
// 28 / 21, (32, 40) 165 / 439, (64, 4) 102 / 101, (80, 40) 1300 / 1176; 20,000 x
// (4, 40) 74 / 1794; float32: 1 x (32, 4) 20 / 17, (64, 8) 47 / 44; 2000 x (64, 4)
// 66 / 72, (96, 40) 1140 / 774; 20,000 x (16, 1) 118 / 78.
// Waves: one per right-hand side and enough for the rows below a block, but in
// all what keeps a CU busy, since they divide the same work: float64 n = 300, one
// right-hand side, of 300 matrices 175 / 162 / 157 / 276 with 1 / 2 / 4 / 8 waves,
// of 1500 306 / 423 / 541 / 898; 20 x (1000, 1000), whose right-hand sides let
// two workgroups into a CU's LDS, 27.6 / 17 / 9.8 / 12.6 ms.
inline int solve_block_waves(long long batch, int n, int nrhs, int elem, long long cus) {
  const long long wgs = batch * ((nrhs + 7) / 8);
  const bool filled = wgs > 4 * cus;
  const int least = nrhs == 1   ? (elem == 8 || batch <= 4096 ? 17 : 9)
                    : nrhs == 2 ? (elem == 4 ? 24 : filled ? 56 : 32)
                    : nrhs <= 4 ? (elem == 8 ? 88 : filled ? 80 : 32)
                    : nrhs <= 8 ? (elem == 4 && !filled ? 64 : 96)
                                : (filled ? 88 : nrhs >= 32 ? 48 : 64);
  if (n < least) return 0;
  int want = n <= 64 ? 1 : n <= 256 ? 2 : 8;
  while (want < 8 && want < nrhs) want *= 2;
  const long long lds = (long long)n * (nrhs < 8 ? nrhs : 8) * elem;
  long long here = (wgs + cus - 1) / cus, fit = 160 * 1024 / lds;  // workgroups on a CU
  if (here > fit) here = fit > 1 ? fit : 1;
  int w = 8;
  while (w > 1 && w * here > (elem == 8 ? 10 : 20)) w /= 2;
  return want < w ? want : w;
}

}  // namespace mmpi
