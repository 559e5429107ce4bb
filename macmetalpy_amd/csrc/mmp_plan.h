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

// Strided layouts: the split of the reduced axis that leaves the CUs most
// evenly loaded, up to `per_cu` workgroups each and at least 64 steps of rows
// (`steps`: rows over the rows a workgroup's lanes lie on side by side) to a
// split.  Workgroups of a launch of this size all run together, so what
// counts is that each CU gets as many: 40 column blocks x 6 splits (240
// workgroups on 256 CUs) sum 10,000 x 10,001 float32 in 69 us, x 7 (280)
// in 91.  Measured on 16384^2 float32 over axis 0: the column-vector sum runs
// best with one workgroup per CU (256: 6.2 TB/s; 128: 5.3, 512: 5.8, 1024:
// 5.4, 2048: 5.3), the arg kernel with four (argmax 4.76 TB/s; 512: 3.2,
// 2048: 4.45).
constexpr int kColVecPerCu = 1, kColPerCu = 4;
inline int col_splits(long long col_blocks, long long steps, int per_cu, long long cus) {
  long long most = steps / 64;
  if (most > 1024) most = 1024;
  // enough workgroups already without splitting, or too few rows to split
  if (col_blocks >= 4 * cus * per_cu || most <= 1) return 1;
  // up to per_cu per CU; where the column blocks alone are about that many,
  // a few more, which fill the CUs better
  long long top = cus * per_cu / col_blocks;
  if (top < 4) top = 4;
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
// rows are shorter than that.
inline ColPlan reduce_cols_plan(long long outer, long long len, long long inner, int vec,
                                long long cus) {
  const int vi = inner >= vec ? vec : 1;
  ColPlan p{0, 0, 0, 1};
  while (p.lanes < 6 && ((long long)vi << p.lanes) < inner) ++p.lanes;
  p.cw = vi << p.lanes;
  p.ncb = (inner + p.cw - 1) / p.cw;
  p.splits = col_splits(outer * p.ncb, len >> (6 - p.lanes), kColVecPerCu, cus);
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

}  // namespace mmpi
