"""Launch plans (mmp_plan.h), compiled for the host: where a reduction's
partials lie, and grids that HIP accepts."""
import ctypes
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "macmetalpy_amd",
                    "csrc")
SOURCE = r"""
#include "mmp_plan.h"
extern "C" {
// out: splits, second kernel, slot of the partials, workgroups along the columns
void t_reduce(int arg, int elem, long long outer, long long len, long long inner, long long *out) {
  const int vec = arg ? 1 : elem == 1 ? 4 : 16 / elem;
  if (mmpi::short_axis(outer, len, inner, vec, 16, false)) {
    out[0] = 1;
    out[1] = 0;
    out[2] = mmpi::partials_slot(false);
    out[3] = (outer * ((inner + vec - 1) / vec) + 255) / 256;
    return;
  }
  const mmpi::ColPlan p = arg ? mmpi::argreduce_cols_plan(outer, len, inner, 256)
                              : mmpi::reduce_cols_plan(outer, len, inner, vec, elem == 2, elem, 256);
  out[0] = p.splits;
  out[1] = mmpi::second_kernel(p.splits, outer * len * inner * elem);
  out[2] = mmpi::partials_slot(out[1]);
  out[3] = p.ncb;
}
// out: tile, K ranges, workgroups of a matrix
void t_gemm(long long batch, int m, int n, int k, int elem, int may_split, long long *out) {
  const mmpi::GemmPlan p = mmpi::gemm_plan(batch, m, n, k, elem, may_split != 0, 256);
  out[0] = p.tile;
  out[1] = p.splits;
  out[2] = p.tile ? ((m + (long long)p.tile - 1) / p.tile) * ((n + (long long)p.tile - 1) / p.tile) : 0;
}
// workgroups of a strided reduction
long long t_groups(int heavy, int elem, long long outer, long long len, long long inner) {
  const mmpi::ColPlan p =
      mmpi::reduce_cols_plan(outer, len, inner, elem == 1 ? 4 : 16 / elem, heavy != 0, elem, 256);
  return outer * p.ncb * p.splits;
}
int t_scan(long long len, long long inner, int in, int out) {
  return mmpi::scan_cols_by_vector(len, inner, in, out);
}
int t_solve(long long batch, int n, int nrhs, int elem) {
  return mmpi::solve_block_waves(batch, n, nrhs, elem, 256);
}
long long t_scan_rows(int in, int out) { return mmpi::scan_by_rows_least(in, out); }
int t_tagged_slot() { return mmpi::SCRATCH_REDUCE_PARTIALS; }
int t_slots() { return mmpi::SCRATCH_NSLOTS; }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, so = str(d / "plan.cpp"), str(d / "plan.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    cmd = [shutil.which("g++") or "g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC",
           f"-I{CSRC}", src, "-o", so]
    p = subprocess.run(cmd, capture_output=True, text=True)
    assert p.returncode == 0, p.stderr
    return ctypes.CDLL(so)


def _reduce(plans, arg, elem, outer, length, inner):
    out = (ctypes.c_longlong * 4)()
    i64 = ctypes.c_longlong
    plans.t_reduce(arg, elem, i64(outer), i64(length), i64(inner), out)
    return tuple(out)


def test_raw_partials_stay_out_of_the_tagged_words(plans):
    """The words that a reader trusts by their tag hold tagged partials only:
    a reduction that leaves raw partials for a second kernel (an int32
    maximum's would carry array values where a tag stands) uses other memory."""
    seen = set()
    for arg in (0, 1):
        for elem in (1, 2, 4, 8):
            for outer in (1, 3, 500):
                for length in (2, 300, 5000, 100_000, 2_000_000):
                    for inner in (2, 3, 50, 257, 1001, 20_000):
                        if outer * length * inner > 2e9:
                            continue
                        splits, second, slot, _ = _reduce(plans, arg, elem, outer, length, inner)
                        assert splits >= 1 and slot < plans.t_slots()
                        assert (slot == plans.t_tagged_slot()) == (not second)
                        seen.add((splits > 1, second))
    assert seen == {(False, 0), (True, 0), (True, 1)}  # every kind came up


def test_workgroups_of_strided_reductions(plans):
    """About one workgroup a CU (256), two and four where comparisons of floats
    are what an element costs, and no short axis cut although its column blocks
    alone outnumber the CUs."""
    plans.t_groups.restype = ctypes.c_longlong

    def groups(heavy, elem, *shape):
        return plans.t_groups(heavy, elem, *(ctypes.c_longlong(v) for v in shape))

    for shape in ((1, 10_000, 10_001), (8, 4000, 1001), (1, 300_000, 333)):
        assert 200 <= groups(0, 4, *shape) <= 256 and 200 <= groups(0, 2, *shape) <= 256
        assert 400 <= groups(1, 4, *shape) <= 512 and 800 <= groups(1, 2, *shape) <= 1024
    assert groups(0, 1, 1, 10_000, 10_001) > 400 and groups(0, 1, 20, 30_000, 30) <= 256
    assert groups(0, 4, 300, 300, 300) == 600 and groups(0, 4, 1, 300, 90_000) == 352


MAX_ITEMS = 0xFFFFFFFF  # work-items per grid dimension


def test_reductions_of_very_wide_rows_fit_a_grid(plans):
    """Down the columns of rows as wide as the memory of a device holds (two
    of 2^33 bytes and more): as many columns as a thread each could cover."""
    for elem in (1, 2, 4, 8):
        for inner in ((1 << 31) - 1, (1 << 31) + 1, (1 << 32) - 257):
            for length in (2, 3, 8, 16, 17, 40):
                if elem * inner * length > 288 * 10**9:
                    continue
                for arg in (0, 1):
                    assert _reduce(plans, arg, elem, 1, length, inner)[3] * 256 <= MAX_ITEMS


def _gemm(plans, batch, m, n, k, elem, may_split=True):
    out = (ctypes.c_longlong * 3)()
    plans.t_gemm(ctypes.c_longlong(batch), m, n, k, elem, int(may_split), out)
    return tuple(out)


@pytest.mark.parametrize("elem", [2, 4, 8])
def test_product_grids_fit(plans, elem):
    """Tall and wide products: no tile whose workgroups pass the limit of a
    grid is chosen, and wherever 128 wide tiles fit there is a plan."""
    for rows in (1 << 20, 500_000_000, (1 << 29) - 31, 1 << 29, (1 << 29) + 1, 600_000_000, 1 << 30,
                 (1 << 31) - 200):
        for cols in (1, 2, 31, 32, 33, 100, 129):
            for k in (1, 2, 32, 100):
                for m, n in ((rows, cols), (cols, rows)):
                    tile, splits, wgs = _gemm(plans, 1, m, n, k, elem)
                    wide = -(-m // 128) * -(-n // 128)
                    assert (tile != 0) == (wide * 256 <= MAX_ITEMS), (m, n, k)
                    assert wgs * 256 <= MAX_ITEMS and 1 <= splits <= 65535, (m, n, k, tile)
    assert _gemm(plans, 1, (1 << 31) - 1, 1, 2, elem)[0] == 0  # 2^24 tiles of 128
    # the largest that 32 wide tiles are laid over
    assert _gemm(plans, 1, (1 << 29) - 32, 1, 2, elem)[0] == 32


@pytest.mark.parametrize("batch,m,n,k,elem,tiles", [
    (300, 200, 200, 200, 8, (64, 128)), (1000, 200, 200, 200, 8, (64, 128)), (200, 224, 224, 224, 8, (64, 128)),
    (1000, 160, 160, 160, 8, (64,)), (1, 1500, 700, 900, 8, (32,)), (5000, 32, 32, 32, 8, (32,)),
    (300, 200, 250, 33, 4, (32,)), (500, 120, 100, 90, 4, (128,))])
def test_product_tiles(plans, batch, m, n, k, elem, tiles):
    """The tiles that were quicker."""
    assert _gemm(plans, batch, m, n, k, elem, batch == 1)[0] in tiles


@pytest.mark.parametrize("length,inner,sizes,vector", [
    (10_000, 33, (4, 4), 1), (30_000, 1001, (4, 4), 1), (10_382, 2258, (4, 4), 1), (256, 100_001, (4, 4), 1), (3000, 1001, (4, 4), 1),
    (1000, 1001, (4, 4), 0), (3000, 3001, (4, 4), 0), (256, 16_385, (4, 4), 0), (256, 65_537, (4, 4), 0),
    (1_000_000, 33, (4, 4), 0), (10_000, 3, (4, 4), 0), (10_000, 333, (4, 8), 1), (100_000, 33, (4, 8), 1),
    (3000, 1001, (4, 8), 0), (100_000, 5, (4, 8), 0), (1000, 40_001, (4, 8), 0), (10_000, 1001, (2, 2), 0),
    (200, 50_001, (2, 2), 0), (10_000, 1001, (8, 8), 0)])
def test_column_scans_by_vector(plans, length, inner, sizes, vector):
    """The layout that was quicker for rows that are no whole aligned vectors."""
    assert plans.t_scan(ctypes.c_longlong(length), ctypes.c_longlong(inner), *sizes) == vector


def test_substitution_plan(plans):
    """The block kernel's waves: a power of two, none for a few unknowns, and
    never more of them in a CU than its LDS and registers are planned for."""
    seen = set()
    for elem in (4, 8):
        for batch in (1, 7, 300, 5000, 100_000):
            for n in (1, 2, 8, 9, 16, 17, 23, 24, 31, 32, 64, 65, 100, 256, 257, 2000, 4096):
                for nrhs in (1, 2, 3, 8, 9, 31, 32, 1000, 0x7FFFFFFF):
                    w = plans.t_solve(ctypes.c_longlong(batch), n, nrhs, elem)
                    assert w in (0, 1, 2, 4, 8)
                    assert w or n < 97
                    assert not w or n > 8
                    seen.add(w)
    assert seen == {0, 1, 2, 4, 8}


@pytest.mark.parametrize("sizes,tiled,by_rows", [((4, 4), 255, 260), ((4, 8), 255, 260), ((2, 2), 260, 416),
                                                 ((8, 8), 260, 416), ((2, 8), 900, 2000), ((1, 8), 900, 2000)])
def test_unaligned_rows_scanned_by_workgroups(plans, sizes, tiled, by_rows):
    """Row counts at which scans in tiles, and by rows, were quicker."""
    plans.t_scan_rows.restype = ctypes.c_longlong
    assert tiled < plans.t_scan_rows(*sizes) <= by_rows
