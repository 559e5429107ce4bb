"""Launch plans (mmp_plan.h), compiled for the host: where a reduction's
partials lie."""
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
// out: splits, second kernel, slot of the partials
void t_reduce(int arg, int elem, long long outer, long long len, long long inner, long long *out) {
  const int vec = elem == 1 ? 4 : 16 / elem;
  const mmpi::ColPlan p = arg ? mmpi::argreduce_cols_plan(outer, len, inner, 256)
                              : mmpi::reduce_cols_plan(outer, len, inner, vec, 256);
  out[0] = p.splits;
  out[1] = mmpi::second_kernel(p.splits, outer * len * inner * elem);
  out[2] = mmpi::partials_slot(out[1]);
}
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
    out = (ctypes.c_longlong * 3)()
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
                        splits, second, slot = _reduce(plans, arg, elem, outer, length, inner)
                        assert splits >= 1 and slot < plans.t_slots()
                        assert (slot == plans.t_tagged_slot()) == (not second)
                        seen.add((splits > 1, second))
    assert seen == {(False, 0), (True, 0), (True, 1)}  # every kind came up
