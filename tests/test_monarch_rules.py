"""The rules by which the two steps take Kbar and Y through the caches or past them (csrc/monarch_rules.hpp), compiled for the host."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "monarch_rules.hpp"
extern "C" void rules(int D, int units, int na, int nf, int b1, int b2, int causal, int new_kv, int kbar_alone, size_t* rows, int* through, int* past) {
    sfm::MonarchArgs a;
    memset(&a, 0, sizeof(a));
    a.D = D; a.na = na; a.nf = nf; a.b1 = b1; a.b2 = b2; a.causal = causal; a.skip_masked = 1;
    a.new_kv = new_kv;
    *rows = sfm::scratch_rows(a, units, causal != 0);
    *through = sfm::step1_through_caches(a, units, kbar_alone);
    *past = sfm::step2_past_caches(a, units);
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.hip").write_text("#include <string.h>\n" + SOURCE)
    csrc = os.path.join(ROOT, "self-forcing_amd", "csrc")
    subprocess.run([hipcc, "--offload-host-only", "-std=c++17", "-shared", "-fPIC", "-I" + csrc, "-I" + os.path.join(ROOT, "include"),
                    str(d / "rules.hip"), "-o", str(d / "rules.so")], check=True, capture_output=True)
    fn = C.CDLL(str(d / "rules.so")).rules

    def call(na, nf, b1, b2, units, D=128, causal=0, new_kv=0, kbar_alone=0):
        rows, through, past = C.c_size_t(0), C.c_int(0), C.c_int(0)
        fn(D, units, na, nf, b1, b2, causal, new_kv, kbar_alone, C.byref(rows), C.byref(through), C.byref(past))
        return rows.value, bool(through.value), bool(past.value)
    return call


@pytest.mark.parametrize("na,causal", [(1, 1), (3, 1), (6, 3), (9, 3), (9, 9), (12, 6), (20, 4)])
def test_masked_rows_are_not_counted(rules, na, causal):
    pairs = sum((a // causal + 1) * causal for a in range(na))
    assert rules(na, na, 5, 7, 2, causal=causal)[0] == 2 * pairs * 5 * 7
    assert rules(na, na, 5, 7, 2)[0] == 2 * na * na * 5 * 7


def test_block_causal_calls_are_too_small_by_the_rows_they_write(rules):
    assert rules(5, 5, 32, 40, 4)[1] and not rules(5, 5, 32, 40, 4, causal=1)[1]       # 37 MiB of 62
    assert rules(5, 5, 32, 40, 5, causal=1)[1]
    assert rules(5, 5, 32, 40, 4, causal=1, new_kv=1)[1]                               # with a new chunk step 1 forms all rows


def test_the_most_depends_on_the_query_block_frames(rules):
    for na, most in ((1, 1100), (3, 1100), (5, 1100), (6, 240), (12, 240)):
        per_head = na * 12 * 32 * 40 * 512 / 2**20
        fits = int(most / per_head)
        assert rules(na, 12, 32, 40, fits)[1] and not rules(na, 12, 32, 40, fits + 1)[1], na
        assert rules(na, 12, 32, 40, int(512 / per_head), kbar_alone=1)[1] and not rules(na, 12, 32, 40, int(512 / per_head) + 1, kbar_alone=1)[1]
    # masked pairs count from six block-frames on, where step 2 reads past the caches, and not below: 1069 MiB of 1604
    assert rules(3, 3, 90, 52, 78, causal=1)[1] and rules(6, 6, 45, 52, 5, causal=2)[1] and not rules(6, 6, 45, 52, 6, causal=2)[1]


def test_step_2_reads_past_the_caches_from_240_mib_on(rules):
    assert not rules(3, 21, 30, 52, 5)[2] and rules(3, 21, 30, 52, 6)[2]               # 239.9 and 288 MiB
    assert rules(3, 3, 90, 52, 12, causal=1)[2]                                        # masked pairs count


def test_teams_need_more(rules):
    assert rules(2, 8, 32, 26, 7)[1] and not rules(2, 8, 33, 26, 7)[1]                 # 46 and 47 MiB
    assert rules(2, 8, 33, 26, 10)[1] and not rules(2, 8, 32, 26, 6)[1]                # 67 and 39
    assert rules(2, 8, 33, 26, 14, kbar_alone=1)[1]                                    # 47 of Kbar alone, which step 2 does not read
