"""The counters of a decode attention that merges its splits in one launch lie behind the 8 MiB of partial results, in an array that a library of
its own holds: a copy of it without them (libcutile_hip_scratch.so of an earlier build) gets the two kernels, which count nothing.  So do launches of
more workgroups than the compute units hold at once."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

STUB = r"""
#include <stddef.h>
static char memory[%d];
int cutile_scratch_lookup(void** ptr, size_t* bytes, int* ordinal) {
  *ptr = memory, *bytes = sizeof(memory);
  if (ordinal) *ordinal = 0;
  return 0;
}
"""

CALL = r"""
import sys, torch
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
from __graft_entry__ import load_package
ct = load_package(testing=True)
ct.LIB_PATH = sys.argv[2]
ct.check(ct.lib().cutile_testing_use_fake_hip(1))
for size in sys.argv[3:]:
    heads, group, d, splits = map(int, size.split(","))
    ct.lib().cutile_testing_clear_log()
    q, kv = torch.zeros(heads, group, d).half(), torch.zeros(heads, 500, d).half()
    ct.fmha_decode_gqa_noalloc(q, kv, kv, ct.partition(torch.zeros_like(q), [1, group, d]), 0.1, torch.zeros(1, dtype=torch.int32), splits)
    print(ct.lib().cutile_testing_launch_count(), ct.last_resolved()["symbol"])
"""


def _run(ct, tmp_path, scratch_bytes, *sizes):
    """launches and last kernel of a call of each (heads, GROUP, D, splits), beside a scratch library of that size"""
    lib = str(tmp_path / os.path.basename(ct.TESTING_LIB_PATH))
    shutil.copy(ct.TESTING_LIB_PATH, lib)
    (tmp_path / "stub.c").write_text(STUB % scratch_bytes)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "libcutile_hip_scratch.so"), str(tmp_path / "stub.c")], check=True)
    got = subprocess.run([sys.executable, "-c", CALL, ROOT, lib, *[",".join(map(str, s)) for s in sizes]], capture_output=True, text=True)
    assert got.returncode == 0, got.stderr[-2000:]
    return [tuple(line.split()) for line in got.stdout.splitlines()]


PARTIALS, COUNTERS = 8 << 20, 64 * 64 * 4
MERGE = ("2", "splitk_reduce_merge_entry__f16")


def test_counters_only_where_there_is_room_for_them(fake_hip, tmp_path):
    assert _run(fake_hip, tmp_path, PARTIALS, (2, 4, 128, 8)) == [MERGE]
    assert _run(fake_hip, tmp_path, PARTIALS + COUNTERS, (2, 4, 128, 8)) == [("1", "fmha_decode_gqa_split_entry__f16_g4_d128_mfma_merge")]


def test_one_launch_while_the_compute_units_hold_it(fake_hip, tmp_path):
    """256 compute units: 384 workgroups, at D = 256 as many as compute units"""
    got = _run(fake_hip, tmp_path, PARTIALS + COUNTERS, (6, 1, 64, 64), (7, 1, 64, 64), (64, 2, 128, 6), (64, 2, 128, 7), (8, 4, 256, 32), (9, 4, 256, 32), (64, 4, 64, 64))
    assert [g[0] for g in got] == ["1", "2", "1", "2", "1", "2", "2"]
    assert got[1] == MERGE and got[4][1] == "fmha_decode_gqa_split_entry__f16_g4_d256_mfma_merge"
