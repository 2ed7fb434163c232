"""The counters of a decode attention that merges its splits in one launch lie behind the 8 MiB of partial results, in an array that a library of
its own holds: a copy of it without them (libcutile_hip_scratch.so of an earlier build) gets the two kernels, which count nothing."""
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
import ctypes, sys, torch
sys.path[:0] = [sys.argv[1], sys.argv[1] + "/tests"]
from __graft_entry__ import load_package
ct = load_package(testing=True)
ct.LIB_PATH = sys.argv[2]
ct.check(ct.lib().cutile_testing_use_fake_hip(1))
q, kv = torch.zeros(2, 4, 128).half(), torch.zeros(2, 500, 128).half()
ct.fmha_decode_gqa_noalloc(q, kv, kv, ct.partition(torch.zeros(2, 4, 128).half(), [1, 4, 128]), 0.1, torch.zeros(1, dtype=torch.int32), 8)
print(ct.lib().cutile_testing_launch_count(), ct.last_resolved()["symbol"])
"""


@pytest.mark.parametrize("size,launches,symbol", [(8 << 20, 2, "splitk_reduce_merge_entry__f16"), ((8 << 20) + 64 * 64 * 4, 1, "fmha_decode_gqa_split_entry__f16_g4_d128_mfma_merge")])
def test_counters_only_where_there_is_room_for_them(fake_hip, tmp_path, size, launches, symbol):
    lib = str(tmp_path / os.path.basename(fake_hip.TESTING_LIB_PATH))
    shutil.copy(fake_hip.TESTING_LIB_PATH, lib)
    (tmp_path / "stub.c").write_text(STUB % size)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "libcutile_hip_scratch.so"), str(tmp_path / "stub.c")], check=True)
    got = subprocess.run([sys.executable, "-c", CALL, ROOT, lib], capture_output=True, text=True)
    assert got.returncode == 0, got.stderr[-2000:]
    assert got.stdout.split() == [str(launches), symbol]
