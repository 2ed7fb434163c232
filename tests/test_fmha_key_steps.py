"""Attention whose keys several workgroups share, with keys behind the last one that any row sees: every key step of every query tile has one workgroup, and the kernel
counts on no more of them than are launched."""
import ctypes as C
import os
import struct
import subprocess

import pytest
import torch

from test_fmha_keys import _close, _reference

KERNELS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutile-rs_amd", "csrc", "kernels")


class KeySteps(C.Structure):
    _fields_ = [("first", C.c_int32), ("end", C.c_int32), ("shares", C.c_uint32)]


@pytest.fixture(scope="module")
def kernel_steps(tmp_path_factory):
    """(keys_seen, key_steps) as the kernels compute them"""
    at = tmp_path_factory.mktemp("key_steps")
    (at / "steps.cpp").write_text('#include "key_steps.h"\nextern "C" int32_t seen(int32_t e, int32_t q, int32_t p, int32_t k, int32_t c) { return cutile::keys_seen(e, q, p, k, c); }\n'
                                  'extern "C" cutile::KeySteps steps(int32_t k, int32_t s, int32_t e, uint32_t z, uint32_t n) { return cutile::key_steps(k, s, e, z, n); }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-Wno-return-type-c-linkage", "-I", KERNELS, "-o", str(at / "steps.so"), str(at / "steps.cpp")], check=True)
    lib = C.CDLL(str(at / "steps.so"))
    lib.seen.argtypes, lib.seen.restype = [C.c_int32] * 5, C.c_int32
    lib.steps.argtypes, lib.steps.restype = [C.c_int32] * 3 + [C.c_uint32] * 2, KeySteps
    return lib.seen, lib.steps


def test_every_step_has_its_workgroup(kernel_steps):
    """also where the launcher planned for fewer keys than there are"""
    _, steps = kernel_steps
    for keys in (0, 1, 255, 256, 257, 1000, 4111):
        for each in (1, 2, 3, 7, 1 << 25):
            for launched in (1, 2, 5, 32):
                got = [steps(keys, 256, each, z, launched) for z in range(launched)]
                taken = [j for r in got for j in range(r.first, r.end)]
                assert taken == list(range(-(-keys // 256))), (keys, each, launched)
                assert all(r.shares == sum(r.first < r.end for r in got) for r in got), (keys, each, launched)


def test_keys_seen(kernel_steps):
    seen, _ = kernel_steps
    assert seen(32, 17, 4079, 4200, 1) == 4096 and seen(32, 32, 4079, 4200, 1) == 4111 and seen(64, 100, 4079, 4100, 1) == 4100
    assert seen(32, 17, 4079, 4200, 0) == 4200 and seen(32, 17, 0x7fffffff, 4200, 1) == 4200 and seen(32, 17, 5, 0, 1) == 0


@pytest.mark.parametrize("d", [64, 128])
def test_a_launch_has_the_workgroups_that_its_kernel_counts(fake_hip, kernel_steps, d):
    ct, (seen, steps) = fake_hip, kernel_steps
    from test_host_abi import _last
    shared = 0
    for heads, rows in ((8, 17), (3, 33), (4, 65), (1, 129), (2, 200), (12, 28)):
        for start in [n * 256 + i for n in (2, 8, 15) for i in (-rows, -rows - 1, 1 - rows, -32, -1, 0, 100)]:
            for there in (start + rows, start + rows + 121):
                q, kv = torch.empty(1, heads, rows, d).half(), torch.empty(1, heads, there, d).half()
                for causal in (True, False):
                    for seq in (False, True):
                        if seq:
                            ct.fmha_seq_f16(q[0].transpose(0, 1), kv[0], kv[0], ct.partition(torch.empty(rows, heads, d).half(), [128, 1, d]), 0.1, 1, kv_len=there, query_start=start, causal=causal)
                        else:
                            ct.fmha(ct.partition(torch.empty(heads, rows, d).half(), [1, 128, d]), q, kv, kv, 0.1, start, 1, causal=causal)
                        rec, args = _last(ct)
                        name = rec.symbol.decode()
                        if not name.endswith("_keys"):
                            continue
                        tile, step = map(int, name.split("16_")[1].replace("few_", "").split("x")[:2])
                        if tile == 64 and d == 128 and "few" not in name:
                            step = 256
                        each, launched = struct.unpack("<i", args[-8:-4])[0], rec.grid[2]
                        shared += launched > 1
                        for end in range(tile, rows + tile, tile):
                            keys = seen(end, rows, start, there, causal)
                            assert (keys == there or keys == start + min(end, rows)) and -(-keys // step) <= each * launched, (heads, rows, start, there, causal, name)
                            assert launched == 1 or steps(keys, step, each, 0, launched).shares == -(-keys // (step * each)), (heads, rows, start, there, causal, name)
    assert shared > 100


@pytest.mark.parametrize("start", [0, 300])
def test_a_launch_that_covers_nothing_is_refused(fake_hip, start):
    ct = fake_hip
    q, kv, out = torch.empty(1, 4, 300, 128).half(), torch.empty(1, 4, 300 + start, 128).half(), torch.empty(4, 300, 128).half()
    seq, position = torch.empty(300, 4, 128).half(), torch.tensor([start], dtype=torch.int32)
    for causal in (True, False):
        for grid in ((0, 2, 1), (4, 0, 1), (0, 0, 1)):
            with pytest.raises(ct.CutileError, match="zero axis"):
                ct.fmha(ct.partition(out, [1, 256, 128], prefix=True), q, kv, kv, 0.1, start, 1, causal=causal, grid=grid)
        for grid in ((3, 0, 1), (0, 4, 1)):
            for where in (dict(kv_len=300 + start, query_start=start), dict(position_start=position)):
                with pytest.raises(ct.CutileError, match="zero axis"):
                    ct.fmha_seq_f16(seq, kv[0], kv[0], ct.partition(torch.empty_like(seq), [128, 1, 128], prefix=True), 0.1, 1, causal=causal, grid=grid, **where)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("heads,group,rows,start,there", [(8, 4, 17, 4079, 4200), (4, 1, 33, 2015, 2100), (2, 1, 129, 895, 1100), (8, 4, 17, 4079, 4096)])
def test_gpu_keys_behind_the_last_row(ct, dev, d, heads, group, rows, start, there):
    """then a product on the same stream, whose workgroups meet on the same counters"""
    g = torch.Generator().manual_seed(rows + start)
    normal = lambda *s: torch.randn(*s, generator=g).half().to(dev)
    q, k, v = normal(1, heads, rows, d), normal(1, heads // group, there, d), normal(1, heads // group, there, d)
    k[:, :, start + rows:] = 100.0
    out, seq = torch.full((heads, rows, d), 7.0, dtype=torch.half, device=dev), torch.full((rows, heads, d), 7.0, dtype=torch.half, device=dev)
    x, y = normal(16, 9216), normal(9216, 64) / 96
    z = torch.zeros(16, 64, dtype=torch.half, device=dev)
    ct.fmha(ct.partition(out, [1, 128, d]), q, k, v, d ** -0.5, start, group, causal=True)
    assert ct.last_resolved()["symbol"].endswith("_keys")
    ct.fmha_seq_f16(q[0].transpose(0, 1), k[0], v[0], ct.partition(seq, [64, 1, d]), d ** -0.5, group, kv_len=there, query_start=start, causal=True)
    ct.gemm(ct.partition(z, [64, 64]), x, y, 9216, accumulate=False, generics=["f16", 64, 64, 1])
    torch.cuda.synchronize()
    ref = _reference(q, k, v, d ** -0.5, start, group, True)
    assert _close(out, ref, torch.half) and _close(seq.permute(1, 0, 2), ref, torch.half)
    want = x.double() @ y.double()
    assert (z.double() - want).norm() <= 2.0 ** -11 * want.norm()      # one rounding to f16 over f32 sums
