"""192 x 384 GEMM tiles (gemm_wide.h): which launches take them, ragged rows, columns that end in a tile's first unit and on its edge, an even and an odd
number of K tiles, rows further apart than they are long, z as the initial accumulator; and that the compiler moves no accumulator inside the K loop."""
import os
import re
import subprocess

import pytest
import torch

from util import rel_l2

WIDE = "_wide_192x256x64_q2x4_mix"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,n,k,accumulate", [(532, 27904, 896, False), (529, 28040, 960, True), (576, 28424, 1024, True), (1329, 12296, 640, False)])
def test_gpu_tiles_of_384_columns(ct, dev, dtype, m, n, k, accumulate):
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + 24, device=dev, generator=g).to(dt)[:, :k]
    y = (torch.randn(k, n + 8, device=dev, generator=g) / k ** 0.5).to(dt)[:, :n]
    z0 = torch.randn(m, n, device=dev, generator=g).to(dt)
    z = torch.full((m + 1, n + 8), 7.0, dtype=dt, device=dev)
    z[:m, :n] = z0
    ct.gemm(ct.partition(z[:m, :n], [256, 256]), x, y, k, accumulate=accumulate)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith(WIDE)
    want = x.double() @ y.double() + (z0.double() if accumulate else 0)
    # one rounding to the output type over f32 sums
    got, unit = z[:m, :n].double(), {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
    assert rel_l2(got.cpu().numpy(), want.cpu().numpy()) <= unit
    assert (got - want).abs().amax(0).max() <= unit * 1.01 * want.abs().max()      # no column was left out or written by two tiles
    assert torch.all(z[m] == 7.0) and torch.all(z[:, n:] == 7.0)


def test_which_sizes_take_them(fake_hip):
    """one round of them where 256 x 256 is more than one; not with a ragged K, columns of z in units of 4, fewer or more tiles, or a kernel named"""
    ct = fake_hip
    from test_gemm_tiles import _workgroups
    bufs = {dt: torch.empty(120 << 20, dtype=dt) for dt in (torch.half, torch.bfloat16)}
    for m, n, k, wide in ((1344, 12032, 4608, True), (900, 18432, 5120, True), (560, 28672, 4096, True), (532, 27904, 896, True), (529, 28040, 960, True),
                          (576, 28424, 1024, True), (1329, 12296, 640, True), (1344, 12032, 4616, False), (1344, 12036, 4608, False), (2048, 8960, 3584, False),
                          (1024, 8192, 4096, False), (1500, 14336, 4096, False), (4096, 16384, 512, False)):
        for dt, buf in bufs.items():
            view, name = lambda rows, cols: buf[:rows * cols].view(rows, cols), {torch.half: "f16", torch.bfloat16: "bf16"}[dt]
            ct.gemm(ct.partition(view(m, n), [256, 256]), view(m, k), view(k, (n + 7) // 8 * 8), k, accumulate=False, generics=[name, 256, 256, 8])
            assert ct.last_resolved()["symbol"].endswith(WIDE) == wide, (m, n, k, dt, ct.last_resolved()["symbol"])
            if wide:
                assert _workgroups(ct) == -(-m // 192) * -(-n // 384)
                ct.gemm(ct.partition(view(m, n), [256, 256]), view(m, k), view(k, n), k, accumulate=False, variant=name + "_192x256x64_q2x4")
                assert not ct.last_resolved()["symbol"].endswith(WIDE)


def test_no_accumulator_is_moved_in_the_k_loop():
    """The matrix instructions of these kernels are written so that the compiler does not know them for such, and puts no wait states between one and another
    instruction on its result: between the first and the last of them there is no spill, and no move into or out of a register that they accumulate in."""
    lib = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutile-rs_amd", "lib", "gemmtiles.hsaco")
    text = subprocess.run(["/opt/rocm/llvm/bin/llvm-objdump", "-d", "--no-show-raw-insn", lib], stdout=subprocess.PIPE, text=True, check=True).stdout
    kernels = {m[1]: m[2] for m in re.finditer(r"<(gemm_entry__\w+%s)>:\n(.*?)(?=\n\n|\Z)" % WIDE, text, re.S)}
    assert sorted(kernels) == ["gemm_entry__bf16" + WIDE, "gemm_entry__f16" + WIDE]
    registers = lambda operand: set(range(int(operand[1] or operand[3]), int(operand[2] or operand[3]) + 1))
    for name, body in kernels.items():
        lines = [line.split("//")[0].strip() for line in body.splitlines()]
        at = [i for i, line in enumerate(lines) if line.startswith("v_mfma")]
        inputs, sums = set(), set()
        for i in at:
            ops = [registers(o) for o in re.finditer(r"v\[(\d+):(\d+)\]|\bv(\d+)\b", lines[i])]
            assert len(ops) == 4 and ops[0] == ops[3], lines[i]      # in place
            sums |= ops[0]
            inputs |= ops[1] | ops[2]
        assert len(at) == 2 * 72 and len(sums) == 144 and not sums & inputs, name
        for line in lines[at[0]:at[-1]]:
            assert not line.startswith("scratch_"), (name, line)
            if line.startswith("v_") and not line.startswith("v_mfma"):
                used = set().union(*(registers(o) for o in re.finditer(r"v\[(\d+):(\d+)\]|\bv(\d+)\b", line)))
                assert not used & sums, (name, line)
