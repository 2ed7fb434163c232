"""GEMM tiles of 320 to 448 columns (gemm_wide.h): which launches take them, ragged rows, columns that end in a tile's first unit and on its edge, an even and an
odd number of K tiles, rows further apart than they are long, z as the initial accumulator; and that the compiler moves no accumulator inside the K loop."""
import os
import re
import subprocess

import pytest
import torch

from util import rel_l2

FAMILY = "_192x256x64_q2x4_mix"
TILES = [(192, 320), (192, 384), (192, 448), (256, 320)]
symbol = lambda dtype, bm, bn: f"gemm_entry__{dtype}_w{bm}x{bn}{FAMILY}"
# each tile: rows that end in the last tile and columns in the first unit of one; whole tiles
SIZES = [(566, 22088, TILES[0]), (576, 22400, TILES[0]), (627, 22280, TILES[1]), (768, 22272, TILES[1]), (627, 25096, TILES[2]), (768, 25088, TILES[2]), (993, 17288, TILES[3]),
         (1024, 17280, TILES[3])]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("k,accumulate", [(576, False), (640, True)])
@pytest.mark.parametrize("m,n,tile", SIZES)
def test_gpu_wide_tiles(ct, dev, dtype, m, n, tile, k, accumulate):
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + 24, device=dev, generator=g).to(dt)[:, :k]
    y = (torch.randn(k, n + 8, device=dev, generator=g) / k ** 0.5).to(dt)[:, :n]
    z0 = torch.randn(m, n, device=dev, generator=g).to(dt)
    z = torch.full((m + 1, n + 8), 7.0, dtype=dt, device=dev)
    z[:m, :n] = z0
    ct.gemm(ct.partition(z[:m, :n], [256, 256]), x, y, k, accumulate=accumulate)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"] == symbol(dtype, *tile)
    want = x.double() @ y.double() + (z0.double() if accumulate else 0)
    # one rounding to the output type over f32 sums
    got, unit = z[:m, :n].double(), {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
    assert rel_l2(got.cpu().numpy(), want.cpu().numpy()) <= unit
    assert (got - want).abs().amax(0).max() <= unit * 1.01 * want.abs().max()      # no column was left out or written by two tiles
    assert torch.all(z[m] == 7.0) and torch.all(z[:, n:] == 7.0)


def test_which_sizes_take_them(fake_hip):
    """outputs that come out even on them; not with a ragged K, columns of z in units of 4, one round of other tiles, or a kernel named"""
    ct = fake_hip
    from test_gemm_tiles import _workgroups
    bufs = {"f16": torch.empty(120 << 20, dtype=torch.half), "bf16": torch.empty(120 << 20, dtype=torch.bfloat16)}
    for m, n, k, tile in [(m, n, k, tile) for m, n, tile in SIZES for k in (576, 640)] + [
            (1500, 14336, 4096, (192, 448)), (2048, 8960, 3584, (256, 320)), (1344, 12032, 4608, (192, 384)), (1344, 12032, 4616, None), (1344, 12036, 4608, None),
            (1024, 8192, 4096, None), (2048, 12288, 4096, None), (4096, 16384, 512, None)]:
        for dt, buf in bufs.items():
            view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
            ct.gemm(ct.partition(view(m, n), [256, 256]), view(m, k), view(k, (n + 7) // 8 * 8), k, accumulate=False, generics=[dt, 256, 256, 8])
            took = ct.last_resolved()["symbol"]
            if not tile:
                assert not re.search(r"_w\d+x", took), (m, n, k, took)
                continue
            assert took == symbol(dt, *tile) and _workgroups(ct) == -(-m // tile[0]) * -(-n // tile[1]), (m, n, k, took)
            ct.gemm(ct.partition(view(m, n), [256, 256]), view(m, k), view(k, n), k, accumulate=False, variant=dt + "_192x256x64_q2x4")
            assert not re.search(r"_w\d+x", ct.last_resolved()["symbol"])


def test_no_accumulator_is_moved_in_the_k_loop():
    """The matrix instructions of these kernels are written so that the compiler does not know them for such, and puts no wait states between one and another
    instruction on its result: between the first and the last of them there is no spill, and no move into or out of a register that they accumulate in."""
    lib = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutile-rs_amd", "lib", "gemmtiles.hsaco")
    text = subprocess.run(["/opt/rocm/llvm/bin/llvm-objdump", "-d", "--no-show-raw-insn", lib], stdout=subprocess.PIPE, text=True, check=True).stdout
    kernels = {m[1]: m[2] for m in re.finditer(r"<(gemm_entry__\w+_w\d+x\w+)>:\n(.*?)(?=\n\n|\Z)", text, re.S)}
    shapes = {symbol(dt, bm, bn): bm // 32 * bn // 64 for dt in ("f16", "bf16") for bm, bn in TILES}    # 16 x 16 blocks of a wavefront
    assert kernels.keys() == shapes.keys()
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
        assert len(at) == 2 * 2 * shapes[name] and len(sums) == 4 * shapes[name] and not sums & inputs, name
        for line in lines[at[0]:at[-1]]:
            assert not line.startswith("scratch_"), (name, line)
            if line.startswith("v_") and not line.startswith("v_mfma"):
                used = set().union(*(registers(o) for o in re.finditer(r"v\[(\d+):(\d+)\]|\bv(\d+)\b", line)))
                assert not used & sums, (name, line)
