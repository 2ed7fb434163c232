"""Partial sums of outputs whose K is shared by more workgroups than are read at once (split_k.h): nine and sixteen of them, one row to a full strip."""
import os
import re
import subprocess

import pytest
import torch

from util import rel_l2


SHAPES = [(1, 64, 9216, 9), (15, 67, 9300, 9), (16, 64, 16384, 16), (17, 130, 10240, 10), (33, 64, 16389, 16), (48, 65, 9216, 9)]   # workgroups to a strip, f16 and bf16


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [s[:3] for s in SHAPES])
def test_gpu_sums_of_more_than_eight_splits(ct, dev, m, n, k, dtype):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device=dev, generator=g).to(dtype)
    y = (torch.randn(k, n, device=dev, generator=g) / k ** 0.5).to(dtype)
    z0 = torch.randn(m, n, device=dev, generator=g).to(dtype)
    want = z0.double() + x.double() @ y.double()
    name = {torch.float16: "f16", torch.bfloat16: "bf16", torch.float32: "f32"}[dtype]
    first = None
    for _ in range(3):                                  # later launches find the counters at 0 and the same sum in the same order
        z = torch.full((m + 1, n), 7.0, dtype=dtype, device=dev)          # a row behind z that nothing may touch
        z[:m] = z0
        ct.gemm(ct.partition(z[:m], [64, 64]), x, y, k, generics=[name, 64, 64, 1])
        torch.cuda.synchronize()
        # one rounding to the output type over f32 sums of k products (f32: 2^-24 an addition, K / 512 of them in a row and the splits')
        assert rel_l2(z[:m].double().cpu().numpy(), want.cpu().numpy()) <= {"f16": 2.0 ** -11, "bf16": 2.0 ** -8, "f32": 4e-6}[name]
        assert torch.all(z[m] == 7.0)
        assert first is None or torch.equal(first, z)
        first = z


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_as_many_splits_as_the_test_above_means(fake_hip, dtype):
    """f32 strips share K by powers of two: sixteen of them in each of the six"""
    ct = fake_hip
    from test_gemm_tiles import _workgroups
    for m, n, k, splits in SHAPES:
        ct.gemm(ct.partition(torch.empty(m, n, dtype=dtype), [64, 64]), torch.empty(m, k, dtype=dtype), torch.empty(k, n, dtype=dtype), k)
        variant = ct.last_resolved()["variant"]
        rows, cols = map(int, variant.split("strip" if dtype == torch.float32 else "thin")[1].split("x"))
        strips = -(-m // rows) * -(-n // cols)
        assert _workgroups(ct) == strips * (16 if dtype == torch.float32 else splits), (m, n, k, variant, _workgroups(ct))


def test_no_wide_store_leaves_its_data_unguarded():
    """A 16-byte buffer store with its offset in a scalar register reads its data registers for some cycles after it issues; the compiler guards their next write only
    where there is no such offset.  In every code object each store of that form has two idle cycles behind it."""
    lib = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutile-rs_amd", "lib")
    objects = sorted(f for f in os.listdir(lib) if f.endswith(".hsaco"))
    assert "gemmsmall.hsaco" in objects
    guarded = 0
    for name in objects:
        text = subprocess.run(["/opt/rocm/llvm/bin/llvm-objdump", "-d", "--no-show-raw-insn", os.path.join(lib, name)], stdout=subprocess.PIPE, text=True, check=True).stdout
        lines = text.splitlines()
        for store, behind in zip(lines, lines[1:]):
            if re.match(r"\s*buffer_store_dwordx[34] v\[\d+:\d+\], (v\d+|off), s\[\d+:\d+\], (s\d+|m0|vcc|exec|ttmp)", store):
                assert re.match(r"\s*s_nop [1-9]", behind), (name, store, behind)
                guarded += 1
    assert guarded > 0      # those of the streaming kernels, which wait by themselves
