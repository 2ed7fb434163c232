"""The GEMM kernels between few rows and 256 x 256 tiles: register-staged tiles (any row alignment, K split over
workgroups) and the ring on 192 x 256, 128 x 256, 256 x 128 and 192 x 128 tiles."""
import numpy as np
import pytest
import torch

import oracle
from util import normal_bf16_bits, normal_f16_bits, rel_l2, to_dev_bf16, to_dev_f16

BOUND = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11, "bf16f32": 2e-6}      # unit roundoff of the output type (a few outputs can all sit near it); f32 sums


def _run(ct, dev, m, n, k, dtype, variant, accumulate, tile=(128, 128)):
    bits, to_dev = (normal_f16_bits, to_dev_f16) if dtype == "f16" else (normal_bf16_bits, to_dev_bf16)
    widen = oracle.f16_bits_to_f32 if dtype == "f16" else oracle.bf16_bits_to_f32
    a, b = bits((m, k), 931), bits((k, n), 932)
    out = {"bf16": torch.bfloat16, "f16": torch.float16, "bf16f32": torch.float32}[dtype]
    x, y = to_dev(a, dev), to_dev(b, dev)
    z0 = torch.from_numpy(oracle.normal_f32((m, n), 933)).to(dev).to(out)
    z = torch.full((m + 1, n), 7.0, dtype=out, device=dev)           # a row behind z that nothing may touch
    ref = widen(a).astype(np.float64) @ widen(b).astype(np.float64) + (z0.double().cpu().numpy() if accumulate else 0)
    for _ in range(2):                                                # the second launch finds the first one's counters at 0
        z[:m] = z0
        ct.gemm(ct.partition(z[:m], list(tile)), x, y, k, accumulate=accumulate, generics=[dtype, *tile, 1], variant=variant)
        torch.cuda.synchronize()
        assert rel_l2(z[:m].double().cpu().numpy(), ref) <= BOUND[dtype]
        assert torch.all(z[m] == 7.0)
    return ct.last_resolved()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", ["64x64", "64x128", "128x128", "256x128"])
@pytest.mark.parametrize("m,n,k", [(1, 128, 65), (65, 129, 64), (129, 255, 127), (128, 128, 200), (200, 131, 8), (67, 640, 4100), (130, 1001, 1030), (257, 260, 192)])
@pytest.mark.parametrize("dtype,accumulate", [("bf16", True), ("f16", False), ("bf16f32", True)])
def test_gpu_staged_gemm(ct, dev, tile, m, n, k, dtype, accumulate):
    _run(ct, dev, m, n, k, dtype, f"{dtype}_staged{tile}", accumulate)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", ["192x256x64_q2x4", "128x256x64_q2x4", "256x128x64_q4x2", "192x128x64_q2x2"])
@pytest.mark.parametrize("m,n,k", [(192, 256, 64), (257, 264, 72), (500, 520, 640), (1, 8, 1032)])
@pytest.mark.parametrize("dtype,accumulate", [("bf16", True), ("f16", False)])
def test_gpu_ring_tiles(ct, dev, tile, m, n, k, dtype, accumulate):
    _run(ct, dev, m, n, k, dtype, f"{dtype}_{tile}", accumulate, tile=(256, 256))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,aligned", [(300, 512, 2048, True), (1500, 1024, 1024, True), (300, 515, 1000, False), (2100, 129, 700, False)])
def test_gpu_medium_gemm_by_size(ct, dev, m, n, k, aligned):
    got = _run(ct, dev, m, n, k, "f16", None, True)
    assert got["source"] == "size" and ("_staged" in got["variant"] or (aligned and "_q" in got["variant"]))


def test_rows_of_x_or_columns_of_y_missing_leave_the_size_rule(fake_hip):
    """x with fewer rows, or y with fewer columns, than the output reads zeros there: the kernels of the size rule do not"""
    ct = fake_hip
    h = torch.half
    z = torch.empty(300, 512, dtype=h)
    ct.gemm(ct.partition(z, [128, 128]), torch.empty(300, 1001, dtype=h), torch.empty(1001, 512, dtype=h), 1001)
    assert "_staged" in ct.last_resolved()["variant"]
    ct.gemm(ct.partition(z, [128, 128]), torch.empty(299, 1001, dtype=h), torch.empty(1001, 512, dtype=h), 1001)
    assert ct.last_resolved()["variant"] == "f16_generic"
    ct.gemm(ct.partition(z, [128, 128]), torch.empty(300, 1001, dtype=h), torch.empty(1001, 511, dtype=h), 1001)
    assert ct.last_resolved()["variant"] == "f16_generic"


def test_staged_launches_split_what_the_size_rule_prices(fake_hip):
    """64 x 64 tiles share K between workgroups, the larger staged tiles never do: chosen by size or named by the caller"""
    ct = fake_hip
    from test_host_abi import _workgroups
    h = torch.half
    for m, n, k, variant, tiles, split in ((336, 2575, 1350, None, 6 * 21, False), (300, 515, 4000, None, 5 * 9, True),
                                           (336, 2575, 1350, "f16_staged64x64", 6 * 41, True), (300, 515, 4000, "f16_staged128x128", 3 * 5, False),
                                           (300, 515, 4000, "f16_staged64x128", 5 * 5, False), (300, 515, 4000, "f16_staged256x128", 2 * 5, False)):
        ct.gemm(ct.partition(torch.empty(m, n, dtype=h), [128, 128]), torch.empty(m, k, dtype=h), torch.empty(k, n, dtype=h), k, variant=variant)
        got = ct.last_resolved()["variant"]
        assert got == (variant or ("f16_staged64x64" if split else "f16_staged64x128"))
        assert _workgroups(ct) % tiles == 0 and (_workgroups(ct) > tiles) == split


def test_small_outputs_of_middling_inner_size_take_staged_tiles(fake_hip):
    """the size rule where the 128 x 128 ring was taken and is the slowest: few tiles of K between 512 and 1500, and somewhat more
    tiles than compute units"""
    ct = fake_hip
    buf = torch.empty(48 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
    for m, n, k, want in ((220, 64, 1408, "staged64x64"), (665, 320, 704, "staged64x64"), (221, 256, 1088, "staged64x64"), (562, 384, 640, "staged64x64"),
                          (1623, 2944, 14016, "192x128x64_q2x2"), (619, 8832, 4096, "256x128x64_q4x2"), (2048, 2048, 2048, "128x128x64_q2x2"),
                          (1500, 14336, 2048, "192x256x64_q2x4"), (4096, 4096, 4096, "256x256x64_q2x4")):
        ct.gemm(ct.partition(view(m, n), [128, 128]), view(m, k), view(k, n), k)
        assert ct.last_resolved()["variant"] == "f16_" + want, (m, n, k)
