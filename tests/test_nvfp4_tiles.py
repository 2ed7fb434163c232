"""NVFP4 products on whole tiles (nvfp4_gemm.hip): one to seven K tiles of 64 (an odd number is followed by one of zeros), edges of the tiles in both
directions, and outputs of a 128 x 128 partition that 256 x 256 tiles compute."""
import pytest
import torch

import oracle
from util import rel_l2


def _dev(a, dev):
    return torch.from_numpy(a).to(dev)


@pytest.mark.gpu
@pytest.mark.parametrize("variant", ["32x32x64_w1x1", "64x64x64_w1x1", "128x128x64_w2x2", "256x256x64_q2x4", "256x256x64_q4x2", "256x256x64_w4x2"])
@pytest.mark.parametrize("m,n,tiles", [(1, 4, 1), (130, 132, 2), (257, 260, 3), (128, 256, 6), (300, 516, 7)])
def test_gpu_tiles_of_k(ct, dev, variant, m, n, tiles):
    k = 64 * tiles
    xq, xs = oracle.nvfp4_quantize(oracle.normal_f32((m, k), 971))
    yq, ys = oracle.nvfp4_quantize(oracle.normal_f32((n, k), 972))
    ref = oracle.nvfp4_gemm_f32(xq, yq, xs, ys, 0.5)
    z = torch.full((m + 1, n), 7.0, dtype=torch.float32, device=dev)
    ct.linear_tile_nvfp4(ct.partition(z[:m], [int(variant.split("x")[0])] * 2), *[_dev(v, dev) for v in (xq, yq, xs, ys)], 0.5, variant="f32_" + variant)
    assert rel_l2(z[:m].cpu().numpy(), ref) <= 2e-6          # exact products, f32 sums of at most 448 of them in another order
    assert torch.all(z[m] == 7.0)


def test_size_rule_of_a_128_partition(fake_hip):
    """whole outputs of 240 tiles of 256 x 256 run on those, of a few more than 256 on 128 x 128, of few rows on strips, and of a long K in some rounds too"""
    ct = fake_hip
    for m, n, k, want in ((2476, 6080, 896, "256x256x64_q2x4"), (2940, 5568, 1152, "128x128x64_w2x2"), (200, 14336, 4096, "flat128x128"), (8, 4096, 4096, "flat16x64"),
                          (1587, 3328, 7040, "flat64x128"), (3174, 1472, 7168, "flat64x64"), (305, 11456, 1664, "flat64x128")):
        u8 = lambda rows, cols: torch.empty(rows, cols, dtype=torch.uint8)
        ct.linear_tile_nvfp4(ct.partition(torch.empty(m, n, dtype=torch.bfloat16), [128, 128]), u8(m, k // 2), u8(n, k // 2), u8(m, k // 16), u8(n, k // 16), 1.0)
        assert ct.last_resolved()["variant"] == "bf16_" + want


def test_two_tiles_of_k_in_a_256_partition(fake_hip):
    """up to K = 128 the output of a 256 x 256 partition runs on 128 x 128 tiles while they are one round, two to a compute unit"""
    ct = fake_hip
    u8 = lambda rows, cols: torch.empty(rows, cols, dtype=torch.uint8)
    for m, n, k, want in ((256, 128, 128, "128x128x64_w2x2"), (988, 5056, 64, "128x128x64_w2x2"), (2048, 4096, 128, "128x128x64_w2x2"),
                          (2048, 4224, 128, "256x256x64_q2x4"), (256, 512, 256, "256x256x64_q2x4")):
        ct.linear_tile_nvfp4(ct.partition(torch.empty(m, n), [256, 256]), u8(m, k // 2), u8(n, k // 2), u8(m, k // 16), u8(n, k // 16), 1.0)
        assert ct.last_resolved()["variant"] == "f32_" + want, (m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 4, 64), (257, 260, 128), (130, 516, 64), (300, 1000, 128)])
def test_gpu_two_tiles_of_k_in_a_256_partition(ct, dev, m, n, k):
    xq, xs = oracle.nvfp4_quantize(oracle.normal_f32((m, k), 981))
    yq, ys = oracle.nvfp4_quantize(oracle.normal_f32((n, k), 982))
    z = torch.full((m + 1, n), 7.0, dtype=torch.float32, device=dev)
    ct.linear_tile_nvfp4(ct.partition(z[:m], [256, 256]), *[_dev(v, dev) for v in (xq, yq, xs, ys)], 0.5)
    assert ct.last_resolved()["variant"] == "f32_128x128x64_w2x2"
    assert rel_l2(z[:m].cpu().numpy(), oracle.nvfp4_gemm_f32(xq, yq, xs, ys, 0.5)) <= 2e-6          # exact products, f32 sums of at most 128 of them in another order
    assert torch.all(z[m] == 7.0)
