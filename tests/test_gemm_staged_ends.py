"""The register-staged GEMM tiles (gemm_small.hip, GemmStaged) at the ends of K: shorter than a 16-byte unit, cut at every place of a unit, one to
eight K tiles of 64, and the last tile among the loads in front of the loop; NaN behind every row, which a load past an end would bring in."""
import pytest
import torch

from util import rel_l2

TILES = {"staged64x64": 64, "staged64x128": 128, "staged128x128": 128, "staged256x128": 128, "staged256x256": 256}


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gpu_every_end_of_k(ct, dev, tile, dtype):
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(len(tile) + len(dtype))
    wide = TILES[tile] - 128 if TILES[tile] > 128 else 0                      # a tile lies inside the columns of y
    for m, n, k in [(70, 133, 1), (65, 131, 5), (3, 129, 8), (257, 135, 9), (70, 130, 64), (70, 131, 65), (66, 132, 66 + 64), (70, 133, 67 + 128), (70, 134, 68 + 192),
                    (70, 135, 69 + 256), (70, 136, 70 + 320), (70, 137, 71 + 384), (70, 138, 512), (301, 260, 447), (64, 128, 449)]:
        n += wide
        xs = torch.full((m, k + 3), float("nan"), device=dev, dtype=dt)       # rows that go on behind K
        ys = torch.full((k, n + 5), float("nan"), device=dev, dtype=dt)
        xs[:, :k] = torch.randn(m, k, device=dev, generator=g).to(dt)
        ys[:, :n] = (torch.randn(k, n, device=dev, generator=g) / k ** 0.5).to(dt)
        x, y = xs[:, :k], ys[:, :n]
        z = torch.full((m + 1, n), 7.0, dtype=dt, device=dev)
        ct.gemm(ct.partition(z[:m], [64, 64]), x, y, k, accumulate=False, generics=[dtype, 64, 64, 1], variant=f"{dtype}_{tile}")
        assert ct.last_resolved()["symbol"].endswith(tile)
        want = x.double() @ y.double()
        # one rounding to the output type over f32 sums of k products
        assert rel_l2(z[:m].double().cpu().numpy(), want.cpu().numpy()) <= {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype], (m, n, k)
        assert torch.all(z[m] == 7.0)
