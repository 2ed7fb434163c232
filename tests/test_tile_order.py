"""Every output tile is computed once whatever their number: the order that gives each XCD a contiguous share of the tiles."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", [(1, 1), (1, 7), (9, 1), (3, 3), (8, 2), (11, 13)])
@pytest.mark.parametrize("tile,variant", [(256, "f16_256x256x64_q2x4"), (128, "f16_128x128x64_d2x2")])
def test_gpu_every_tile_once(ct, dev, tiles, tile, variant):
    m, n, k = tiles[0] * tile, tiles[1] * tile, 128
    rows, cols = torch.arange(m, device=dev)[:, None], torch.arange(n, device=dev)[None, :]
    x, y = torch.zeros(m, k, device=dev), torch.zeros(k, n, device=dev)
    x[:, 0], x[:, 1] = (rows[:, 0] // tile) * 16, 1                    # z[r, c] = 16 * tile row + tile column + 1, exact in f16
    y[0], y[1] = 1, cols[0] // tile + 1
    z = torch.zeros(m, n, dtype=torch.half, device=dev)
    ct.gemm(ct.partition(z, [tile, tile]), x.half(), y.half(), k, accumulate=True, variant=variant)   # a tile computed twice would double
    torch.cuda.synchronize()
    assert torch.equal(z, ((rows // tile) * 16 + cols // tile + 1).half())


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", [(1, 1), (3, 3), (4, 2), (9, 11)])
def test_gpu_every_tile_once_of_one_k_tile(ct, dev, tiles):
    """K = 64 takes another order where the tiles are no multiple of 8"""
    tm, tn = tiles
    m, n = tm * 256 - 5, tn * 256 - 16
    rows, cols = torch.arange(m, device=dev)[:, None] // 256, torch.arange(n, device=dev)[None, :] // 256
    x, y = torch.zeros(m, 64, device=dev), torch.zeros(64, n, device=dev)
    x[:, 0], x[:, 1], y[0], y[1] = rows[:, 0] * 16, 1, 1, cols[0] + 1
    z = torch.zeros(m, n, dtype=torch.half, device=dev)
    ct.gemm(ct.partition(z, [256, 256]), x.half(), y.half(), 64, accumulate=True, variant="f16_256x256x64_q2x4")
    torch.cuda.synchronize()
    assert torch.equal(z, (rows * 16 + cols + 1).half())
