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
