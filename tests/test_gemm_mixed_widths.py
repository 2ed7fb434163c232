"""GEMM outputs of one to two rounds of 192 x 256 tiles, whose second round is of 192 x 192 (gemm_tiles.h): which launches take the mix, ragged rows, columns
that end inside a narrow tile, inside its last fragment row and on its edge, ragged K, and z as the initial accumulator."""
import pytest
import torch

from util import rel_l2


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,n,k,accumulate", [(1500, 14336, 1024, False), (1344, 12032, 1096, True), (900, 18440, 1024, False), (701, 25600, 1032, True), (560, 28672, 1024, False)])
def test_gpu_two_widths_in_one_launch(ct, dev, dtype, m, n, k, accumulate):
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device=dev, generator=g).to(dt)
    y = (torch.randn(k, n, device=dev, generator=g) / k ** 0.5).to(dt)
    z0 = torch.randn(m, n, device=dev, generator=g).to(dt)
    z = torch.full((m + 1, n), 7.0, dtype=dt, device=dev)
    z[:m] = z0
    ct.gemm(ct.partition(z[:m], [256, 256]), x, y, k, accumulate=accumulate, generics=[dtype, 256, 256, 1], variant=f"{dtype}_192x256x64_q2x4")
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_mix")
    want = x.double() @ y.double() + (z0.double() if accumulate else 0)
    # one rounding to the output type over f32 sums
    assert rel_l2(z[:m].double().cpu().numpy(), want.cpu().numpy()) <= {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
    edge = (z[:m].double() - want).abs().amax(0)                       # no column was left out or written by two tiles
    assert edge.max() <= {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype] * 1.01 * want.abs().max()
    assert torch.all(z[m] == 7.0)


def test_launch_of_two_widths(fake_hip):
    """8 rows of tiles and 256 compute units: 32 wide columns, and narrow ones for the rest; a full second round, or none, keeps one width"""
    ct = fake_hip
    from test_gemm_tiles import _workgroups
    buf = torch.empty(60 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
    for m, n, k, mix, groups in ((1500, 14336, 4096, True, 8 * (32 + 32)), (1344, 12032, 4608, True, 7 * (36 + 15)), (1536, 16384, 3072, False, 512), (1536, 8192, 4096, False, 256)):
        ct.gemm(ct.partition(view(m, n), [256, 256]), view(m, k), view(k, n), k, variant="f16_192x256x64_q2x4")
        assert ct.last_resolved()["symbol"].endswith("_mix") == mix and _workgroups(ct) == groups, (m, n, k)


def test_which_sizes_take_two_widths(fake_hip):
    """nobody names a kernel: f16 and bf16, partitions of 256 x 256 and of 128 x 128; two rounds of one width and outputs of one round keep that"""
    ct = fake_hip
    bufs = {dt: torch.empty(118 << 20, dtype=dt) for dt in (torch.half, torch.bfloat16)}
    for m, n, k, mix in ((1344, 12032, 4608, True), (900, 18432, 5120, True), (560, 28672, 4096, True), (2048, 8960, 3584, True), (1536, 16384, 3072, False), (1536, 8192, 4096, False)):
        for dt, buf in bufs.items():
            view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
            for tile in (256, 128):
                ct.gemm(ct.partition(view(m, n), [tile, tile]), view(m, k), view(k, n), k, accumulate=False)
                assert ct.last_resolved()["symbol"].endswith("_192x256x64_q2x4" + ("_mix" if mix else "")), (m, n, k, dt, tile, ct.last_resolved()["symbol"])
