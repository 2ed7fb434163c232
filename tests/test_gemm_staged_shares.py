"""64 x 64 staged tiles of aligned rows, by how many workgroups share their K (staged_plan, gemm_choice.h): which launches share it and how, and results there."""
import pytest
import torch

from util import rel_l2

# m, n, k, workgroups to a tile
SIZES = [(272, 2176, 1536, 1), (230, 3072, 1024, 1), (557, 1408, 1728, 1), (374, 1344, 1024, 1), (403, 960, 1344, 2), (222, 1152, 3520, 3), (587, 256, 9024, 6)]


def test_how_many_share_a_tile(fake_hip):
    ct = fake_hip
    from test_gemm_tiles import _new_stream, _workgroups
    buf = torch.empty(16 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)

    def launch(m, n, k, **kw):
        ct.gemm(ct.partition(view(m, n), [128, 128]), view(m, k), view(k, n), k, **kw)
        return ct.last_resolved()["variant"], _workgroups(ct) / (-(-m // 64) * -(-n // 64))

    for m, n, k, shares in SIZES:
        assert launch(m, n, k) == ("f16_staged64x64", shares), (m, n, k, launch(m, n, k))
    # more tiles than two to a compute unit, and strips: as before
    assert launch(1500, 4096, 4096)[0] != "f16_staged64x64" and launch(40, 2240, 2304)[0] == "f16_thin64x64"
    # a long K unshared is dearer from memory than from the caches
    assert launch(262, 2240, 2304)[0] == launch(174, 2048, 2048)[0] == "f16_128x128x64_q2x2"
    # a kernel that the caller names shares K as it always did
    assert launch(262, 2240, 2304, variant="f16_staged64x64") == ("f16_staged64x64", 2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("m,n,k,shares", SIZES)
def test_gpu_shares(ct, dev, dtype, m, n, k, shares):
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, device=dev, generator=g).to(dt)
    y = (torch.randn(k, n, device=dev, generator=g) / k ** 0.5).to(dt)
    z = torch.full((m + 1, n), 7.0, dtype=dt, device=dev)
    for _ in range(2):      # the counters of a shared tile are ready for the next launch
        ct.gemm(ct.partition(z[:m], [128, 128]), x, y, k, accumulate=False)
    torch.cuda.synchronize()
    assert ct.last_resolved()["variant"] == dtype + "_staged64x64"
    # one rounding to the output type over f32 sums
    assert rel_l2(z[:m].double().cpu().numpy(), (x.double() @ y.double()).cpu().numpy()) <= {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype]
    assert torch.all(z[m] == 7.0)
