"""Partial sums of outputs whose K is shared by more workgroups than are read at once (split_k.h): nine and sixteen of them, one row to a full strip."""
import pytest
import torch

from util import rel_l2


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k,splits", [(1, 64, 9216, 9), (15, 67, 9300, 9), (16, 64, 16384, 16), (17, 130, 10240, 10), (33, 64, 16389, 16), (48, 65, 9216, 9)])
def test_gpu_sums_of_more_than_eight_splits(ct, dev, m, n, k, splits, dtype):
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


def test_as_many_splits_as_the_test_above_means(fake_hip):
    ct = fake_hip
    from test_gemm_tiles import _workgroups
    buf = torch.empty(1 << 21, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
    for m, n, k, splits in ((1, 64, 9216, 9), (16, 64, 16384, 16), (33, 64, 16389, 16)):
        ct.gemm(ct.partition(view(m, n), [64, 64]), view(m, k), view(k, n), k, generics=["f16", 64, 64, 1])
        assert "thin" in ct.last_resolved()["variant"] and _workgroups(ct) == splits, (m, n, k, _workgroups(ct))
