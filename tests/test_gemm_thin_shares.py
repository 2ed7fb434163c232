"""Products of few rows whose K is dealt to the workgroups in single 64-row steps of their eight wavefronts (gemm_choice.h, thin_splits): one position short of
one more share and one past it, shares that are all of one step, and the largest count."""
import pytest
import torch

from util import rel_l2

KS = [(511, 1), (1023, 1), (1536, 3), (2047, 3), (2049, 4), (3001, 5), (4095, 7), (4097, 8), (7777, 8)]       # K positions, workgroups to a strip


@pytest.mark.parametrize("m,strip", [(1, 16), (16, 16), (17, 32), (32, 32), (33, 64), (64, 64)])
def test_k_goes_to_a_workgroup_for_each_eight_steps(fake_hip, m, strip):
    ct = fake_hip
    from test_host_abi import _workgroups
    for k, shares in KS:
        ct.gemm(ct.partition(torch.empty(m, 130, dtype=torch.bfloat16), [64, 64]), torch.empty(m, k, dtype=torch.bfloat16),
                torch.empty(k, 130, dtype=torch.bfloat16), k, accumulate=False, generics=["bf16", 64, 64, 1], variant=f"bf16_thin{strip}x64")
        assert _workgroups(ct) == 3 * shares, k


@pytest.mark.gpu
@pytest.mark.parametrize("m,strip", [(1, 16), (16, 16), (17, 32), (31, 32), (33, 64), (70, 64)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gpu_shares_of_one_step(ct, dev, m, strip, dtype):
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[dtype]
    g = torch.Generator(device="cuda").manual_seed(m)
    for k, _ in KS:
        xs = torch.full((m, k + 3), float("nan"), device=dev, dtype=dt)       # rows that go on behind K
        ys = torch.full((k, 135), float("nan"), device=dev, dtype=dt)
        xs[:, :k] = torch.randn(m, k, device=dev, generator=g).to(dt)
        ys[:, :130] = (torch.randn(k, 130, device=dev, generator=g) / k ** 0.5).to(dt)
        x, y = xs[:, :k], ys[:, :130]
        z = torch.full((m + 1, 130), 7.0, dtype=dt, device=dev)
        for _ in range(2):                                                    # the second launch finds the first one's counters at 0
            ct.gemm(ct.partition(z[:m], [64, 64]), x, y, k, accumulate=False, generics=[dtype, 64, 64, 1], variant=f"{dtype}_thin{strip}x64")
            # one rounding to the output type over f32 sums of k products
            want = x.double() @ y.double()
            assert rel_l2(z[:m].double().cpu().numpy(), want.cpu().numpy()) <= {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dtype], k
            assert torch.all(z[m] == 7.0)
