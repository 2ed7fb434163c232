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


def test_shares_where_strips_fill_a_quarter_of_the_compute_units_and_more(fake_hip):
    """a short K of aligned rows in fewer shares than there are steps, even shares as they are, a second workgroup to a compute unit only for a
    shorter or a nearly full round; rows off 16-byte boundaries are shared as far as steps go"""
    ct = fake_hip
    from test_host_abi import _workgroups
    for m, n, k, shares in [(8, 5632, 1536, 1), (7, 4288, 2048, 2), (22, 7616, 1600, 1), (56, 7808, 1088, 1), (24, 5120, 1536, 3), (24, 3520, 1536, 3), (10, 4224, 2240, 3),
                            (12, 3072, 3072, 3), (1, 2048, 5120, 5), (1, 4480, 4096, 3), (3, 6080, 3072, 2), (1, 4096, 4096, 8), (1, 6144, 4096, 8), (1, 10304, 2496, 1),
                            (1, 9984, 2688, 3), (8, 5633, 1536, 3), (7, 4283, 2048, 4), (22, 7610, 1600, 2)]:
        x, y, z = torch.empty(m, k, dtype=torch.half), torch.empty(k, n, dtype=torch.half), torch.empty(m, n, dtype=torch.half)
        ct.gemm(ct.partition(z, [128, 128]), x, y, k, accumulate=False, generics=["f16", 128, 128, 1])
        assert "thin" in ct.last_resolved()["variant"] and _workgroups(ct) == -(-n // 64) * shares, (m, n, k, _workgroups(ct) / -(-n // 64))


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
