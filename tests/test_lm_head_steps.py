"""LM-head argmax (lm_head_argmax_blocks_entry__f16, elementwise.hip): steps of 2048 columns of two rows, and of 512 columns of eight where those would be less than three quarters
(runs of blocks: seven eighths) full, at the sizes around that rule and with one, a few and several blocks to a workgroup."""

import pytest
import torch


# K: one partial span; the last of eight rows below 2048 columns and the first of two; past one full step; a span short of two steps; ragged last spans
@pytest.mark.gpu
@pytest.mark.parametrize("k", [32, 512, 544, 1536, 1568, 2048, 2080, 3072, 3616, 4608, 5152])
@pytest.mark.parametrize("vocab", [61, 64 * 521 - 3, 64 * 1030])
def test_gpu_blocks_winners(ct, k, vocab):
    g = torch.Generator(device="cuda").manual_seed(k * 7 + vocab)
    w = torch.randn(vocab, k, dtype=torch.float16, device="cuda", generator=g)
    h = torch.randn(1, k, dtype=torch.float16, device="cuda", generator=g)
    blocks = (vocab + 63) // 64
    best = torch.full((blocks,), float("nan"), dtype=torch.float32, device="cuda")
    index = torch.zeros(blocks, dtype=torch.uint32, device="cuda")
    ct.lm_head_argmax_blocks_f16(w, h, ct.partition(best, [1]), ct.partition(index, [1]), vocab)
    logits = torch.full((blocks * 64,), -1e30, dtype=torch.float64, device="cuda")
    logits[:vocab] = w.double() @ h[0].double()
    logits = logits.view(blocks, 64)
    # an f32 sum of k products, each rounded once: k roundings of at most the sum of magnitudes
    bound = (w.double().abs() @ h[0].double().abs()).max() * k * 2.0**-24
    assert (best.double() - logits.max(1).values).abs().max() <= bound
    taken = logits.gather(1, (index.long() % 64).view(-1, 1))[:, 0]
    assert torch.equal(index.long() // 64, torch.arange(blocks, device="cuda"))
    assert (logits.max(1).values - taken).max() <= 2 * bound


@pytest.mark.parametrize("blocks,k,runs", [(1792, 4096, True), (1700, 4096, False), (2150, 1024, False), (2194, 4096, False), (2195, 4096, True), (2304, 4096, True)])
def test_runs_that_single_blocks_even_out(fake_hip, blocks, k, runs):
    """more than a sixth above the mean run, and fewer blocks on the busiest compute unit"""
    from test_host_abi import _workgroups
    ct = fake_hip
    ct.lm_head_argmax_blocks_f16(torch.empty(1, 1, dtype=torch.half).expand(blocks * 64, k), torch.empty(1, k, dtype=torch.half),
                                 ct.partition(torch.empty(blocks), [1]), ct.partition(torch.empty(blocks, dtype=torch.int32), [1]), blocks * 64)
    assert _workgroups(ct) == (512 if runs else blocks)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [512, 1024, 2048])
def test_gpu_rows_without_an_order(ct, k):
    # equal rows: the smallest index wins; a NaN in a block's first row stays its winner, infinities compare as numbers
    w = torch.ones(64 * 5, k, dtype=torch.float16, device="cuda")
    w[64, 0] = float("nan")
    w[128 + 7, 0] = float("inf")
    w[192:256, 0] = float("-inf")
    h = torch.ones(1, k, dtype=torch.float16, device="cuda")
    best = torch.zeros(5, dtype=torch.float32, device="cuda")
    index = torch.zeros(5, dtype=torch.uint32, device="cuda")
    ct.lm_head_argmax_blocks_f16(w, h, ct.partition(best, [1]), ct.partition(index, [1]), 64 * 5 - 10)
    assert index.tolist() == [0, 64, 135, 192, 256]
    assert best[[0, 2, 3, 4]].tolist() == [k, float("inf"), float("-inf"), k] and best[1].isnan()
