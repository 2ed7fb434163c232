"""LM-head argmax of four blocks to the busiest compute unit (more than 768 of 64 rows, a workgroup to each): rows of more than 768 and up to 1024 columns take two rows a step there, and
the winners do not depend on which step a launch takes."""
import pytest
import torch


def _winners(ct, w, h):
    blocks = (w.shape[0] + 63) // 64
    best, index = torch.full((blocks,), float("nan"), dtype=torch.float32, device="cuda"), torch.zeros(blocks, dtype=torch.int32, device="cuda")
    ct.lm_head_argmax_blocks_f16(w, h, ct.partition(best, [1]), ct.partition(index, [1]), w.shape[0])
    return best, index


@pytest.mark.gpu
@pytest.mark.parametrize("k", [768, 800, 960, 1024])
@pytest.mark.parametrize("blocks", [768, 769, 853])
def test_gpu_two_and_eight_rows_agree(ct, k, blocks):
    """bit for bit: a lane's sums run over the same columns in the same order; the first 500 blocks by themselves are on eight rows"""
    g = torch.Generator(device="cuda").manual_seed(k + blocks)
    w = torch.randn(blocks * 64 - 5, k, dtype=torch.float16, device="cuda", generator=g)
    h = torch.randn(1, k, dtype=torch.float16, device="cuda", generator=g)
    best, index = _winners(ct, w, h)
    few, few_index = _winners(ct, w[:500 * 64], h)
    assert torch.equal(best[:500], few) and torch.equal(index[:500], few_index)
    logits = w.double() @ h[0].double()
    bound = (w.double().abs() @ h[0].double().abs()).max() * k * 2.0**-24      # k roundings of at most the sum of magnitudes
    assert (best.double() - logits[index.long()]).abs().max() <= bound and torch.equal(index.long() // 64, torch.arange(blocks, device="cuda"))
    assert (torch.nn.functional.pad(logits, (0, 5), value=-1e30).view(blocks, 64).max(1).values - logits[index.long()]).max() <= 2 * bound
