"""Split decode attention whose last workgroup merges the splits (fmha.hip, merge_if_last) against the split kernel and the merge kernel with
memory of their own, bit for bit, where one takes the place of the other: one split, as many as there are lanes, one more; as many heads as
there are counters, one more; groups and head sizes; more launches in a row than there are sets of counters."""
import pytest
import torch

from test_zz_no_alloc import _reference_step


@pytest.mark.gpu
@pytest.mark.parametrize("heads,group,d,keys,splits,merged", [(1, 1, 64, 1, 1, True), (3, 2, 64, 700, 64, True), (2, 4, 64, 4097, 65, False), (64, 1, 128, 200, 4, True),
                                                              (65, 1, 128, 200, 4, False), (5, 2, 128, 333, 7, True), (4, 4, 128, 4096, 63, True), (2, 4, 256, 1000, 33, True),
                                                              (3, 1, 256, 90, 2, True), (2, 8, 128, 500, 8, False)])
def test_gpu_merge_in_the_split_launch(ct, dev, heads, group, d, keys, splits, merged):
    g = torch.Generator(device="cuda").manual_seed(heads * 1000 + group * 100 + d + splits)
    rand = lambda *shape: torch.randn(shape, device=dev, generator=g).half()
    k, v, scale = rand(heads, keys + 5, d), rand(heads, keys + 5, d), d ** -0.5
    out = torch.full((heads, group, d), float("nan"), dtype=torch.float16, device=dev)
    op = ct.partition(out, [1, group, d])
    for it in range(140 if heads == 5 else 3):
        q = rand(heads, group, d)
        p = torch.tensor([(keys - 1) >> it % 4], dtype=torch.int32, device=dev)          # splits without keys among them
        if it == 0:
            ct.fmha_decode_gqa_noalloc_prepare(q, k, v, op, p, splits)
        ct.fmha_decode_gqa_noalloc(q, k, v, op, scale, p, splits)
        assert ct.last_resolved()["symbol"].startswith("fmha_decode_gqa_split") == merged
        want = _reference_step(ct, dev, q, k, v, scale, p, 64, splits)
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))


@pytest.mark.gpu
def test_gpu_rows_of_out_off_16_bytes_take_the_two_kernels(ct, dev):
    q, kv = torch.randn(2, 2, 64, device=dev).half(), torch.randn(2, 100, 64, device=dev).half()
    p = torch.tensor([99], dtype=torch.int32, device=dev)
    out = torch.zeros(2, 2, 68, dtype=torch.float16, device=dev)[:, :, :64]
    ct.fmha_decode_gqa_noalloc(q, kv, kv, ct.partition(out, [1, 2, 64]), 0.125, p, 4)
    assert ct.last_resolved()["symbol"].startswith("splitk_reduce_merge")
    assert torch.equal(out, _reference_step(ct, dev, q, kv, kv, 0.125, p, 64, 4))
