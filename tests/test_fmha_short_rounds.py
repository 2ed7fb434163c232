"""Causal attention at D = 128 of 830 to 3000 keys on two rounds of 64-row workgroups: which launches take them, and results there."""
import pytest
import torch

from test_fmha_keys import _call, _close, _reference

TAKES = [   # heads, rows, keys in front of them, on two rounds
    (8, 2312, 0, True), (16, 1355, 0, True), (20, 868, 0, True), (24, 830, 0, True), (24, 829, 0, False), (20, 830, 0, False), (24, 1100, 0, True), (24, 1099, 0, False), (12, 2664, 0, True), (8, 3000, 0, True),
    (8, 3001, 0, False), (12, 2800, 0, False), (16, 1355, 1, False), (8, 2048, 0, True),
]


@pytest.mark.parametrize("heads,rows,start,takes", TAKES)
def test_which_launches(fake_hip, heads, rows, start, takes):
    ct = fake_hip
    from test_host_abi import _last
    q, kv, out = torch.empty(1, heads, rows, 128).half(), torch.empty(1, heads, rows + start, 128).half(), torch.empty(heads, rows, 128).half()
    for causal in (True, False):
        ct.fmha(ct.partition(out, [1, 256, 128]), q, kv, kv, 0.1, start, 1, causal=causal)
        rec = _last(ct)[0]
        on_64 = (takes and causal) or heads * -(-rows // 64) <= 256
        assert (rec.symbol.decode(), tuple(rec.grid)) == (("fmha_entry__f16_64x128x128_keys", (heads, -(-rows // 64), 1)) if on_64 else ("fmha_entry__f16_256x64x128_pp", (heads, -(-rows // 256), 1)))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("heads,group,rows", [(24, 4, 830), (24, 1, 1100), (12, 4, 1999)])
def test_gpu_short_rounds(ct, dev, dtype, heads, group, rows):
    q, k, v, out = _call(ct, dtype, 1, heads, group, rows, rows, 128, True, bm=256, dev=dev)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_64x128x128_keys")
    assert _close(out, _reference(q, k, v, 128 ** -0.5, 0, group, True), dtype)
