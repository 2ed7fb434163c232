"""Causal attention at D = 128 on two rounds of 64-row workgroups that share their keys: long keys whose tiles differ in length (few keys in front of the
rows), and not otherwise."""
import pytest
import torch

from test_fmha_keys import _call, _close, _reference

TAKES = [   # heads, rows, keys in front of them, on two rounds
    (8, 4096, 0, True), (8, 3072, 0, True), (8, 3071, 0, False), (4, 8192, 1024, True), (4, 8192, 2048, False), (8, 2408, 1204, True), (8, 2408, 4816, False),
    (6, 3240, 900, True), (8, 4097, 0, False), (32, 1024, 3000, False), (40, 512, 7000, False), (16, 2048, 1024, False),
]


@pytest.mark.parametrize("heads,rows,start,takes", TAKES)
def test_keys_in_front_of_the_rows(fake_hip, heads, rows, start, takes):
    ct = fake_hip
    from test_host_abi import _last
    q, kv, out = torch.empty(rows, heads, 128).half(), torch.empty(heads, rows + start, 128).half(), torch.empty(rows, heads, 128).half()
    ct.fmha_seq_f16(q, kv, kv, ct.partition(out, [128, 1, 128]), 0.1, 1, kv_len=rows + start, query_start=start)
    seq = _last(ct)[0].symbol.decode(), tuple(_last(ct)[0].grid)
    q, kv, out = torch.empty(1, heads, rows, 128).half(), torch.empty(1, heads, rows + start, 128).half(), torch.empty(heads, rows, 128).half()
    ct.fmha(ct.partition(out, [1, 256, 128]), q, kv, kv, 0.1, start, 1, causal=True)
    assert seq == (_last(ct)[0].symbol.decode(), tuple(_last(ct)[0].grid))
    assert seq == (("fmha_entry__f16_64x128x128_keys", (heads, -(-rows // 64), 1)) if takes else ("fmha_entry__f16_256x64x128_pp", (heads, -(-rows // 256), 1)))


def test_a_position_that_only_the_device_knows(fake_hip):
    ct = fake_hip
    from test_host_abi import _last
    q, kv = torch.empty(1024, 32, 128).half(), torch.empty(8, 8192, 128).half()
    ct.fmha_seq_f16(q, kv, kv, ct.partition(torch.empty_like(q), [128, 1, 128]), 0.1, 4, position_start=torch.zeros(1, dtype=torch.int32))
    assert _last(ct)[0].symbol == b"fmha_seq_entry__f16_64x128x128_keys"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("heads,group,rows,start", [(8, 4, 3100, 0), (6, 1, 2775, 301), (5, 1, 3333, 0)])
def test_gpu_two_rounds(ct, dev, dtype, heads, group, rows, start):
    q, k, v, out = _call(ct, dtype, 1, heads, group, rows, rows + start, 128, True, pos=start, bm=256, dev=dev)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_64x128x128_keys")
    assert _close(out, _reference(q, k, v, 128 ** -0.5, start, group, True), dtype)
