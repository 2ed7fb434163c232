"""Attention at D = 64 with two wavefronts to 32 query rows (fmha_keys.hip, "halves"): launches of many tiles, ragged in rows and keys, key groups, keys hidden
from every row of a wavefront, and a position on the device."""
import pytest
import torch

from test_fmha_keys import _call, _close, _reference


@pytest.mark.parametrize("heads,rows,causal,takes", [
    (32, 2048, False, True), (32, 2049, True, True), (160, 221, False, False), (112, 447, False, False), (96, 448, False, True), (260, 300, False, True), (260, 299, False, False),
    (160, 256, True, False), (160, 257, True, True), (300, 199, True, False), (300, 200, True, True), (128, 578, True, False), (132, 600, True, True), (192, 294, True, False), (80, 931, True, False), (64, 1100, True, True), (512, 150, True, False),
    (240, 380, True, True),
])
def test_which_launches_have_two_wavefronts_to_a_row_block(fake_hip, heads, rows, causal, takes):
    """D = 64, of 256 compute units: a round is 512 workgroups"""
    ct = fake_hip
    from test_host_abi import _last
    _call(ct, torch.half, 1, heads, 1, rows, rows, 64, causal)
    assert _last(ct)[0].symbol.decode() == "fmha_entry__f16_128x64x64" + ("_halves" if takes else "")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("batch,heads,group,rows,keys,causal,pos", [
    (1, 600, 4, 5, 301, True, 296), (2, 36, 4, 449, 640, True, 191), (1, 130, 1, 257, 257, True, 0), (1, 130, 2, 256, 1000, False, 0), (1, 72, 8, 500, 333, True, 100),
    (3, 24, 1, 1025, 1025, False, 0),
])
def test_gpu_two_wavefronts_to_a_row_block(ct, dev, dtype, batch, heads, group, rows, keys, causal, pos):
    q, k, v, out = _call(ct, dtype, batch, heads, group, rows, keys, 64, causal, pos=pos, dev=dev)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_128x64x64_halves")
    assert _close(out, _reference(q, k, v, 64 ** -0.5, pos, group, causal), dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,start,on_device", [(600, 0, False), (450, 301, True)])
def test_gpu_sequence_form(ct, dev, rows, start, on_device):
    g = torch.Generator().manual_seed(rows)
    normal = lambda *s: torch.randn(*s, generator=g).half().to(dev)
    q, k, v = normal(rows, 80, 64), normal(20, 900, 64), normal(20, 900, 64)
    out = torch.full((rows, 80, 64), 7.0, dtype=torch.half, device=dev)
    where = dict(position_start=torch.tensor([start], dtype=torch.int32, device=dev)) if on_device else dict(kv_len=start + rows, query_start=start)
    ct.fmha_seq_f16(q, k, v, ct.partition(out, [64, 1, 64]), 0.125, 4, **where)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"] == ("fmha_seq" if on_device else "fmha") + "_entry__f16_128x64x64_halves"
    seen = 900 if on_device else start + rows
    assert _close(out.permute(1, 0, 2), _reference(q.permute(1, 0, 2)[None], k[None, :, :seen], v[None, :, :seen], 0.125, start, 4, True), torch.half)
