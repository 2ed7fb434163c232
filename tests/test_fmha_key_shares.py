"""Attention of few query tiles whose keys several workgroups share (their results meet in the stream's workspace), and the 64-row kernel of few keys"""
import pytest
import torch

from test_fmha_keys import _call, _close, _reference


# ---- launcher on the recording runtime (CPU) ----------------------------------------------------
@pytest.mark.parametrize("heads,rows,start,d,tile,shares", [
    (8, 17, 3905, 128, 32, 8), (8, 17, 200, 128, 32, 1), (8, 17, 256, 128, 32, 1), (1, 129, 2000, 128, 32, 9), (128, 32, 8000, 128, 32, 2), (129, 32, 8000, 128, 32, 1),
    (20, 50, 7299, 128, 32, 6), (4, 40, 4000, 64, 32, 8), (16, 1000, 0, 64, 64, 1), (40, 200, 900, 64, 64, 1), (9, 800, 4000, 64, 32, 1),
])
def test_shares_of_a_launch(fake_hip, heads, rows, start, d, tile, shares):
    """one round of workgroups at most, at least a key step to each"""
    ct = fake_hip
    from test_host_abi import _last
    q, kv = torch.empty(rows, heads, d).half(), torch.empty(heads, rows + start, d).half()
    ct.fmha_seq_f16(q, kv, kv, ct.partition(torch.empty_like(q), [128, 1, d]), 0.1, 1, kv_len=rows + start, query_start=start)
    rec = _last(ct)[0]
    assert rec.symbol.decode().endswith(f"_{tile}x{8192 // tile}x{d}_keys")
    assert tuple(rec.grid) == (heads, -(-rows // tile), shares) and (shares == 1 or heads * -(-rows // tile) * shares <= 256)


def test_few_keys_on_64_rows(fake_hip):
    ct = fake_hip
    from test_host_abi import _last
    for keys, few in ((129, True), (256, True), (257, False)):
        _call(ct, torch.bfloat16, 1, 64, 1, keys if keys < 256 else 256, keys, 128, False, bm=256)
        assert _last(ct)[0].symbol == (b"fmha_entry__bf16_few_64x128x128_keys" if few else b"fmha_entry__bf16_64x128x128_keys")


# ---- HIP kernels (GPU) --------------------------------------------------------------------------
@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("heads,group,rows,start,on_device", [
    (8, 4, 17, 3905, False), (2, 1, 33, 511, False), (4, 4, 1, 4096, False), (1, 1, 129, 1000, False), (20, 4, 50, 2299, False), (4, 2, 200, 1500, False),
    (8, 4, 130, 1333, True), (2, 1, 300, 0, True),
])
def test_gpu_keys_shared_by_workgroups(ct, dev, d, heads, group, rows, start, on_device):
    """against 64 bits, twice on the same workspace; behind the last key lies what must not be seen; and from inside a captured graph, where keys are not shared"""
    g = torch.Generator().manual_seed(rows)
    normal = lambda *s: torch.randn(*s, generator=g).half().to(dev)
    there = start + rows + 40
    q, k, v = normal(rows, heads, d), normal(heads // group, there, d), normal(heads // group, there, d)
    k[:, start + rows:], v[:, start + rows:] = 100.0, float("nan") if not on_device else 100.0
    out = [torch.full((rows, heads, d), 7.0, dtype=torch.half, device=dev) for _ in range(3)]
    position = torch.tensor([start], dtype=torch.int32, device=dev)
    where = dict(position_start=position) if on_device else dict(kv_len=start + rows, query_start=start)
    launch = lambda o, **kw: ct.fmha_seq_f16(q, k, v, ct.partition(o, [64, 1, d]), d ** -0.5, group, causal=True, **where, **kw)
    launch(out[0])
    launch(out[1])
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_keys")
    graph = ct.CapturedGraph().capture(lambda stream: launch(out[2], stream=stream))
    try:
        for _ in range(2):
            graph.launch()
            graph.synchronize()
    finally:
        graph.close()
    ref = _reference(q.permute(1, 0, 2)[None], k[None, :, :start + rows], v[None, :, :start + rows], d ** -0.5, start, group, True)
    for o in out:
        assert _close(o.permute(1, 0, 2), ref, torch.half)
    assert torch.equal(out[0], out[1])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("heads,rows,keys,causal", [(80, 132, 132, True), (40, 256, 256, False), (48, 200, 131, True), (40, 257, 257, True), (20, 700, 513, False)])
def test_gpu_64_rows_around_one_step(ct, dev, dtype, heads, rows, keys, causal):
    q, k, v, out = _call(ct, dtype, 1, heads, 1, rows, keys, 128, causal, bm=256, dev=dev)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_few_64x128x128_keys" if keys <= 256 else "16_64x128x128_keys")
    assert _close(out, _reference(q, k, v, 128 ** -0.5, 0, 1, causal), dtype)


@pytest.mark.gpu
def test_gpu_two_streams_share_keys_at_once(ct, dev):
    """a workspace to each stream: launches that overlap do not meet in one"""
    g = torch.Generator().manual_seed(5)
    normal = lambda *s: torch.randn(*s, generator=g).half().to(dev)
    q, k, v = normal(17, 8, 128), normal(8, 4000, 128), normal(8, 4000, 128)
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [[torch.empty(17, 8, 128, dtype=torch.half, device=dev) for _ in range(6)] for _ in streams]
    torch.cuda.synchronize()
    for i in range(6):
        for s, o in zip(streams, outs):
            ct.fmha_seq_f16(q, k, v, ct.partition(o[i], [64, 1, 128]), 128 ** -0.5, 1, kv_len=4000, query_start=3983, stream=s.cuda_stream)
    torch.cuda.synchronize()
    for o in outs:
        for t in o:
            assert torch.equal(t, outs[0][0])
