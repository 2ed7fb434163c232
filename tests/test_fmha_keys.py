"""Attention whose workgroups share the keys of 32 or 64 query rows (short launches), or of 128 (D = 64): which calls take it, and its results"""
import numpy as np
import pytest
import torch


def _call(ct, dtype, batch, heads, group, rows, keys, d, causal, pos=0, bm=128, dev="cpu", **kw):
    g = torch.Generator().manual_seed(rows * 7 + keys + d)
    normal = lambda *s: torch.randn(*s, generator=g).to(dtype).to(dev)
    q, k, v = normal(batch, heads, rows, d), normal(batch, heads // group, keys, d), normal(batch, heads // group, keys, d)
    out = torch.full((batch * heads, rows, d), 7.0, dtype=dtype, device=dev)
    ct.fmha(ct.partition(out, [1, bm, d]), q, k, v, d ** -0.5, pos, group, causal=causal, **kw)
    return q, k, v, out


# ---- launcher on the recording runtime (CPU) ----------------------------------------------------
@pytest.mark.parametrize("heads,rows,d,causal,takes", [
    (4, 2048, 128, True, 32), (4, 2049, 128, True, 64), (8, 2048, 128, False, 64), (8, 2049, 128, True, 0), (1, 128, 128, True, 0), (1, 129, 128, False, 32),
    (8, 1024, 64, True, 32), (8, 1025, 64, True, 64), (32, 1024, 64, False, 64), (128, 256, 64, True, 0), (32, 2048, 64, True, 64), (32, 2048, 64, False, 128),
    (32, 2049, 64, True, 128), (4, 512, 256, True, 0),
])
def test_short_attention_shares_keys(fake_hip, heads, rows, d, causal, takes):
    ct = fake_hip
    from test_host_abi import _last
    bm = 256 if d == 128 and rows > 128 else 128
    _call(ct, torch.bfloat16, 1, heads, 1, rows, rows, d, causal, bm=bm)
    rec = _last(ct)[0]
    assert rec.symbol.endswith((b"_keys", b"_halves")) == (takes > 0)
    assert tuple(rec.grid) == (heads, -(-rows // (takes or bm)), 1)
    if takes:
        assert rec.symbol.decode() == f"fmha_entry__bf16_{takes}x{8192 // takes}x{d}_{'halves' if takes == 128 else 'keys'}" and tuple(rec.block) == (512, 1, 1)
        for kw in ({"variant": f"bf16_128x64x{d}"}, {"generics": [128, 64, d]}):      # a kernel or a key tile that the caller names
            _call(ct, torch.bfloat16, 1, heads, 1, rows, rows, d, causal, **kw)
            assert _last(ct)[0].symbol.decode() == f"fmha_entry__bf16_128x64x{d}"
        ct.set_preferred_variant("fmha", f"bf16_128x64x{d}")
        try:
            _call(ct, torch.bfloat16, 1, heads, 1, rows, rows, d, causal)
            assert _last(ct)[0].symbol.decode() == f"fmha_entry__bf16_128x64x{d}"
        finally:
            ct.set_preferred_variant("fmha", None)


def test_a_member_is_described_as_the_kernel_that_it_is(fake_hip):
    """cutile_last_resolved_kernel: symbol, block, LDS and tile of the kernel that was launched, the variant's name that of its family"""
    import ctypes as C
    ct = fake_hip
    from test_host_abi import _last
    for rows, d, tile, lds in ((300, 128, (32, 256, 128, 0), 512 * 128 * 2 + 2048), (1500, 64, (64, 128, 64, 0), 512 * 64 * 2 + 2048)):
        _call(ct, torch.half, 1, 4 if d == 128 else 16, 1, rows, rows, d, True)
        function, info = C.c_char_p(), ct.KernelInfo()
        ct.check(ct.lib().cutile_last_resolved_kernel(C.byref(function), C.byref(info)))
        assert info.variant == f"f16_128x64x{d}".encode() and info.symbol == _last(ct)[0].symbol and tuple(info.block) == (512, 1, 1)
        assert tuple(info.tile) == tile and info.lds_bytes == lds


# ---- HIP kernels (GPU) --------------------------------------------------------------------------
def _reference(q, k, v, scale, pos, group, causal):
    q, k, v = (t.double().cpu() for t in (q, k, v))
    k, v = k.repeat_interleave(group, dim=1), v.repeat_interleave(group, dim=1)
    s = q @ k.transpose(-1, -2).contiguous() * scale
    if causal:
        s = s.masked_fill(torch.arange(k.shape[2])[None, :] > torch.arange(q.shape[2])[:, None] + pos, float("-inf"))
    return (torch.softmax(s, -1) @ v).flatten(0, 1).numpy()


def _close(got, ref, dtype):
    u = 2.0 ** -11 if dtype == torch.half else 2.0 ** -8       # one rounding of the probabilities and one of the result
    return np.linalg.norm(got.double().cpu().numpy() - ref) <= 2 * u * np.linalg.norm(ref)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("batch,heads,group,rows,keys,causal,pos", [
    (1, 1, 1, 129, 129, True, 0), (1, 1, 1, 1, 257, True, 256), (2, 8, 4, 33, 700, True, 650), (1, 4, 2, 300, 131, True, 0),     # 32 rows
    (1, 2, 1, 65, 513, False, 0), (1, 1, 1, 1000, 1000, True, 0), (2, 2, 1, 256, 256, False, 0),
    (1, 16, 1, 801, 801, True, 0), (2, 16, 4, 449, 640, False, 0), (1, 32, 1, 511, 140, True, 30),                                # 64 rows
])
def test_gpu_attention_sharing_keys(ct, dev, dtype, d, batch, heads, group, rows, keys, causal, pos):
    q, k, v, out = _call(ct, dtype, batch, heads, group, rows, keys, d, causal, pos=pos, dev=dev)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith(f"_64x128x{d}_keys" if heads >= 16 else f"_32x256x{d}_keys")
    assert _close(out, _reference(q, k, v, d ** -0.5, pos, group, causal), dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("rows,start,on_device", [(130, 0, False), (17, 400, False), (200, 311, True), (400, 100, True)])
def test_gpu_sequence_attention_sharing_keys(ct, dev, d, rows, start, on_device):
    g = torch.Generator().manual_seed(rows)
    normal = lambda *s: torch.randn(*s, generator=g).half().to(dev)
    q, k, v = normal(rows, 8, d), normal(2, 600, d), normal(2, 600, d)
    out = torch.full((rows, 8, d), 7.0, dtype=torch.half, device=dev)
    where = dict(position_start=torch.tensor([start], dtype=torch.int32, device=dev)) if on_device else dict(kv_len=start + rows, query_start=start)
    ct.fmha_seq_f16(q, k, v, ct.partition(out, [64, 1, d]), d ** -0.5, 4, **where)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"] == f"{'fmha_seq' if on_device else 'fmha'}_entry__f16_32x256x{d}_keys"
    seen = 600 if on_device else start + rows
    ref = _reference(q.permute(1, 0, 2)[None], k[None, :, :seen], v[None, :, :seen], d ** -0.5, start, 4, True)
    assert _close(out.permute(1, 0, 2), ref, torch.half)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("rows,heads,position,causal,member", [(129, 8, 0, True, 32), (200, 8, 255, True, 32), (200, 8, 256, False, 32), (400, 8, 131, False, 32), (300, 32, 599, True, 64),
                                                               (300, 32, 700, False, 64)])
def test_gpu_sequence_attention_sharing_keys_up_to_the_position(ct, dev, d, rows, heads, position, causal, member):
    """keys 0 .. position, which only the device knows: the kernel cuts them off itself; what lies behind them must not be seen"""
    g = torch.Generator().manual_seed(rows + position)
    normal = lambda *s: torch.randn(*s, generator=g).half().to(dev)
    q, k, v = normal(rows, heads, d), normal(2, 640, d), normal(2, 640, d)
    seen = min(position + 1, 640)
    k[:, seen:], v[:, seen:] = 100.0, 1000.0
    out = torch.full((rows, heads, d), 7.0, dtype=torch.half, device=dev)
    where = torch.tensor([position], dtype=torch.int32, device=dev)
    ct.fmha_seq_f16(q, k, v, ct.partition(out, [64, 1, d]), d ** -0.5, heads // 2, position_start=where, kv_len_from_position=True, causal=causal)
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"] == f"fmha_seq_entry__f16_{'32x256' if member == 32 else '64x128'}x{d}_keys"
    ref = _reference(q.permute(1, 0, 2)[None], k[None, :, :seen], v[None, :, :seen], d ** -0.5, position, heads // 2, causal)
    assert _close(out.permute(1, 0, 2), ref, torch.half)
