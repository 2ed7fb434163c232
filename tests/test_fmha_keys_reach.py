"""Causal attention whose wavefronts have keys of their own: a value of V that is not finite reaches the rows that see its key and, in their block of 32 rows, those that share
its strip of 32 keys (a zero times it is not zero); no row of another block."""
import pytest
import torch

# heads, group, D, rows, keys in front of them, the poisoned key, the first row that it may reach (the block of 32 rows with one that sees its strip), on 64 rows
CASES = [(8, 4, 128, 2000, 0, 1970, 1952, True), (8, 1, 128, 1985, 100, 2082, 1952, True), (32, 4, 128, 200, 4000, 4116, 96, True), (32, 4, 128, 200, 4000, 4030, 0, True),
         (4, 1, 128, 1000, 0, 940, 928, False), (16, 4, 64, 1000, 0, 940, 928, True), (8, 4, 64, 200, 1000, 1130, 96, False)]


@pytest.mark.parametrize("heads,group,d,rows,start,key,reach,on_64", CASES)
def test_cases(fake_hip, heads, group, d, rows, start, key, reach, on_64):
    """`reach` follows from the strips, and the cases run where they are meant to"""
    ct = fake_hip
    from test_host_abi import _last
    first_seen_strip = key // 32 * 32 - start        # the first row that sees a key of the strip
    assert reach == max(first_seen_strip, 0) // 32 * 32 and key - start < rows
    q, kv, out = torch.empty(1, heads, rows, d).half(), torch.empty(1, heads // group, start + rows, d).half(), torch.empty(heads, rows, d).half()
    ct.fmha(ct.partition(out, [1, 128, d]), q, kv, kv, 0.1, start, group, causal=True)
    name = _last(ct)[0].symbol.decode()
    assert name.endswith("_keys") and (f"_64x128x{d}_" in name) == on_64 and "few" not in name


@pytest.mark.gpu
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
@pytest.mark.parametrize("heads,group,d,rows,start,key,reach,on_64", CASES)
def test_gpu_reach(ct, dev, heads, group, d, rows, start, key, reach, on_64, value):
    g = torch.Generator().manual_seed(rows + key)
    normal = lambda *s: torch.randn(*s, generator=g).half().to(dev)
    q, k, v = normal(1, heads, rows, d), normal(1, heads // group, start + rows, d), normal(1, heads // group, start + rows, d)
    clean, out = torch.empty(heads, rows, d, dtype=torch.half, device=dev), torch.empty(heads, rows, d, dtype=torch.half, device=dev)
    ct.fmha(ct.partition(clean, [1, 128, d]), q, k, v, d ** -0.5, start, group, causal=True)
    v[:, :, key] = value
    ct.fmha(ct.partition(out, [1, 128, d]), q, k, v, d ** -0.5, start, group, causal=True)
    torch.cuda.synchronize()
    assert torch.isfinite(clean).all() and torch.equal(out[:, :reach], clean[:, :reach])
    assert not torch.isfinite(out[:, key - start:]).any()
