"""The attention kernels whose wavefronts read common stages (64 and 128 rows at D = 64, 64 rows of up to 256 keys at D = 128) take all keys of a query tile: no launch of them deals keys out."""
import pytest
import torch


@pytest.mark.parametrize("d", [64, 128])
def test_one_workgroup_to_a_query_tile(fake_hip, d):
    ct = fake_hip
    from test_host_abi import _last
    seen = set()
    for heads, rows in ((5, 1664), (8, 1025), (9, 900), (16, 513), (40, 200), (43, 161), (65, 97), (100, 129), (129, 33), (200, 40), (256, 64), (300, 300)):
        for start in (0, 56, 100, 900, 4000):
            q, kv, out = torch.empty(1, heads, rows, d).half(), torch.empty(1, heads, rows + start, d).half(), torch.empty(heads, rows, d).half()
            for causal in (True, False):
                ct.fmha(ct.partition(out, [1, 128, d]), q, kv, kv, 0.1, start, 1, causal=causal)
                rec = _last(ct)[0]
                name = rec.symbol.decode().split("__f16_")[1]
                if name in ("few_64x128x128_keys", "64x128x64_keys", "128x64x64_halves"):
                    seen.add(name)
                    assert rec.grid[2] == 1, (heads, rows, start, causal, name)
    assert seen == ({"64x128x64_keys", "128x64x64_halves"} if d == 64 else {"few_64x128x128_keys"})
