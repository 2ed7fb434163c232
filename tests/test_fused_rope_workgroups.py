"""Fused Q/K norm + rotary embedding + KV-cache update: how many workgroups take the heads of a position, and the results where there are several"""
import numpy as np
import pytest
import torch

import oracle
from test_fused_qk_norm_rope_kv import _bits, _case, _close, _dev16


@pytest.mark.parametrize("seq,nq,nkv,grid,block", [(1, 32, 8, 2, 192), (1, 28, 28, 3, 256), (1, 8, 1, 1, 128), (1023, 36, 9, 2, 256), (1024, 36, 9, 1, 256), (5, 198, 1, 7, 256)])
def test_workgroups_of_a_position(fake_hip, seq, nq, nkv, grid, block):
    ct = fake_hip
    from test_host_abi import _last
    h = torch.half
    w, inv = torch.zeros(128, dtype=h), torch.zeros(64)
    q, k, cache = torch.zeros(seq, nq, 128, dtype=h), torch.zeros(seq, nkv, 128, dtype=h), torch.zeros(nkv, seq, 128, dtype=h)
    ct.qk_norm_rope_kv_prefill_raw_f16(q, k, k, w, w, inv, q, cache, cache.clone(), 1e-6, 0, seq)
    rec = _last(ct)[0]
    assert tuple(rec.grid) == (seq, grid, 1) and rec.block[0] == block


@pytest.mark.gpu
@pytest.mark.parametrize("seq,nq,nkv,d", [(1, 28, 28, 128), (3, 36, 9, 128), (2, 130, 3, 64), (5, 9, 4, 1024), (1030, 30, 3, 128)])
def test_gpu_heads_of_several_workgroups(ct, dev, seq, nq, nkv, d):
    """one workgroup to each pass over the heads, passes that end inside a workgroup, and (seq >= 1024) several passes to one workgroup"""
    q, k, v, qw, kw, inv_freq, kc, vc = _case(seq, nq, nkv, d, seq + 3, 941)
    q_out, kcd, vcd = torch.zeros(seq, nq, d, dtype=torch.half, device=dev), _dev16(kc, dev), _dev16(vc, dev)
    ct.qk_norm_rope_kv_prefill_raw_f16(_dev16(q, dev), _dev16(k, dev), _dev16(v, dev), _dev16(qw, dev), _dev16(kw, dev), torch.from_numpy(inv_freq).to(dev), q_out, kcd, vcd,
                                       1e-6, 2, seq)
    torch.cuda.synchronize()
    rq, rk, rv = oracle.qk_norm_rope_kv_f16(q, k, v, qw, kw, inv_freq, kc, vc, 1e-6, 2)
    assert _close(_bits(q_out), rq) and _close(_bits(kcd), rk) and np.array_equal(_bits(vcd), rv)
