"""MXFP8 on 128 x 128 tiles that have a compute unit each (four stages, K shared by workgroups): against the oracle's rule, and who takes it."""
import numpy as np
import pytest
import torch

import oracle
from test_host_abi import _new_stream, _workgroups
from util import rel_l2


def _operands(rows, k, seed, dev):
    g = np.random.default_rng(seed)
    q = g.integers(0, 256, (rows, k), dtype=np.uint8)
    q[(q & 0x7f) == 0x7f] = 0x38                                       # no NaN
    s = g.integers(120, 132, (rows, k // 32), dtype=np.uint8)
    return q, s, torch.from_numpy(q).to(dev), torch.from_numpy(s).to(dev)


# K tiles: 2 (the smallest), 4, 5 and 31 (a last scale block of one and three tiles), 64 (K shared by 8); edges of a tile in both directions
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(128, 128, 256), (1, 4, 512), (129, 132, 640), (200, 260, 3968), (250, 508, 8192)])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_gpu_mxfp8_tiles(ct, dev, m, n, k, out):
    xq, xs, x, sx = _operands(m, k, 11, dev)
    yq, ys, y, sy = _operands(n, k, 12, dev)
    xw, yw = (oracle.mx_dequantize_e4m3(q, s).astype(np.float64) for q, s in ((xq, xs), (yq, ys)))
    want = 0.5 * (xw @ yw.T)
    z = torch.full((m + 1, n), 7.0, dtype=out, device=dev)
    name = "mxfp8_%s_128x128x128_e2x2" % ("bf16" if out == torch.bfloat16 else "f32")
    for _ in range(2):                                                  # the second launch finds the first one's counters at 0
        z[:m] = 0
        ct.linear_tile_mxfp8(ct.partition(z[:m], [128, 128]), x, y, sx, sy, 0.5, variant=name)
        torch.cuda.synchronize()
        got = ct.last_resolved()
        assert got["variant"] == name and got["symbol"].endswith("_lone")
        # bf16: one rounding; f32: the scaled instruction keeps about 14 bits below the largest of its products (measured 1.6e-5)
        assert rel_l2(z[:m].double().cpu().numpy(), want) <= (2.0 ** -8 if out == torch.bfloat16 else 1e-4)
        assert torch.all(z[m] == 7.0)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(2050, 2180, 640), (130, 33028, 256)])
def test_gpu_mxfp8_two_stages_beyond_a_tile_to_each_compute_unit(ct, dev, m, n, k):
    """more tiles than compute units: the two-stage kernel of that name, edges in both directions and a last scale block of one K tile"""
    xq, xs, x, sx = _operands(m, k, 13, dev)
    yq, ys, y, sy = _operands(n, k, 14, dev)
    xw, yw = (torch.from_numpy(oracle.mx_dequantize_e4m3(q, s).astype(np.float64)).to(dev) for q, s in ((xq, xs), (yq, ys)))
    want = xw @ yw.T.contiguous()
    z = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=dev)
    ct.linear_tile_mxfp8(ct.partition(z[:m], [128, 128]), x, y, sx, sy, 1.0, variant="mxfp8_bf16_128x128x128_e2x2")
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_e2x2")
    assert float((z[:m].double() - want).norm()) <= 2.0 ** -8 * float(want.norm()) and torch.all(z[m] == 7.0)


@pytest.mark.gpu
def test_gpu_mxfp8_scales_behind_a_row(ct, dev):
    """K = 640: the tile's last scale block reads on into the next row's scales, which are NaN here"""
    k = 640
    x, y = torch.full((2, k), 0x38, dtype=torch.uint8, device=dev), torch.full((128, k), 0x38, dtype=torch.uint8, device=dev)
    sx, sy = torch.full((2, k // 32), 127, dtype=torch.uint8, device=dev), torch.full((128, k // 32), 127, dtype=torch.uint8, device=dev)
    sx[1], sy[1::2] = 255, 255
    z = torch.zeros(2, 128, device=dev)
    ct.linear_tile_mxfp8(ct.partition(z, [128, 128]), x, y, sx, sy, 1.0, variant="mxfp8_f32_128x128x128_e2x2")
    torch.cuda.synchronize()
    assert torch.all(z[0, ::2] == k) and torch.all(z[0, 1::2].isnan()) and torch.all(z[1].isnan())


def test_mxfp8_tiles_by_size(fake_hip):
    """up to as many tiles as compute units the four stages, K shared where that is cheaper; beyond, and without a workspace, the kernels that were there"""
    ct = fake_hip
    u8 = torch.uint8

    def linear(m, n, k, stream=None, variant=None):
        ct.linear_tile_mxfp8(ct.partition(torch.empty(m, n, dtype=torch.bfloat16), [128, 128]), torch.empty(m, k, dtype=u8), torch.empty(n, k, dtype=u8),
                             torch.empty(m, k // 32, dtype=u8), torch.empty(n, k // 32, dtype=u8), stream=stream, variant=variant)
        return ct.last_resolved()

    got = linear(200, 14336, 4096)
    assert got["variant"] == "mxfp8_bf16_128x128x128_e2x2" and got["symbol"].endswith("_lone") and _workgroups(ct) == 224
    got = linear(859, 1600, 5888)
    assert got["symbol"].endswith("_lone") and _workgroups(ct) == 2 * 91
    got = linear(2100, 4096, 4096)
    assert got["variant"] == "mxfp8_bf16_128x128x128_e2x2" and not got["symbol"].endswith("_lone")
    dev, stream = _new_stream(ct)
    for variant in (None, "mxfp8_bf16_128x128x128_e2x2"):
        ct.check(ct.lib().cutile_testing_inject_failure(b"hipMallocAsync", 2, 1))
        got = linear(859, 1600, 5888, stream.value, variant)
        assert _workgroups(ct) == 91 if got["symbol"].endswith("_lone") else "flat" in got["variant"]
    ct.check(ct.lib().cutile_stream_release(dev, stream))
