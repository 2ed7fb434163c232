"""Block-scaled products of few to medium many rows (scaled_flat.hip, and the 128 x 128 direct pipeline of mxfp8_gemm.hip)."""
import numpy as np
import pytest
import torch

import oracle
from util import rel_l2

# rows, n, k: edges of the 16-row blocks, of the 64-column strip, of one 128-byte step (128 fp8 or 256 fp4 values) and of the steps that one
# wavefront keeps in flight; 1 x 64 x 8192 and 70 x 128 x 8192 split K over workgroups
SIZES = [(1, 64, 256), (16, 68, 384), (17, 60, 640), (33, 132, 1024), (64, 4, 2176), (70, 128, 8192), (1, 64, 8192), (129, 260, 1152)]
TILES = ["16x64", "32x64", "64x64", "64x128", "128x128"]


def _dev(a, dev):
    return torch.from_numpy(a).to(dev)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("out", ["f32", "bf16"])
def test_gpu_scaled_flat(ct, dev, m, n, k, out):
    dt = torch.float32 if out == "f32" else torch.bfloat16
    x, y = oracle.normal_f32((m, k), 951), oracle.normal_f32((n, k), 952) * np.exp2(oracle.uniform_f32((n, 1), 953, -3, 3))
    for fmt in ("mxfp8", "nvfp4"):
        mx = fmt == "mxfp8"
        (xq, xs), (yq, ys) = [(oracle.mx_quantize_e4m3 if mx else oracle.nvfp4_quantize)(v) for v in (x, y)]
        ref = (oracle.mx_gemm_f32 if mx else oracle.nvfp4_gemm_f32)(xq, yq, xs, ys, 0.75)
        launch = ct.linear_tile_mxfp8 if mx else ct.linear_tile_nvfp4
        args = [_dev(v, dev) for v in (xq, yq, xs, ys)]
        variants = [f"{'mxfp8_' if mx else ''}{out}_flat{t}" for t in TILES] + ([f"mxfp8_{out}_128x128x128_e2x2"] if mx else [])
        for variant in variants + [None]:
            z = torch.full((m + 1, n), 7.0, dtype=dt, device=dev)       # a row behind z that nothing may touch
            for _ in range(2):                                           # the second launch finds the first one's counters at 0
                z[:m] = float("nan")
                launch(ct.partition(z[:m], [128, 128]), *args, 0.75, variant=variant)
                torch.cuda.synchronize()
                got = z[:m].float().cpu().numpy()
                # mxfp8: the scaled instruction keeps about 14 bits below its largest product; nvfp4: order of f32 additions; bf16: one rounding
                assert rel_l2(got, ref) <= ((1e-4 if mx else 1e-5) if out == "f32" else 4e-3), variant
                assert torch.all(z[m] == 7.0), variant


@pytest.mark.gpu
def test_gpu_scaled_flat_nan_scales_stay_in_their_row(ct, dev):
    """K that ends inside a 256-value step, beside rows whose scales are NaN: no other row sees them"""
    m, n, k = 5, 72, 320 + 256
    xq, xs = oracle.nvfp4_quantize(oracle.normal_f32((m, k), 961))
    yq, ys = oracle.nvfp4_quantize(oracle.normal_f32((n, k), 962))
    xs, ys = xs.copy(), ys.copy()
    ref = oracle.nvfp4_gemm_f32(xq, yq, xs, ys, 1.0)
    xs[3], ys[40] = 0x7F, 0x7F
    z = torch.zeros(m, n, device=dev)
    ct.linear_tile_nvfp4(ct.partition(z, [128, 128]), *[_dev(v, dev) for v in (xq, yq, xs, ys)], 1.0, variant="f32_flat16x64")
    got = z.cpu().numpy()
    assert np.all(np.isnan(got[3])) and np.all(np.isnan(got[:, 40]))
    keep = np.ix_([0, 1, 2, 4], [c for c in range(n) if c != 40])
    assert rel_l2(got[keep], ref[keep]) <= 1e-5


@pytest.mark.gpu
def test_gpu_scaled_rule(ct, dev):
    """the rule's own choices, and launches it leaves alone: one or two steps, scale rows off 4-byte boundaries, a part of z"""
    def chosen(m, n, k, tile=(128, 128), scales=None, **kw):
        z = torch.zeros(m, n, dtype=torch.bfloat16, device=dev)
        u8 = lambda r, c: torch.zeros(r, c, dtype=torch.uint8, device=dev)
        xs = u8(m, k // 16) if scales is None else scales(m, k // 16)
        ct.linear_tile_nvfp4(ct.partition(z, list(tile), **({"prefix": True} if kw else {})), u8(m, k // 2), u8(n, k // 2), xs, u8(n, k // 16), 1.0, **kw)
        return ct.last_resolved()["variant"]
    assert chosen(1, 4096, 4096) == "bf16_flat16x64"
    assert "flat" not in chosen(1, 512, 512)
    assert "flat" not in chosen(16, 4096, 4096, scales=lambda r, c: torch.zeros(r, c + 2, dtype=torch.uint8, device=dev)[:, :c])
    assert "flat" not in chosen(512, 512, 4096, tile=(256, 256), grid=(1, 1, 1))
    torch.cuda.synchronize()


def test_register_staged_mxfp8_tiles_of_128_by_name(fake_hip):
    """a caller's or a tuner's name for the register-staged 128 x 128 kernel holds; left to itself a launch takes the direct one"""
    ct = fake_hip
    u8 = lambda *shape: torch.zeros(*shape, dtype=torch.uint8)
    for out, dt in (("bf16", torch.bfloat16), ("f32", torch.float32)):
        launch = lambda **kw: ct.linear_tile_mxfp8(ct.partition(torch.zeros(128, 128, dtype=dt), [128, 128]), u8(128, 128), u8(128, 128), u8(128, 4),
                                                   u8(128, 4), **kw)
        launch()
        assert ct.last_resolved()["variant"] == f"mxfp8_{out}_128x128x128_e2x2"
        launch(variant=f"mxfp8_{out}_128x128x128_w2x2")
        assert ct.last_resolved()["variant"] == f"mxfp8_{out}_128x128x128_w2x2" and ct.last_resolved()["source"] == "caller"
        ct.set_preferred_variant("linear_tile", f"mxfp8_{out}_128x128x128_w2x2")
        try:
            launch()
            assert ct.last_resolved()["variant"] == f"mxfp8_{out}_128x128x128_w2x2" and ct.last_resolved()["source"] == "pinned"
        finally:
            ct.set_preferred_variant("linear_tile", None)


@pytest.mark.gpu
@pytest.mark.parametrize("out", ["f32", "bf16"])
def test_gpu_register_staged_mxfp8_tiles_of_128(ct, dev, out):
    m, n, k = 130, 260, 640
    (xq, xs), (yq, ys) = [oracle.mx_quantize_e4m3(oracle.normal_f32(s, 971)) for s in ((m, k), (n, k))]
    ref = oracle.mx_gemm_f32(xq, yq, xs, ys, 1.0)
    z = torch.full((m + 1, n), 7.0, dtype=torch.float32 if out == "f32" else torch.bfloat16, device=dev)
    ct.linear_tile_mxfp8(ct.partition(z[:m], [128, 128]), *[_dev(v, dev) for v in (xq, yq, xs, ys)], 1.0, variant=f"mxfp8_{out}_128x128x128_w2x2")
    torch.cuda.synchronize()
    assert rel_l2(z[:m].float().cpu().numpy(), ref) <= (1e-4 if out == "f32" else 4e-3) and torch.all(z[m] == 7.0)


def test_strips_are_shared_by_as_many_workgroups_as_there_are_compute_units(fake_hip):
    """K of strips of up to 64 x 64 outputs, by the extents, on 256 compute units; short ones, and mxfp8 of less than 90 pieces in pairs, by their prices alone"""
    ct = fake_hip
    from test_host_abi import _workgroups
    u8 = lambda rows, cols: torch.empty(rows, cols, dtype=torch.uint8)
    for fp4, m, n, k, shares in [(0, 16, 2048, 2048, 1), (0, 8, 896, 5248, 5), (0, 1, 5120, 5120, 3), (0, 8, 4096, 4096, 4), (0, 60, 4096, 4096, 4), (0, 15, 8128, 4736, 1),
                                 (0, 12, 7424, 5632, 1), (0, 2, 8192, 7552, 2), (0, 16, 512, 8192, 8), (1, 8, 4096, 4096, 1), (1, 1, 1088, 6656, 2), (1, 8, 896, 5248, 2)]:
        args = (u8(m, k // 2), u8(n, k // 2), u8(m, k // 16), u8(n, k // 16)) if fp4 else (u8(m, k), u8(n, k), u8(m, k // 32), u8(n, k // 32))
        (ct.linear_tile_nvfp4 if fp4 else ct.linear_tile_mxfp8)(ct.partition(torch.empty(m, n, dtype=torch.bfloat16), [128, 128]), *args, 1.0)
        rows, cols = map(int, ct.last_resolved()["variant"].split("flat")[1].split("x"))
        assert _workgroups(ct) == -(-m // rows) * -(-n // cols) * shares, (fp4, m, n, k, ct.last_resolved()["variant"], _workgroups(ct))
