"""Row kernels on rows of unit stride that are not whole 16-byte vectors (the register-resident path of the any-layout
kernels): lengths at the edges of one lane's vector, of a wavefront, of a workgroup and of the longest row held."""
import numpy as np
import pytest
import torch

import oracle
from util import f16_ulp_diff, from_dev_f16_bits, normal_f16_bits, to_dev_f16

LENGTHS = [1, 7, 9, 63, 511, 513, 2047, 2049, 8191, 8193, 16383, 16387]     # 16387: beyond the registers, the element walk
ROWS = [1, 5]


def _odd_view(bits, dev):
    """a matrix whose rows start on odd halves: one spare column in front"""
    wide = np.zeros((bits.shape[0], bits.shape[1] + 2), np.uint16)
    wide[:, 1:-1] = bits
    return to_dev_f16(wide, dev)[:, 1:-1]


@pytest.mark.gpu
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("rows", ROWS)
def test_gpu_norms_of_any_length(ct, dev, rows, n):
    xb, rb, wb = normal_f16_bits((rows, n), 941), normal_f16_bits((rows, n), 942), oracle.f32_to_f16_bits(oracle.uniform_f32(n, 943, 0.5, 1.5))
    x, r, w = _odd_view(xb, dev), to_dev_f16(rb, dev), to_dev_f16(wb, dev)
    out, res = torch.full((rows + 1, n), 7.0, dtype=torch.half, device=dev), torch.full((rows + 1, n), 7.0, dtype=torch.half, device=dev)
    ct.rms_norm_f16(x, w, ct.partition(out[:rows], [1, n]), 1e-6, variant="generic")
    torch.cuda.synchronize()
    assert np.max(f16_ulp_diff(from_dev_f16_bits(out[:rows]), oracle.rms_norm_f16(xb, wb, 1e-6))) <= 1     # one rounding: a tie may go either way
    assert torch.all(out[rows] == 7.0)
    ct.add_rms_norm_f16(r, x, w, ct.partition(out[:rows], [1, n]), ct.partition(res[:rows], [1, n]), 1e-6, variant="generic")
    torch.cuda.synchronize()
    want, want_res = oracle.add_rms_norm_f16(rb, xb, wb, 1e-6)
    assert np.max(f16_ulp_diff(from_dev_f16_bits(out[:rows]), want)) <= 1
    assert np.array_equal(from_dev_f16_bits(res[:rows]), want_res) and torch.all(out[rows] == 7.0) and torch.all(res[rows] == 7.0)


@pytest.mark.gpu
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_gpu_softmax_of_any_length(ct, dev, n, dtype):
    rows = 5
    x = oracle.normal_f32((rows, n), 951)
    bits = oracle.f32_to_f16_bits(x)
    xd = _odd_view(bits, dev) if dtype == "f16" else torch.from_numpy(x).to(dev)
    y = torch.full((rows + 1, n), 7.0, dtype=xd.dtype, device=dev)
    bn = n if n < 100 else n - 1                                   # a second, ragged tile of one column: padding takes part, as zeros
    ct.softmax(xd, ct.partition(y[:rows], [2, bn]), variant=f"{dtype}_generic")
    torch.cuda.synchronize()
    src = oracle.f16_bits_to_f32(bits).astype(np.float64) if dtype == "f16" else x.astype(np.float64)
    want = np.empty((rows, n))
    for c0 in range(0, n, bn):
        seg = np.zeros((rows, bn))
        valid = min(bn, n - c0)
        seg[:, :valid] = src[:, c0:c0 + valid]
        e = np.exp(seg - seg.max(axis=1, keepdims=True))
        want[:, c0:c0 + valid] = (e / e.sum(axis=1, keepdims=True))[:, :valid]
    # f16: half a unit in the last place (2^-11 relative, 2^-25 absolute below the normals); f32: exp2 of a product of magnitude < 16 and sums of n terms
    tol = 2.0 ** -11 * 1.01 * want + 2.0 ** -25 if dtype == "f16" else 3e-6 * want
    assert np.all(np.abs(y[:rows].double().cpu().numpy() - want) <= tol) and torch.all(y[rows] == 7.0)


def _row_calls(ct, rows, n, stride, dtype=torch.half, dev="cpu"):
    """(launch, outputs) of the four row functions on rows of n elements `stride` apart"""
    g = torch.Generator().manual_seed(971)
    view = lambda *shape: torch.randn(*shape[:-1], shape[-1] * stride, generator=g).to(dtype).to(dev)[..., ::stride]
    x, r, w = view(rows, n), view(rows, n), torch.rand(n, generator=g).to(dtype).to(dev)
    out, out2 = [torch.full((rows, n), 7.0, dtype=dtype, device=dev) for _ in range(2)]
    part = lambda t: ct.partition(t, [1, n])
    half = rows // 2
    return x, r, w, half, out, out2, {
        "rms_norm_f16": lambda **kw: ct.rms_norm_f16(x, w, part(out), 1e-6, **kw), "add_rms_norm_f16": lambda **kw: ct.add_rms_norm_f16(r, x, w, part(out), part(out2), 1e-6, **kw),
        "qk_norm_f16": lambda **kw: ct.qk_norm_f16(x, r, w, w, part(out), 1e-6, half, **kw), "softmax": lambda **kw: ct.softmax(x, part(out), **kw)}


def test_walked_rows_have_a_kernel_of_their_own(fake_hip):
    """adjacent elements of up to 32 KiB: the kernel that holds a row in registers; longer ones and strided ones: the element walk
    alone, one workgroup a row; either can be named for every call"""
    ct = fake_hip
    from test_host_abi import _last
    for n, stride, held in ((1001, 1, True), (16383, 1, True), (16385, 1, False), (64, 2, False), (1001, 2, False)):
        for function, launch in _row_calls(ct, 8, n, stride)[-1].items():
            prefix = "f16_" if function == "softmax" else ""
            launch()
            assert ct.last_resolved()["variant"] == prefix + ("generic" if held else "walk"), (function, n, stride)
            assert held or _last(ct)[0].grid[0] == 8
            for kind in ("generic", "walk"):
                launch(variant=prefix + kind)
                assert ct.last_resolved()["variant"] == prefix + kind
    for n, want in ((8191, "f32_generic"), (8193, "f32_walk")):
        _row_calls(ct, 4, n, 1, torch.float32)[-1]["softmax"]()
        assert ct.last_resolved()["variant"] == want


@pytest.mark.gpu
@pytest.mark.parametrize("rows,n,stride", [(2, 1, 2), (6, 64, 2), (5, 257, 3), (4, 4099, 2), (3, 16385, 1), (300, 33, 2)])
def test_gpu_walked_rows(ct, dev, rows, n, stride):
    """the walk by itself against float64, and bit for bit what the any-layout kernel's walk gives"""
    x, r, w, half, out, out2, calls = _row_calls(ct, rows, n, stride, dev=dev)
    xd, rd, wd = x.double(), r.double(), w.double()
    rms = lambda t: t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6) * wd
    want = {"rms_norm_f16": rms(xd), "add_rms_norm_f16": rms(xd + rd), "qk_norm_f16": rms(torch.cat([xd[:half], rd])[:rows]), "softmax": torch.softmax(xd, -1)}
    for function, launch in calls.items():
        out.fill_(7.0), out2.fill_(7.0)
        launch()
        assert ct.last_resolved()["variant"].endswith("walk")
        torch.cuda.synchronize()
        got, got2 = out.clone(), out2.clone()
        # one rounding to f16 over f32 arithmetic: half a unit in the last place, a hundredth of one for the f32 steps
        assert torch.all((got.double() - want[function]).abs() <= 2.0 ** -11 * 1.01 * want[function].abs() + 2.0 ** -25)
        out.fill_(7.0), out2.fill_(7.0)
        launch(variant="f16_generic" if function == "softmax" else "generic")
        torch.cuda.synchronize()
        assert torch.equal(out, got) and torch.equal(out2, got2)
