"""GEMM tiles whose K tiles several workgroups share (the ring, and the kernels of four and five whole stages), and the rule that picks them."""
import numpy as np
import pytest
import torch

from test_gemm_medium import _run
from test_host_abi import _new_stream, _workgroups

TILES = ["256x256x64_q2x4", "192x256x64_q2x4", "256x128x64_q4x2", "128x256x64_q2x4", "192x128x64_q2x2", "128x128x64_q2x2"]


# K tiles: 5, 5 of 5, 17 and 65 (ragged); tiles: one, edges in both directions, more than one group of rows
@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("m,n,k", [(1, 8, 264), (128, 128, 320), (300, 520, 1032), (257, 264, 4104), (2310, 136, 2048)])
@pytest.mark.parametrize("dtype,accumulate", [("bf16", True), ("f16", False)])
def test_gpu_tiles_that_share_k(ct, dev, tile, m, n, k, dtype, accumulate):
    _run(ct, dev, m, n, k, dtype, f"{dtype}_{tile}", accumulate)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(2200, 2200, 320), (700, 5128, 136)])
def test_gpu_two_workgroups_to_a_compute_unit(ct, dev, m, n, k):
    """more 128 x 128 tiles than compute units: the ring of that tile"""
    _run(ct, dev, m, n, k, "f16", "f16_128x128x64_q2x2", True)


def test_shared_k_needs_a_workspace(fake_hip):
    """1500 x 1024 x 4096 (96 tiles of 128 x 128) shares K; without a workspace (a captured stream, memory refused) the launch takes the
    best of the kernels that need none, one workgroup to a tile"""
    ct = fake_hip
    h = torch.half
    x, y, z = torch.empty(1500, 4096, dtype=h), torch.empty(4096, 1024, dtype=h), torch.empty(1500, 1024, dtype=h)
    launch = lambda s=None, v=None: ct.gemm(ct.partition(z, [128, 128]), x, y, 4096, stream=s, variant=v)
    launch()
    got = ct.last_resolved()
    assert got["variant"] == "f16_128x128x64_q2x2" and got["symbol"].endswith("_lone") and _workgroups(ct) == 2 * 96
    dev, stream = _new_stream(ct)
    for variant in (None, "f16_256x256x64_q2x4"):
        ct.check(ct.lib().cutile_testing_inject_failure(b"hipMallocAsync", 2, 1))
        launch(stream.value, variant)
        got = ct.last_resolved()
        assert _workgroups(ct) == (96 if variant is None else 6 * 4) and not got["symbol"].endswith("_split")
    ct.check(ct.lib().cutile_stream_release(dev, stream))
    launch(None, "f16_256x256x64_q2x4")
    assert ct.last_resolved()["symbol"].endswith("_split") and ct.last_resolved()["variant"] == "f16_256x256x64_q2x4" and _workgroups(ct) > 24


def test_partial_launches_and_short_operands_do_not_share_k(fake_hip):
    """a grid that covers part of z, and an x with fewer rows than z, keep one workgroup to a tile"""
    ct = fake_hip
    h = torch.half
    x, y, z = torch.empty(512, 4096, dtype=h), torch.empty(4096, 512, dtype=h), torch.empty(512, 512, dtype=h)
    ct.gemm(ct.partition(z, [256, 256], prefix=True), x, y, 4096, grid=(1, 2, 1), variant="f16_256x256x64_q2x4")
    assert _workgroups(ct) == 2
    ct.gemm(ct.partition(z, [256, 256]), x[:511], y, 4096, variant="f16_256x256x64_q2x4")
    assert _workgroups(ct) == 4


@pytest.mark.gpu
def test_gpu_captured_product_that_would_share_k(ct, dev):
    m, n, k = 1500, 1024, 4096
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(m, k, device=dev, generator=g).half()
    y = (torch.randn(k, n, device=dev, generator=g) / k ** 0.5).half()
    z = torch.zeros(m, n, dtype=torch.half, device=dev)
    launch = lambda stream=None: ct.gemm(ct.partition(z, [128, 128]), x, y, k, accumulate=False, stream=stream)
    launch()
    torch.cuda.synchronize()
    ref = (x.double() @ y.double()).cpu().numpy()
    norm = np.linalg.norm(ref)
    graph = ct.CapturedGraph().capture(launch)
    try:
        for _ in range(3):
            z.zero_()
            torch.cuda.synchronize()
            graph.launch()
            graph.synchronize()
            assert np.linalg.norm(z.double().cpu().numpy() - ref) <= 2.0 ** -11 * norm
            launch()
            torch.cuda.synchronize()
            assert np.linalg.norm(z.double().cpu().numpy() - ref) <= 2.0 ** -11 * norm
    finally:
        graph.close()
