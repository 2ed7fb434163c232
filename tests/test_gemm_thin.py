"""The GEMM kernels for few rows of x (gemm_small.hip): strips of columns, K split over wavefronts and workgroups."""
import numpy as np
import pytest
import torch

import oracle
from util import normal_bf16_bits, normal_f16_bits, rel_l2, to_dev_bf16

SIZES = [
    # rows, n, k: edges of the 16-row blocks, of the 64-column strip and of the 64-row K step; odd rows start on 2-byte boundaries
    (1, 64, 64), (1, 64, 8), (16, 65, 63), (17, 127, 65), (32, 129, 1), (33, 200, 130), (48, 64, 4096), (64, 1000, 257), (5, 4096, 2048),
    (1, 1024, 8200), (64, 192, 6144),
]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("dtype,accumulate", [("bf16", True), ("f16", False), ("bf16f32", True)])
def test_gpu_thin_gemm(ct, dev, m, n, k, dtype, accumulate):
    f16 = dtype == "f16"
    bits = normal_f16_bits if f16 else normal_bf16_bits
    to_dev = (lambda b: torch.from_numpy(b.view(np.float16)).to(dev)) if f16 else (lambda b: to_dev_bf16(b, dev))
    widen = oracle.f16_bits_to_f32 if f16 else oracle.bf16_bits_to_f32
    a, b = bits((m, k), 901), bits((k, n), 902)
    out = {"bf16": torch.bfloat16, "f16": torch.float16, "bf16f32": torch.float32}[dtype]
    x, y = to_dev(a), to_dev(b)
    z0 = torch.from_numpy(oracle.normal_f32((m, n), 903)).to(dev).to(out)
    z = torch.full((m + 1, n), 7.0, dtype=out, device=dev)      # a row behind z that nothing may touch
    for _ in range(2):                                           # the second launch finds the first one's counters at 0
        z[:m] = z0
        forced = None if k > 64 else f"{dtype}_thin{16 if m <= 16 else 32 if m <= 32 else 64}x64"    # one step: not chosen by itself
        ct.gemm(ct.partition(z[:m], [128, 128]), x, y, k, accumulate=accumulate, generics=[dtype, 128, 128, 1], variant=forced)
        assert "_thin" in ct.last_resolved()["variant"] and ct.last_resolved()["source"] == ("caller" if forced else "size")
        torch.cuda.synchronize()
        ref = widen(a).astype(np.float64) @ widen(b).astype(np.float64) + (z0.double().cpu().numpy() if accumulate else 0)
        # one rounding to the output type (2^-9 bf16, 2^-12 f16 relative) over f32 sums of k products
        assert rel_l2(z[:m].double().cpu().numpy(), ref) <= {"bf16": 2.0 ** -9, "f16": 2.0 ** -12, "bf16f32": 2e-6}[dtype]
        assert torch.all(z[m] == 7.0)


@pytest.mark.gpu
def test_gpu_thin_gemm_streams_and_prefix(ct, dev):
    """split launches on two streams at once (each stream has partial sums of its own), and a launch over the first tile row only"""
    k, n = 8192, 1024
    x = torch.from_numpy(normal_f16_bits((40, k), 911).view(np.float16)).to(dev)
    ys = [torch.from_numpy(normal_f16_bits((k, n), 912 + i).view(np.float16)).to(dev) for i in range(2)]
    want = [(x.double() @ y.double()) for y in ys]
    streams = [torch.cuda.Stream() for _ in ys]
    zs = [torch.zeros(40, n, dtype=torch.float16, device=dev) for _ in range(8)]
    torch.cuda.synchronize()
    for i, z in enumerate(zs):
        ct.gemm(ct.partition(z, [128, 128]), x, ys[i % 2], k, accumulate=False, stream=streams[i % 2].cuda_stream)
    torch.cuda.synchronize()
    for i, z in enumerate(zs):
        assert rel_l2(z.double().cpu().numpy(), want[i % 2].cpu().numpy()) <= 2.0 ** -12 and torch.equal(z, zs[i % 2])
    z = torch.full((40, n), 3.0, dtype=torch.float16, device=dev)
    ct.gemm(ct.partition(z, [16, 64], prefix=True), x, ys[0], k, accumulate=False, grid=(1, 2, 1))
    torch.cuda.synchronize()
    assert torch.equal(z[:16, :128], zs[0][:16, :128]) and torch.all(z[16:] == 3.0) and torch.all(z[:, 128:] == 3.0)


@pytest.mark.gpu
def test_gpu_thin_gemm_captured_and_replayed(ct, dev):
    """a captured launch does not split K (its workspace would belong to a stream); every replay equals float64 to f16 rounding"""
    k, n = 4096, 256
    x = torch.from_numpy(normal_f16_bits((3, k), 921).view(np.float16)).to(dev)
    y = torch.from_numpy(normal_f16_bits((k, n), 922).view(np.float16)).to(dev)
    z = torch.zeros(3, n, dtype=torch.float16, device=dev)
    launch = lambda stream=None: ct.gemm(ct.partition(z, [128, 128]), x, y, k, accumulate=False, stream=stream)
    launch()
    torch.cuda.synchronize()
    graph = ct.CapturedGraph().capture(launch)
    want = (x.double() @ y.double()).cpu().numpy()
    try:
        for _ in range(3):
            z.zero_()
            torch.cuda.synchronize()
            graph.launch()
            graph.synchronize()
            assert rel_l2(z.double().cpu().numpy(), want) <= 2.0 ** -12
            launch()
            torch.cuda.synchronize()
    finally:
        graph.close()


def test_more_than_32_rows_take_strips_while_they_fit_the_chip_once(fake_hip):
    """a workgroup of the 64-row strips fills a compute unit: beyond 256 strips the launch would run twice as long"""
    ct = fake_hip
    buf = torch.empty(32 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
    for m, n, k, want in ((33, 16384, 448, "thin64x64"), (64, 16321, 448, "thin64x64"), (33, 16385, 448, "staged"), (60, 19072, 448, "128x128x64_d2x2"),
                          (46, 16960, 1024, "128x128x64_q2x2"), (49, 22001, 1001, "staged"), (32, 19072, 448, "thin32x64"), (1, 32000, 448, "thin16x128"),
                          (128, 8192, 448, "thin64x64"), (128, 8256, 448, "128x128x64_d2x2")):
        ct.gemm(ct.partition(view(m, n), [128, 128]), view(m, k), view(k, n), k, generics=["f16", 128, 128, 1, k])
        assert ct.last_resolved()["variant"].startswith("f16_" + want), (m, n, k, ct.last_resolved()["variant"])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,member", [(1, 12290, 4100, "thin16x128_nt"), (16, 8201, 6150, "thin16x64_nt"), (3, 24601, 2049, "thin16x128_nt")])
def test_gpu_large_weights_past_the_caches(ct, dev, m, n, k, member, dtype):
    """96 MiB of y and more: strips that read it past the caches, odd rows and ragged K included"""
    g = torch.Generator(device="cuda").manual_seed(m + n)
    x = torch.randn(m, k, device=dev, generator=g).to(dtype)
    y = (torch.randn(k, n, device=dev, generator=g) / k ** 0.5).to(dtype)
    z = torch.full((m + 1, n), 7.0, dtype=dtype, device=dev)             # a row behind z that nothing may touch
    want = (x.double() @ y.double()).cpu().numpy()
    for _ in range(2):                                                    # the second launch finds the first one's counters at 0
        ct.gemm(ct.partition(z[:m], [128, 128]), x, y, k, accumulate=False, generics=["f16" if dtype == torch.float16 else "bf16", 128, 128, 1])
        torch.cuda.synchronize()
        assert ct.last_resolved()["symbol"].endswith(member)
        assert rel_l2(z[:m].double().cpu().numpy(), want) <= (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8)
        assert torch.all(z[m] == 7.0)


def test_weights_that_may_be_cached_keep_plain_loads(fake_hip):
    """below 96 MiB of y, and with more than 16 rows, the strips read through the caches"""
    ct = fake_hip
    buf = torch.empty(80 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
    for m, n, k, want in ((1, 4096, 4096, "thin16x64"), (1, 8192, 6143, "thin16x64"), (1, 8192, 6144, "thin16x64_nt"), (1, 14336, 4096, "thin16x128_nt"),
                          (17, 4096, 14336, "thin32x64"), (33, 4096, 14336, "thin64x64")):
        ct.gemm(ct.partition(view(m, n), [128, 128]), view(m, k), view(k, n), k)
        got = ct.last_resolved()
        assert got["symbol"] == "gemm_entry__f16_" + want and got["variant"] == "f16_" + want.replace("_nt", ""), (m, n, k, got)
    ct.gemm(ct.partition(view(20, 8192), [128, 128]), view(20, 6144), view(6144, 8192), 6144, variant="f16_thin16x64")
    assert ct.last_resolved()["symbol"] == "gemm_entry__f16_thin16x64"


def test_more_than_48_rows_of_a_long_k_share_it_on_tiles(fake_hip):
    """128 x 128 tiles with K shared instead of 64-row strips: from the K on that is worth sharing, and only where there is room for partial sums"""
    ct = fake_hip
    from test_gemm_tiles import _new_stream
    buf = torch.empty(40 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)

    def takes(m, n, k, stream=None, dtype=torch.half):
        ct.gemm(ct.partition(view(m, n).view(dtype), [128, 128]), view(m, k).view(dtype), view(k, n).view(dtype), k, stream=stream)
        return ct.last_resolved()["variant"].split("_", 1)[1]

    for m, n, k, strips in ((112, 3584, 10496, False), (49, 1408, 1792, False), (49, 1408, 1728, True), (128, 4096, 1728, True), (58, 12288, 2048, False),
                            (58, 12416, 2048, True), (32, 512, 8192, True), (33, 1792, 2816, True), (48, 1920, 8192, True), (64, 256, 8192, True), (64, 257, 8192, True), (64, 264, 8192, False),
                            (100, 1001, 8192, True)):
        assert takes(m, n, k).startswith("thin") == strips, (m, n, k)
    assert takes(112, 3584, 10496) == takes(112, 3584, 8192, dtype=torch.bfloat16) == "128x128x64_q2x2"
    dev, stream = _new_stream(ct)
    ct.check(ct.lib().cutile_testing_inject_failure(b"hipMallocAsync", 2, 1))
    assert takes(112, 3584, 10496, stream.value) == "thin64x64"
    ct.check(ct.lib().cutile_stream_release(dev, stream))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,kernel", [(49, 272, 1800, "staged64x64"), (64, 2248, 7680, "staged64x64"), (65, 576, 3976, "staged64x64"), (100, 64, 6408, "staged64x64"),
                                          (50, 3592, 4104, "staged64x64"), (127, 1416, 5128, "staged64x64"), (64, 7688, 6280, "128x128x64_q2x2_lone"),
                                          (50, 7048, 4168, "128x128x64_q2x2_lone"), (128, 3584, 4096, "128x128x64_q2x2_lone"), (127, 2952, 5128, "128x128x64_q2x2_lone")])
def test_gpu_long_k_shared_on_tiles_of_few_rows(ct, dev, m, n, k, kernel, dtype):
    g = torch.Generator(device="cuda").manual_seed(m + n)
    x = torch.randn(m, k, device=dev, generator=g).to(dtype)
    y = (torch.randn(k, n, device=dev, generator=g) / k ** 0.5).to(dtype)
    z = torch.full((m + 1, n), 7.0, dtype=dtype, device=dev)             # a row behind z that nothing may touch
    want = (x.double() @ y.double()).cpu().numpy()
    for _ in range(2):
        ct.gemm(ct.partition(z[:m], [128, 128]), x, y, k, accumulate=False, generics=["f16" if dtype == torch.float16 else "bf16", 128, 128, 1])
        torch.cuda.synchronize()
        assert ct.last_resolved()["symbol"].endswith("_" + kernel)
        assert rel_l2(z[:m].double().cpu().numpy(), want) <= (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8)   # one rounding over f32 sums
        assert torch.all(z[m] == 7.0)


def test_products_without_a_workspace_are_chosen_again(fake_hip):
    """49 to 128 rows whose best kernel shares K, be it tiles or the 64 x 64 staged ones: strips, whose wavefronts share K by themselves, where there is no
    room for partial sums, and the best unshared staged tile beyond 128 rows and for unaligned rows"""
    ct = fake_hip
    from test_gemm_tiles import _new_stream, _workgroups
    buf = torch.empty(40 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)

    def launch(m, n, k, stream=None):
        ct.gemm(ct.partition(view(m, n), [128, 128]), view(m, k), view(k, n), k, stream=stream)
        return ct.last_resolved()["variant"].split("_", 1)[1], _workgroups(ct)

    for shape, shared, alone in (((65, 576, 3976), ("staged64x64", 126), ("thin64x64", 18)), ((100, 64, 6408), ("staged64x64", 16), ("thin64x64", 2)),
                                 ((128, 1920, 2560), ("staged64x64", 300), ("thin64x64", 60)), ((49, 1408, 1792), ("staged64x64", 66), ("thin64x64", 22)),
                                 ((112, 3584, 10496), ("128x128x64_q2x2", 168), ("thin64x64", 112)), ((200, 515, 4099), ("staged64x64", 288), ("staged64x64", 36))):
        assert launch(*shape) == shared, (shape, launch(*shape))
        dev, stream = _new_stream(ct)
        ct.check(ct.lib().cutile_testing_inject_failure(b"hipMallocAsync", 2, 1))
        for _ in range(257):                                             # refused, and not asked for again in the next 256 launches
            assert launch(*shape, stream.value) == alone, shape
        assert launch(*shape, stream.value) == shared
        ct.check(ct.lib().cutile_stream_release(dev, stream))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(65, 576, 3976), (128, 1920, 2560), (200, 515, 4099)])
def test_gpu_captured_product_of_staged_tiles_that_would_share_k(ct, dev, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m)
    x, y = torch.randn(m, k, device=dev, generator=g).half(), (torch.randn(k, n, device=dev, generator=g) / k ** 0.5).half()
    z = torch.zeros(m, n, dtype=torch.half, device=dev)
    launch = lambda stream=None: ct.gemm(ct.partition(z, [128, 128]), x, y, k, accumulate=False, stream=stream, generics=["f16", 128, 128, 1])
    launch()
    torch.cuda.synchronize()
    assert ct.last_resolved()["variant"] == "f16_staged64x64"
    want = (x.double() @ y.double()).cpu().numpy()
    graph = ct.CapturedGraph().capture(launch)
    assert ct.last_resolved()["variant"] == ("f16_thin64x64" if m <= 128 else "f16_staged64x64")
    try:
        for _ in range(3):
            for run in (lambda: (graph.launch(), graph.synchronize()), launch):
                z.zero_()
                torch.cuda.synchronize()
                run()
                torch.cuda.synchronize()
                assert rel_l2(z.double().cpu().numpy(), want) <= 2.0 ** -11        # one rounding over f32 sums
    finally:
        graph.close()


def test_products_of_a_long_k_without_a_workspace(fake_hip):
    """beyond 128 rows, K not shared: 64 x 64 staged tiles while a compute unit has one or two of them (us there and on 128 x 128 ring tiles: 309 x 2240 x 5184
    24.4, 30.9; 332 x 2048 x 1920 11.8, 14.3; 1008 x 768 x 3968 19.8, 25.7; 184 x 4928 x 4736 29.6, 35.1; 300 x 640 x 4096 19.5, 25.5), ring tiles of more outputs (1500 x
    1024 x 4096 30.3, 26.2; 1119 x 1792 x 5056 37.3, 32.2)"""
    ct = fake_hip
    from test_gemm_tiles import _new_stream, _workgroups
    buf = torch.empty(30 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
    for m, n, k, staged in ((309, 2240, 5184, 1), (332, 2048, 1920, 1), (460, 1792, 2304, 1), (1008, 768, 3968, 1), (156, 3392, 2048, 1), (748, 320, 1728, 1), (184, 4928, 4736, 1),
                            (300, 640, 4096, 1), (1500, 1024, 4096, 0), (1800, 1024, 2048, 0)):
        dev, stream = _new_stream(ct)
        ct.check(ct.lib().cutile_testing_inject_failure(b"hipMallocAsync", 2, 1))
        for _ in range(257):
            ct.gemm(ct.partition(view(m, n), [128, 128]), view(m, k), view(k, n), k, stream=stream.value)
        tile = 64 if staged else 128
        assert ct.last_resolved()["symbol"] == "gemm_entry__f16_" + ("staged64x64" if staged else "128x128x64_q2x2_lone"), (m, n, k)
        assert _workgroups(ct) == -(-m // tile) * -(-n // tile), (m, n, k)
        ct.check(ct.lib().cutile_stream_release(dev, stream))


def test_few_outputs_of_aligned_rows_share_k_on_staged_tiles(fake_hip):
    ct = fake_hip
    for m, n, k, want in [(1919, 64, 3264, "staged64x64"), (173, 832, 3328, "staged64x64"), (100, 1024, 4096, "staged64x64"), (335, 832, 1920, "staged64x64"),
                          (54, 7680, 6272, "128x128x64_q2x2"), (64, 4096, 4096, "128x128x64_q2x2"), (64, 2240, 7680, "staged64x64"), (805, 1792, 3264, "128x128x64_q2x2"), (1500, 1024, 4096, "128x128x64_q2x2")]:
        ct.gemm(ct.partition(torch.empty(m, n, dtype=torch.half), [128, 128]), torch.empty(m, k, dtype=torch.half), torch.empty(k, n, dtype=torch.half), k, accumulate=False)
        assert ct.last_resolved()["variant"] == "f16_" + want, (m, n, k)


def test_aligned_partitions_without_kernels_of_their_own(fake_hip):
    """96 x 96: staged tiles while there are less than 128 tiles of 128 x 128, ring tiles beyond, whatever K"""
    ct = fake_hip
    buf = torch.empty(30 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
    for m, n, k, staged in [(335, 832, 1920, True), (700, 640, 136, True), (2966, 9808, 2832, False), (1773, 4064, 608, False), (5390, 1072, 1296, False), (681, 10696, 2368, False),
                            (1556, 9448, 640, False), (1556, 9448, 136, False)]:
        ct.gemm(ct.partition(view(m, n), [96, 96]), view(m, k), view(k, n), k, accumulate=False, generics=["f16", 96, 96, 1])
        assert ("staged" in ct.last_resolved()["variant"]) == staged, (m, n, k, ct.last_resolved()["variant"])
