"""f32 GEMM on the matrix cores: strips of 16, 32 and 64 rows by 64 columns against float64, and the calls that stay on the any-layout kernel."""
import numpy as np
import pytest
import torch

from util import rel_l2


# one strip exactly, its edges, a ragged last step of K, fewer K positions than a step, K dealt to several workgroups, odd row pitches
@pytest.mark.gpu
@pytest.mark.parametrize("variant", ["f32_strip16x64", "f32_strip32x64", "f32_strip64x64", None])
@pytest.mark.parametrize("m,n,k", [(16, 64, 256), (1, 64, 1), (64, 128, 16), (65, 65, 17), (3, 127, 4099), (33, 641, 511), (200, 333, 1300)])
@pytest.mark.parametrize("accumulate", [True, False])
def test_gpu_f32_strips(ct, dev, variant, m, n, k, accumulate):
    g = np.random.default_rng(7 * m + n + k)
    a, b, c = (g.standard_normal(s).astype(np.float32) for s in ((m, k), (k, n), (m, n)))
    want = a.astype(np.float64) @ b.astype(np.float64) + (c if accumulate else 0)
    z = torch.full((m + 1, n), 7.0, device=dev)                         # a row behind z that nothing may touch
    x, y = torch.from_numpy(a).to(dev), torch.from_numpy(b).to(dev)
    for _ in range(2):                                                  # the second launch finds the first one's counters at 0
        z[:m] = torch.from_numpy(c).to(dev)
        ct.gemm(ct.partition(z[:m], [64, 64]), x, y, k, accumulate=accumulate, generics=["f32", 64, 64, 1], variant=variant)
        torch.cuda.synchronize()
        assert ct.last_resolved()["variant"].startswith("f32_strip")
        # a sum of k products in f32 is off by sqrt(k) roundings of 2^-24 of its own size at most, whatever their order
        assert rel_l2(z[:m].double().cpu().numpy(), want) <= 2.0 ** -24 * (2 + np.sqrt(k))
        assert torch.all(z[m] == 7.0)


@pytest.mark.gpu
def test_gpu_f32_partial_cover(ct, dev):
    """a grid over part of z stores that part alone"""
    x, y, z = torch.ones(100, 40, device=dev), torch.ones(40, 200, device=dev), torch.zeros(100, 200, device=dev)
    ct.gemm(ct.partition(z, [16, 48], prefix=True), x, y, 40, grid=(3, 2, 1), accumulate=False, generics=["f32", 16, 48, 8])
    torch.cuda.synchronize()
    want = torch.zeros(100, 200, device=dev)
    want[:48, :96] = 40
    assert torch.equal(z, want)


def test_f32_calls_that_the_strips_do_not_take(fake_hip):
    """strided columns, operands shorter than the output, fewer than 64 columns of y: the any-layout kernel, as before"""
    ct = fake_hip
    e = torch.empty
    for z, x, y in ((e(64, 128), e(64, 64), e(128, 64).T), (e(64, 128), e(63, 64), e(64, 128)), (e(64, 128), e(64, 64), e(64, 127)),
                    (e(64, 63), e(64, 64), e(64, 63)), (e(64, 256)[:, ::2], e(64, 64), e(64, 128))):
        ct.gemm(ct.partition(z, [16, 16]), x, y, 64, generics=["f32", 16, 16, 8])
        assert ct.last_resolved()["variant"] == "f32_generic"
    ct.gemm(ct.partition(e(64, 128), [16, 16]), e(64, 64), e(64, 128), 64, generics=["f32", 16, 16, 8])
    assert ct.last_resolved()["variant"].startswith("f32_strip") and ct.last_resolved()["source"] == "size"


def _products_that_share_k(ct):
    f = lambda m, n, k, s=None, v=None: ct.gemm(ct.partition(torch.empty(m, n), [64, 64]), torch.empty(m, k), torch.empty(k, n), k, stream=s, variant=v,
                                                generics=["f32", 64, 64, 64])
    # (m, n, k): strip and workgroups with room for partial sums, and without
    return f, [((64, 4096, 4096), "64x64", "16x64", 256), ((64, 2048, 8192), "32x64", "16x64", 128), ((128, 1024, 8192), "32x64", "16x64", 128),
               ((200, 512, 8192), "32x64", "16x64", 104)]


def test_f32_strips_without_a_workspace_are_chosen_again(fake_hip):
    """a strip that is the best one only with its K shared gives way to the best of those that share nothing"""
    ct = fake_hip
    from test_host_abi import _new_stream, _workgroups
    launch, cases = _products_that_share_k(ct)
    for shape, shared, alone, blocks in cases:
        launch(*shape)
        assert ct.last_resolved()["variant"] == "f32_strip" + shared and _workgroups(ct) > -(-shape[0] // int(shared[:2])) * shape[1] // 64
        dev, stream = _new_stream(ct)
        ct.check(ct.lib().cutile_testing_inject_failure(b"hipMallocAsync", 2, 1))
        for _ in range(257):                                            # refused, and not asked for again in the next 256 launches
            launch(*shape, stream.value)
            assert ct.last_resolved()["variant"] == "f32_strip" + alone and _workgroups(ct) == blocks
        launch(*shape, stream.value)
        assert ct.last_resolved()["variant"] == "f32_strip" + shared
        ct.check(ct.lib().cutile_stream_release(dev, stream))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(64, 1024, 4096), (130, 520, 4099)])
def test_gpu_captured_f32_product_that_would_share_k(ct, dev, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m)
    x, y, z = torch.randn(m, k, device=dev, generator=g), torch.randn(k, n, device=dev, generator=g), torch.zeros(m, n, device=dev)
    launch = lambda stream=None: ct.gemm(ct.partition(z, [64, 64]), x, y, k, accumulate=False, stream=stream, generics=["f32", 64, 64, 1])
    launch()
    torch.cuda.synchronize()
    want = (x.double() @ y.double()).cpu().numpy()
    graph = ct.CapturedGraph().capture(launch)
    assert ct.last_resolved()["variant"] == "f32_strip16x64"
    try:
        for _ in range(3):
            for run in (lambda: (graph.launch(), graph.synchronize()), launch):
                z.zero_()
                torch.cuda.synchronize()
                run()
                torch.cuda.synchronize()
                assert rel_l2(z.double().cpu().numpy(), want) <= 2.0 ** -24 * (2 + np.sqrt(k))      # (as above)
    finally:
        graph.close()


def test_f32_products_of_many_rows_launch(fake_hip):
    """more strips of rows than a grid's y axis counts (65535), by the rule and by name, on both sides of that line"""
    ct = fake_hip
    from test_host_abi import _last
    x, y, z = torch.empty(4194241, 64), torch.empty(64, 64), torch.empty(4194241, 64)
    for rows, variant, strips in ((4194240, None, 65535), (4194241, None, 65536), (1048560, "f32_strip16x64", 65535), (1048561, "f32_strip16x64", 65536)):
        ct.gemm(ct.partition(z[:rows], [64, 64]), x[:rows], y, 64, generics=["f32", 64, 64, 64], variant=variant)
        grid = _last(ct)[0].grid
        assert ct.last_resolved()["variant"] == (variant or "f32_strip64x64") and grid[0] * grid[1] * grid[2] == strips


@pytest.mark.gpu
def test_gpu_f32_product_of_many_rows(ct, dev):
    m = 4194305                                                         # 65537 strips of 64 rows
    x = torch.arange(m, device=dev, dtype=torch.float32)[:, None] % 4093 + torch.arange(4, device=dev)
    y, z = torch.ones(4, 64, device=dev), torch.zeros(m, 64, device=dev)
    y[:, 1::2] = 2
    ct.gemm(ct.partition(z, [64, 64]), x, y, 4, accumulate=False, generics=["f32", 64, 64, 4])
    torch.cuda.synchronize()
    assert ct.last_resolved()["variant"].startswith("f32_strip")
    want = 4 * x[:, 0] + 6                                              # whole numbers below 2^24: exact
    assert torch.equal(z[:, 0], want) and torch.equal(z[:, ::2], want[:, None].expand(-1, 32)) and torch.equal(z[:, 1::2], 2 * want[:, None].expand(-1, 32))
