"""Grouped products whose last round of tiles shares K, and launches of 256 x 256 tiles that choose their tile on the device"""
import pytest
import torch

from test_group_gemm import _tables


def test_launches_that_choose_their_tile(fake_hip):
    ct = fake_hip
    from test_host_abi import _last
    ptrs, metas = torch.zeros(300, dtype=torch.int64), torch.zeros(300, 8, dtype=torch.int32)
    ring = b"group_gemm_nt_desc_entry__f16_256x256x64_q2x4"
    for groups, num_sm, variant, ahead in [(4, 256, None, True), (256, 129, None, True), (0, 256, None, True), (257, 256, None, False), (4, 128, None, False), (4, 257, None, False),
                                           (4, 256, "f16_256x256x64_q2x4", False)]:
        ct.group_gemm_f16_nt_desc(ptrs, ptrs, ptrs, metas, metas, metas, groups, generics=[256, 256, 64, num_sm], variant=variant)
        rec = _last(ct)[0]
        assert rec.symbol == (ring + b"_ahead" if ahead else ring) and tuple(rec.block) == (512, 1, 1) and rec.grid[0] == num_sm
    with pytest.raises(ct.CutileError, match="variant"):
        ct.group_gemm_f16_nt_desc(ptrs, ptrs, ptrs, metas, metas, metas, 4, generics=[256, 256, 64, 256], variant="f16_256x256x64_q2x4+ahead")


def _groups(shapes, dev):
    g = torch.Generator().manual_seed(len(shapes))
    a = [torch.randn(m, k, generator=g).half().to(dev) for m, n, k in shapes]
    b = [(torch.randn(k, n, generator=g) * max(k, 1) ** -0.5).half().to(dev) for m, n, k in shapes]
    return a, b, lambda: [torch.full((m + 1, n), 7.0, dtype=torch.half, device=dev) for m, n, k in shapes]


def _check(c, a, b):
    for ci, ai, bi in zip(c, a, b):
        assert torch.all(ci[-1] == 7.0)                                       # the row behind C
        ref = ai.double() @ bi.double()
        assert (ci[:-1].double() - ref).norm() <= 2.0 ** -11 * ref.norm()     # one rounding to f16 over f32 sums


@pytest.mark.gpu
@pytest.mark.parametrize("tile,num_sm,shapes", [
    # 128 x 128 tiles in rounds, and a last round of few: shared by two, by eight; uneven inner sizes, one of them empty
    (128, 256, [(40, 128 * 257, 1040)]), (128, 131, [(17, 128 * 100, 1024), (0, 256, 64), (130, 128 * 23, 1600), (5, 16, 0)]), (128, 129, [(8, 128 * 129 + 16, 4096)]),
    (128, 256, [(9, 128 * 150, 512), (9, 128 * 170, 2048)]),
    # 256 x 256: few tiles, on 128 x 128 ones; one round, rows and columns off the tile; several rounds of both kinds, and more of them than are looked up in advance
    (256, 256, [(300, 272, 512), (0, 64, 64), (700, 768, 1040), (16, 528, 0)]), (256, 256, [(256 * 9 + 8, 256 * 13 + 16, 832), (511, 256 * 15, 640)]),
    (256, 131, [(700, 1040, 2064)] * 12), (256, 129, [(4096 - 8, 4352, 512)] * 2 + [(16, 4352, 512)]), (256, 256, [(1 + 97 * i % 600, 256 + 16 * (i % 9), 64 + 16 * i) for i in range(64)]),
])
def test_gpu_rounds_of_tiles(ct, dev, tile, num_sm, shapes):
    """against 64 bits, twice on the same workspace, against the kernel that a name asks for, and from inside a captured graph, where no K is shared"""
    a, b, outputs = _groups(shapes, dev)
    c, r, g = outputs(), outputs(), outputs()
    (ap, am), (bp, bm), (cp, cm), (rp, rm), (gp, gm) = [_tables(t, dev) for t in (a, b, *[[t[:-1] for t in x] for x in (c, r, g)])]
    for _ in range(2):
        ct.group_gemm_f16_nt_desc(ap, bp, cp, am, bm, cm, len(shapes), generics=[tile, tile, 64, num_sm])
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_ahead")
    _check(c, a, b)
    ct.group_gemm_f16_nt_desc(ap, bp, rp, am, bm, rm, len(shapes), generics=[tile, tile, 64, num_sm], variant="f16_256x256x64_q2x4" if tile == 256 else "f16_128x128x64_d2x2")
    graph = ct.CapturedGraph().capture(lambda stream: ct.group_gemm_f16_nt_desc(ap, bp, gp, am, bm, gm, len(shapes), generics=[tile, tile, 64, num_sm], stream=stream))
    try:
        for _ in range(2):
            graph.launch()
            graph.synchronize()
    finally:
        graph.close()
    for x, y in zip(g, r):
        assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [128, 256])
def test_gpu_no_groups(ct, dev, tile):
    ptrs, metas = torch.zeros(1, dtype=torch.int64, device=dev), torch.zeros(1, 8, dtype=torch.int32, device=dev)
    ct.group_gemm_f16_nt_desc(ptrs, ptrs, ptrs, metas, metas, metas, 0, generics=[tile, tile, 64, 256])
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_ahead")
