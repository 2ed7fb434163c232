"""What cutile_last_resolved_kernel reports of a launch on tiles of 320 to 448 columns (gemm_wide.h): the tile that runs, under the name of the family."""
import ctypes as C

import pytest
import torch

from test_gemm_wide_tiles import SIZES, symbol


@pytest.mark.parametrize("m,n,tile", SIZES)
def test_the_record_has_the_tile_that_runs(fake_hip, m, n, tile):
    ct = fake_hip
    buf = torch.empty(20 << 20, dtype=torch.half)
    view = lambda rows, cols: buf[:rows * cols].view(rows, cols)
    ct.gemm(ct.partition(view(m, n), [256, 256]), view(m, 576), view(576, n), 576, accumulate=False)
    function, info = C.c_char_p(), ct.KernelInfo()
    ct.check(ct.lib().cutile_last_resolved_kernel(C.byref(function), C.byref(info)))
    assert (info.variant, info.symbol) == (b"f16_192x256x64_q2x4", symbol("f16", *tile).encode())
    assert tuple(info.tile[:3]) == (*tile, 64) and info.lds_bytes == 2 * sum(tile) * 64 * 2


@pytest.mark.parametrize("tile", sorted({t for _, _, t in SIZES}))
def test_a_partition_of_such_a_tile_has_no_kernel_of_its_own(fake_hip, tile):
    """its launches go by their size like those of any other odd partition"""
    ct = fake_hip
    x, y = torch.empty(2 * tile[0], 256).half(), torch.empty(256, 2 * tile[1]).half()
    z = torch.empty(2 * tile[0], 2 * tile[1]).half()
    ct.gemm(ct.partition(z, list(tile)), x, y, 64, accumulate=False)      # too short a K for the rule on sizes
    assert ct.last_resolved()["variant"] == "f16_generic"
    with pytest.raises(ct.CutileError):
        ct.gemm(ct.partition(z, list(tile)), x, y, 256, accumulate=False, variant="f16_192x256x64_q2x4+w%dx%d" % tile)
