"""The 256-row attention kernel's last key tile, one copy of its code for an even and an odd number of tiles: 1 to 6 tiles, whole and ragged, for both halves of a
workgroup, the two kinds of mask and rows in front of which keys lie; and that the kernel keeps all it has in registers."""
import os
import re
import subprocess

import pytest
import torch

from test_fmha_keys import _call, _close, _reference


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.half, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("rows,keys", [(20, 20), (256, 64), (200, 65), (129, 129), (256, 192), (170, 170), (300, 257), (300, 320), (321, 321), (520, 384), (129, 340), (700, 700)])
def test_gpu_last_tile(ct, dev, dtype, rows, keys, causal):
    pos = keys - rows if keys > rows else 0
    q, k, v, out = _call(ct, dtype, 2, 4, 2, rows, keys, 128, causal, pos=pos, bm=256, dev=dev, variant={torch.half: "f16", torch.bfloat16: "bf16"}[dtype] + "_256x64x128_pp")
    torch.cuda.synchronize()
    assert ct.last_resolved()["symbol"].endswith("_256x64x128_pp")
    assert _close(out, _reference(q, k, v, 128 ** -0.5, pos, 2, causal), dtype)


def test_nothing_is_spilled():
    """a copy of the last tile to each parity had cost 180 bytes a lane of scratch, and 5 to 8 us of every launch with an odd number of tiles"""
    lib = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cutile-rs_amd", "lib", "fmha.hsaco")
    notes = subprocess.run(["/opt/rocm/llvm/bin/llvm-readelf", "--notes", lib], stdout=subprocess.PIPE, text=True, check=True).stdout
    kernels = [k for k in notes.split("- .agpr_count")[1:] if re.search(r"\n    \.name: +\S+_pp\n", k)]
    assert len(kernels) >= 2 and all(int(re.search(r"\.private_segment_fixed_size: (\d+)", k)[1]) == 0 for k in kernels)
