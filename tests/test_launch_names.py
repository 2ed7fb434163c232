"""Names that a launch puts together have a fixed room (csrc/host/names.h): what does not fit it is the name of nothing, and refused as before; errors of a
launcher and streams by number pass through the marshalling extension."""
import pytest
import torch


def test_names_beyond_their_room_are_refused(fake_hip):
    ct = fake_hip
    x, w, out = torch.zeros(4, 64, dtype=torch.half), torch.zeros(64, dtype=torch.half), torch.zeros(4, 64, dtype=torch.half)
    launch = lambda **kw: ct.rms_norm_f16(x, w, ct.partition(out, [1, 64]), 1e-6, **kw)
    launch()
    taken = ct.last_resolved()["symbol"].split("__")[1]
    for name in (taken + "x", taken + "x" * 200, "x" * 45, "x" * 46, "x" * 47):
        with pytest.raises(ct.CutileError):
            launch(variant=name)
    launch(variant=taken)
    with pytest.raises(ct.CutileError):
        ct.set_preferred_variant_for("rms_norm_f16", "n<=256", "x" * 200)
    ct.set_preferred_variant_for("rms_norm_f16", "n<=256" + "x" * 200, "walk")   # a shape class that no launch has
    try:
        launch()
        assert ct.last_resolved()["symbol"].split("__")[1] == taken
    finally:
        ct.set_preferred_variant_for("rms_norm_f16", "n<=256" + "x" * 200, None)


def test_lists_beyond_their_room_keep_every_name(fake_hip):
    """a GEMM partition of 256 x 256 has more kernels than a list holds without allocating: each can be named"""
    ct = fake_hip
    x, y, z = (torch.zeros(256, 256, dtype=torch.half) for _ in range(3))
    names = [n.split(":")[1] for n in ct.kernel_list() if n.startswith("gemm:f16_") and "+" not in n and any(t in n for t in ("256x256", "x64_q", "thin", "staged"))]
    assert len(names) > 12
    for n in names:
        ct.gemm(ct.partition(z, [256, 256]), x, y, 256, accumulate=False, variant=n)
        assert ct.last_resolved()["variant"] == n


def test_streams_and_errors_through_the_extension(fake_hip):
    ct = fake_hip
    x, y = torch.zeros(64), torch.zeros(64)
    assert ct.saxpy(ct.partition(y, [64]), 0.5, x) is None
    assert ct.saxpy(ct.partition(y, [64]), 0.5, x, stream=0) is None
    with pytest.raises((TypeError, ValueError)):
        ct.saxpy(ct.partition(y, [64]), 0.5, x, stream="here")
    with pytest.raises(ct.CutileError, match="x"):
        ct.saxpy(ct.partition(y, [64]), 0.5, torch.zeros(64, dtype=torch.half))
