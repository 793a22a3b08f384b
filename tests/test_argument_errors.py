"""Argument errors of the ops are ValueErrors raised before any GPU work, so
they are the same on a machine without one.  CPU only."""
import pytest
import torch

from diffrast import DiffRast

TRI = torch.zeros((1, 3), dtype=torch.int32)


@pytest.mark.parametrize("call,msg", [
    (lambda: DiffRast.rasterize(torch.zeros(1, 3, 4), TRI, (4, 4)), "pos must be a tensor on a ROCm"),
    (lambda: DiffRast.rasterize(torch.zeros(1, 3, 4, requires_grad=True), TRI, (4, 4)),
     "pos must be on a ROCm"),
    (lambda: DiffRast.rasterize([[0.0]], TRI, (4, 4)), "pos must be a tensor"),
    (lambda: DiffRast.interpolate(torch.zeros(3, 2), torch.zeros(1, 2, 2, 3), TRI), "rast must be"),
    (lambda: DiffRast.interpolate(torch.zeros(3), torch.zeros(1, 2, 2, 4), TRI), "attr must be"),
    (lambda: DiffRast.interpolate(torch.zeros(5, 3, 2), torch.zeros(2, 2, 2, 4), TRI),
     "attr batch dim 5 incompatible with rast batch 2"),
    (lambda: DiffRast.interpolate(torch.zeros(3, 2), torch.zeros(1, 2, 2, 4), TRI[:, :2]),
     r"tri must be \[T, 3\] \(got \[1, 2\]\)"),
    (lambda: DiffRast.texture(torch.zeros(1, 4, 4, 3), torch.zeros(1, 2, 2, 2)), "ROCm device"),
    (lambda: DiffRast.antialias(torch.zeros(2, 2, 3), torch.zeros(1, 2, 2, 4), torch.zeros(1, 3, 4),
                                TRI), "color must be"),
    (lambda: DiffRast.antialias(torch.zeros(1, 2, 2, 3), torch.zeros(1, 2, 3, 4),
                                torch.zeros(1, 3, 4), TRI), "rast must match color"),
])
def test_value_errors(call, msg):
    with pytest.raises(ValueError, match=msg):
        call()


def test_prebuilt_mip_converts_nothing(monkeypatch):
    """A prebuilt pyramid is matched against the texture's shape; the texture
    itself is converted once, by the compiled node."""
    def refuse(*_, **__):
        raise AssertionError("converted")
    tex = torch.zeros(1, 4, 4, 3, dtype=torch.float16)
    monkeypatch.setattr(torch.Tensor, "to", refuse)
    with pytest.raises(ValueError, match="ROCm device"):
        DiffRast.texture(tex, torch.zeros(1, 2, 2, 2), uvDA=torch.zeros(1, 2, 2, 4),
                         filterMode="linear-mipmap-linear", mip=[tex])
