"""The fp32 memory projection (``bf_mem_project_f32``) at the edges of its 32-token tiles, against 64 bits; and the calls that
keep the PyTorch operators. Tolerance: operands carry their 24 bits, sums of D products in fp32: 1e-6 of the norm.
"""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _ref(x, f, scale):
    return F.normalize(torch.einsum("bthd,hde->bthe", x.double().cpu(), f.double().cpu()), dim=-1) * scale


@pytest.mark.parametrize("b,t,h,d,layout", [
    (1, 64, 1, 256, "dense"), (1, 65, 3, 256, "heads first"), (2, 127, 5, 128, "dense"), (1, 200, 16, 64, "wide rows"),
    (3, 100, 2, 64, "heads first"), (1, 129, 2, 128, "unaligned"),
])
def test_projection_tiles(dev, b, t, h, d, layout):
    from heimdall_amd.hibrit import _project_f32
    gen = torch.Generator().manual_seed(t)
    x, f = torch.randn(b, t, h, d, generator=gen), torch.randn(h, d, d, generator=gen)
    if layout == "heads first":
        y = x.transpose(1, 2).contiguous().to(dev).transpose(1, 2)
    elif layout == "wide rows":
        y = torch.zeros(b, t, h, 2 * d, device=dev)[..., :d].copy_(x.to(dev))
    elif layout == "unaligned":
        y = torch.zeros(x.numel() + 1, device=dev)[1:].view(x.shape).copy_(x.to(dev))
    else:
        y = x.to(dev)
    ref = _ref(x, f, 0.25)
    with torch.no_grad():
        o = _project_f32(y, f.to(dev), 0.25)
    assert o.shape == ref.shape and ((o.double().cpu() - ref).norm() / ref.norm()).item() < 1e-6
    zero = _project_f32(torch.zeros_like(y), f.to(dev), 0.25)          # rows of no length stay zero
    assert not zero.any()


@pytest.mark.parametrize("d", [64, 128, 256])
def test_projection_of_nonfinite_values(dev, d):
    """What the operators give in 64 bits: a NaN in a projection makes the head's rows NaN, an infinity their other elements
    zero, a row with an infinity is NaN."""
    from heimdall_amd.hibrit import _project_f32
    gen = torch.Generator().manual_seed(d)
    x, f = torch.randn(1, 70, 3, d, generator=gen), torch.randn(3, d, d, generator=gen)
    f[0, 3, 5], f[1, 4, 6], x[0, 9, 2, 1] = float("nan"), float("inf"), float("inf")
    ref = torch.stack([F.normalize(x[:, :, h].double() @ f[h].double(), dim=-1) for h in range(3)], 2)
    with torch.no_grad():
        o = _project_f32(x.to(dev), f.to(dev), 1.0).cpu()
    assert torch.equal(o.isnan(), ref.isnan()) and not o.isinf().any()
    fin = ref.isfinite()
    assert (o.double() - ref)[fin].abs().max().item() < 1e-6


def test_recorded_and_transformed_calls(dev):
    """Gradients, vmap and forward mode go through PyTorch operators, with the same values."""
    from heimdall_amd.hibrit import _project_f32
    gen = torch.Generator().manual_seed(0)
    x, f = torch.randn(1, 80, 2, 64, generator=gen).to(dev), torch.randn(2, 64, 64, generator=gen).to(dev)
    plain = _project_f32(x, f, 1.0)
    xg = x.clone().requires_grad_(True)
    o = _project_f32(xg, f, 1.0)
    o.sum().backward()
    assert xg.grad is not None and (o - plain).abs().max().item() < 1e-5
    m = torch.vmap(lambda s: _project_f32(s, f, 1.0))(torch.stack((x, 2 * x)))
    assert (m - plain).abs().max().item() < 1e-5
    _, tangent = torch.func.jvp(lambda s: _project_f32(s, f, 1.0), (x,), (x,))
    assert tangent.abs().max().item() < 1e-4                            # along x the normalised rows do not change
