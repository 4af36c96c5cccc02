"""Translate, rotate and centre at strides and starts of every alignment (the
16-byte accesses need only that of the values), around the edges of a wave's
256 atoms, against torch on the same values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _at(offset, *shape, dtype):
    """A contiguous tensor that starts `offset` values into its storage."""
    n = 1
    for s in shape:
        n *= s
    return torch.randn(n + offset, device="cuda", dtype=dtype)[offset:].view(*shape)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("offset", [0, 1, 2, 3])
@pytest.mark.parametrize("A", [1, 5, 255, 256, 257, 1023, 1025, 2050])
def test_any_alignment(dtype, offset, A):
    from torchproteinlibrary_amd import FullAtomModel as F
    B = 4
    n = torch.tensor([A, max(0, A - 1), min(A, 256), min(A, 3)], dtype=torch.int32, device="cuda")
    x, T = _at(offset, B, 3 * A, dtype=dtype).requires_grad_(True), torch.randn(B, 3, device="cuda", dtype=dtype)
    R = torch.linalg.qr(torch.randn(B, 3, 3, dtype=torch.float64))[0].to(dtype).cuda()
    g = _at(offset, B, 3 * A, dtype=dtype)
    mask = (torch.arange(A, device="cuda")[None, :] < n[:, None])[:, :, None]
    xa, ga = x.detach().view(B, A, 3), g.view(B, A, 3)
    eps = torch.finfo(dtype).eps

    out = F.CoordsTranslate()(x, T, n)
    assert torch.equal(out.view(B, A, 3), (xa + T[:, None, :]) * mask)
    assert torch.equal(torch.autograd.grad(out, x, g)[0].view(B, A, 3), ga * mask)

    out = F.CoordsRotate()(x, R, n)
    want = (xa.double() @ R.double().transpose(1, 2)) * mask
    # three products and two sums of values below |x| <= 6
    assert ((out.view(B, A, 3).double() - want).abs() <= 6 * 3 * 3 * eps).all()
    want = (ga.double() @ R.double()) * mask
    assert ((torch.autograd.grad(out, x, g)[0].view(B, A, 3).double() - want).abs() <= 6 * 3 * 3 * eps).all()

    n = n.clamp_min(1)  # a structure with no atoms has no centre (NaN, refused)
    mask = (torch.arange(A, device="cuda")[None, :] < n[:, None])[:, :, None]
    center = F.Coords2Center()(x, n)
    want = (xa.double() * mask).sum(1) / n[:, None]
    assert ((center.double() - want).abs() <= 6 * (eps + A * 2.0 ** -53)).all()
    gc = torch.randn(B, 3, device="cuda", dtype=dtype)
    grad, = torch.autograd.grad(center, x, gc)
    want = (gc.double()[:, None, :] / n[:, None, None].double()).expand(B, A, 3).masked_fill(~mask, 0)
    assert ((grad.view(B, A, 3).double() - want).abs() <= 6 * 2 * eps).all()
