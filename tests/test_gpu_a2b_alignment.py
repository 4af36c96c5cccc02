"""Angles2Backbone on inputs that start at every alignment and rows of every
length: forward and backward give the same bits as on fresh copies of the same
values (the same kernels and arithmetic, other accesses)."""
import pytest
import torch

from torchproteinlibrary_amd import _tuning

pytestmark = pytest.mark.gpu


def _at(offset, t):
    out = torch.empty(t.numel() + offset, dtype=t.dtype, device=t.device)[offset:].view(t.shape)
    return out.copy_(t)


@pytest.mark.parametrize("dtype,config", [(torch.float32, (1, 1)), (torch.float32, (2, 2)), (torch.float32, (4, 4)),
                                          (torch.float32, (8, 4)), (torch.float64, (1, 1)), (torch.float64, (2, 2)),
                                          (torch.float64, (4, 2))])
@pytest.mark.parametrize("B,L", [(3, 64), (5, 257), (3, 1026), (4, 515), (2, 4099)])
def test_any_alignment(dtype, config, B, L):
    from torchproteinlibrary_amd.ReducedModel import Angles2Backbone
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    g = torch.Generator().manual_seed(L)
    a = ((torch.rand(B, 3, L, generator=g) * 6 - 3).to(dtype)).cuda()
    w = torch.randn(B, 9 * L, generator=g).to(dtype).cuda()
    n = torch.tensor([L, L - 1, 1, L // 2, L // 3 + 1][:B], dtype=torch.int32).cuda()
    try:
        _tuning.set_config(a, config)
        want = None
        for offset in (0, 1, 2, 3):
            x = _at(offset, a).requires_grad_(True)
            out = Angles2Backbone()(x, n)
            grad, = torch.autograd.grad(out, x, _at(3 - offset, w))
            step = Angles2BackboneStep(x.detach(), n, config=config)
            step.grad_coords.copy_(w)
            step.replay()
            got = [out.detach(), grad, step.coords.clone(), step.grad_angles.clone()]
            want = want or got
            assert all(torch.equal(p, q) for p, q in zip(got, want)), offset
    finally:
        _tuning.clear()
