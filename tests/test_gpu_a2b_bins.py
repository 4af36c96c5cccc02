"""The packed forward (chains of 3 to 8 chunks, several to a workgroup) against
the float64 host path, whatever the slots that the chains share.  Batch sizes at
the edge of the rule (beyond it the chunk kernels), lengths at the edges of the
chunks."""
import numpy as np
import pytest
import torch

from torchproteinlibrary_amd import _tuning

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,R", [(torch.float32, 1), (torch.float32, 2), (torch.float32, 4), (torch.float32, 8),
                                     (torch.float64, 1), (torch.float64, 2), (torch.float64, 4)])
@pytest.mark.parametrize("chunks,B", [(3, 4096), (4, 2100), (5, 700), (8, 300), (8, 4097)])
def test_packed_forward_matches_oracle(dtype, R, chunks, B):
    from torchproteinlibrary_amd.ReducedModel import Angles2Backbone
    C = 64 * R
    L = chunks * C - (3 if chunks % 2 else 0)
    if B * L > 2_500_000:
        B = max(9, 2_500_000 // L)
    rng = np.random.default_rng(B + L)
    edges = [0, 1, C, C + 1, 2 * C, 2 * C + 1, L - 1, L, 4 * C, 4 * C + 1]
    lens = np.minimum(np.concatenate([rng.choice(edges, B // 2), rng.integers(0, L + 1, B - B // 2)]), L)
    rng.shuffle(lens)
    lens = torch.from_numpy(lens.astype(np.int32)).cuda()
    angles = torch.rand(B, 3, L, device="cuda", dtype=dtype) * 6 - 3
    layer = Angles2Backbone()
    b = 2 if dtype == torch.float64 else 4
    try:
        _tuning.set_config(angles, (R, min(R, b)))
        out = layer(angles, lens)
        # Positions reach 3.8 A a residue and are rounded to the dtype twice
        # (the lane's own position, the result); the frames are products of 3 n
        # FP64 steps in another order than the host's.
        want = Angles2Backbone()(angles.double().cpu(), lens.cpu())
        n = lens.double().cpu().clamp_min(1)[:, None]
        tol = 3.8 * n * (2 * torch.finfo(dtype).eps + 64 * 3 * n * 2.0 ** -53)
        assert ((out.double().cpu() - want).abs() <= tol).all()
        past = torch.arange(9 * L, device="cuda")[None, :] >= 9 * lens[:, None]
        assert not out[past].any()
        bad = lens.clone()
        bad[B // 2] = L + 1
        with pytest.raises(ValueError, match="angles_length"):
            layer(angles, bad)
    finally:
        _tuning.clear()


def _check_forward(B, L, R, dtype, lens):
    from torchproteinlibrary_amd.ReducedModel import Angles2Backbone
    angles = torch.rand(B, 3, L, device="cuda", dtype=dtype, generator=torch.Generator("cuda").manual_seed(B)) * 6 - 3
    lens = torch.as_tensor(lens, dtype=torch.int32).cuda()
    try:
        _tuning.set_config(angles, (R, min(R, 2 if dtype == torch.float64 else 4)))
        out = Angles2Backbone()(angles, lens)
    finally:
        _tuning.clear()
    want = Angles2Backbone()(angles.double().cpu(), lens.cpu())
    n = lens.double().cpu().clamp_min(1)[:, None]
    tol = 3.8 * n * (2 * torch.finfo(dtype).eps + 64 * 3 * n * 2.0 ** -53)
    assert ((out.double().cpu() - want).abs() <= tol).all()
    assert not out[torch.arange(9 * L, device="cuda")[None, :] >= 9 * lens[:, None]].any()


# One workgroup per chain, 1 to 4 slots: the padding goes over the slots without
# a chunk, and a chain of one slot has some only if it is empty.
@pytest.mark.parametrize("dtype,R", [(torch.float32, 1), (torch.float32, 2), (torch.float32, 4), (torch.float64, 2)])
@pytest.mark.parametrize("slots", [1, 2, 3, 4])
def test_padding_of_one_workgroup_per_chain(dtype, R, slots):
    from torchproteinlibrary_amd.ReducedModel import Angles2Backbone
    C = 64 * R
    L = slots * C - (slots % 2)
    lens = torch.tensor([min(v, L) for v in (0, 1, C - 1, C, C + 1, 2 * C, 3 * C + 1, L, 0)], dtype=torch.int32).cuda()
    angles = torch.rand(9, 3, L, device="cuda", dtype=dtype, generator=torch.Generator("cuda").manual_seed(L)) * 6 - 3
    g = torch.randn(9, 9 * L, device="cuda", dtype=dtype, generator=torch.Generator("cuda").manual_seed(R))
    try:
        _tuning.set_config(angles, (R, R))
        torch.full((1 << 22,), float("nan"), device="cuda")  # what the outputs' memory may have held
        a = angles.clone().requires_grad_(True)
        out = Angles2Backbone()(a, lens)
        out.backward(g)
    finally:
        _tuning.clear()
    ac = angles.double().cpu().requires_grad_(True)
    want = Angles2Backbone()(ac, lens.cpu())
    want.backward(g.double().cpu())
    eps = torch.finfo(dtype).eps
    acc = 64 * 3 * L * 2.0 ** -53
    assert (out.detach().double().cpu() - want.detach()).abs().max() <= 3.8 * L * (2 * eps + acc)
    scale = ac.grad.abs().amax(dim=(1, 2), keepdim=True)
    assert ((a.grad.double().cpu() - ac.grad).abs() <= scale * 64 * eps + 3 * L * 3.8 * L * 6 * acc).all()
    for b, n in enumerate(lens.tolist()):
        assert not out[b, 9 * n:].any() and not a.grad[b, :, n:].any()


# Few workgroups with work, so that the zeros go over others too: batches below,
# at and above the 256 of these, one chain in all, none with a residue.
@pytest.mark.parametrize("dtype,R", [(torch.float32, 1), (torch.float32, 4), (torch.float64, 2)])
@pytest.mark.parametrize("B", [1, 9, 255, 256, 257, 300])
@pytest.mark.parametrize("kind", ["short", "one", "none"])
def test_packed_forward_of_short_chains_in_a_long_stride(dtype, R, B, kind):
    L = 64 * R * 8 - 5 if R < 4 else 64 * R * 7 - 5
    rng = np.random.default_rng(B)
    lens = rng.integers(0, 64 * R, B) if kind == "short" else np.zeros(B)
    if kind == "one":
        lens[B // 2] = L
    _check_forward(B, L, R, dtype, lens)


# The edges of the rule for packing.
@pytest.mark.parametrize("dtype,R,chunks,B", [
    (torch.float32, 1, 3, 2048), (torch.float32, 1, 3, 2049), (torch.float32, 1, 4, 3072), (torch.float32, 1, 4, 3073),
    (torch.float64, 1, 5, 512), (torch.float64, 1, 5, 513), (torch.float32, 2, 7, 513), (torch.float32, 4, 6, 127),
    (torch.float32, 4, 6, 128), (torch.float64, 4, 5, 191), (torch.float64, 4, 5, 192), (torch.float64, 4, 5, 256),
    (torch.float64, 4, 5, 257), (torch.float32, 8, 5, 192), (torch.float32, 1, 8, 4096)])
def test_packed_forward_at_the_edges_of_its_rule(dtype, R, chunks, B):
    L = 64 * R * chunks - 3
    rng = np.random.default_rng(B)
    lens = rng.integers(0, L + 1, B)
    lens[:3] = L, 0, 64 * R
    _check_forward(B, L, R, dtype, lens)
