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
