"""Few large structures, several workgroups each, against the same structures
in a batch of 65, which take one workgroup each: sizes at the edges of the rule
(10240 atoms, 32 structures), counts at the edges of a workgroup's share, strides
of every alignment."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("B,A", [(1, 8191), (1, 8192), (3, 8193), (2, 20002), (64, 8195), (40, 13000), (1, 66001),
                                 (1, 10239), (1, 10240), (3, 10241), (32, 10243), (33, 10243), (32, 17000)])
def test_split_matches_one_workgroup(dtype, B, A):
    from torchproteinlibrary_amd.RMSD import Coords2RMSD
    rng = np.random.default_rng(B * 7 + A)
    counts = [A, A - 1, 1024, 1025, 0, 1, 2, 1023, 4, 8191]
    n = torch.tensor([min(counts[k % len(counts)], A) for k in range(B)], dtype=torch.int32).cuda()
    step = rng.standard_normal((B, A, 3))
    x = np.cumsum(1.5 * step / np.linalg.norm(step, axis=2, keepdims=True), axis=1) + 50.0
    q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
    y = x @ q + 2.0 * rng.standard_normal((B, A, 3)) - 20.0
    x, y = (torch.from_numpy(v.reshape(B, 3 * A)).to(dtype).cuda() for v in (x, y))
    rep = -(-65 // B)
    got, want = [], []
    for k, out in ((1, got), (rep, want)):
        xx = x.repeat(k, 1).requires_grad_(True)
        layer = Coords2RMSD()
        r = layer(xx, y.repeat(k, 1), n.repeat(k))
        g, = torch.autograd.grad(r.sum(), xx)
        out += [r.detach()[:B], layer.UT[:B], g[:B]]
    # r^2 n = R2 - 2 lambda: both sums in another order, each within some units
    # of 2^-53 of R2 <= n d^2, d the largest distance of two atoms; U turns by
    # as much as the sums change against the spread of the structure.
    ref = torch.isfinite(want[0]) & (n > 3)
    assert torch.equal(torch.isfinite(got[0]), torch.isfinite(want[0]))
    for b in torch.nonzero(ref).flatten().tolist():
        k = int(n[b])
        c = x[b, :3 * k].double().view(-1, 3)
        c = c - c.mean(0)
        r2 = 4 * (c ** 2).sum().item()
        rmsd = want[0][b].double().item()
        tol = 256 * 2.0 ** -53 * r2 / (k * rmsd) + 2 * torch.finfo(dtype).eps * rmsd
        assert abs(got[0][b].double().item() - rmsd) <= tol, (b, k)
        spread = torch.linalg.svdvals(c)[1].item() ** 2
        turn = 256 * 2.0 ** -53 * r2 / spread + 2 * torch.finfo(dtype).eps
        assert (got[1][b] - want[1][b]).abs().max().double().item() <= turn, (b, k)
        far = c.norm(dim=1).max().item()
        tol = (turn * far + 2 * torch.finfo(dtype).eps * (far + 100)) / (k * rmsd) * 4
        assert (got[2][b] - want[2][b]).abs().max().double().item() <= tol, (b, k)
        assert not got[2][b, 3 * k:].any()


def test_split_errors():
    from torchproteinlibrary_amd.RMSD import Coords2RMSD
    x = torch.randn(2, 3 * 12000, device="cuda")
    y = torch.randn(2, 3 * 12000, device="cuda")
    n = torch.tensor([12000, 12000], dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError, match="num_atoms"):
        Coords2RMSD()(x, y, n + 1)
    x[1, 3 * 11999] = float("nan")
    with pytest.raises(Exception, match="forward Nan"):
        Coords2RMSD()(x, y, n)


@pytest.mark.parametrize("B,A", [(1, 10240), (8, 12001), (32, 10300), (2, 66001)])
def test_split_accuracy(B, A):
    """rmsd in float64 against the residuals of the layer's own rotation, summed
    in extended precision (the rotation's rounding counts in second order)."""
    from torchproteinlibrary_amd.RMSD import Coords2RMSD
    rng = np.random.default_rng(A)
    n = rng.integers(A // 2, A + 1, B)
    x, y = np.zeros((B, A, 3)), np.zeros((B, A, 3))
    for b, k in enumerate(n):
        step = rng.standard_normal((k, 3))
        x[b, :k] = np.cumsum(1.5 * step / np.linalg.norm(step, axis=1, keepdims=True), axis=0) + 30.0
        q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        q *= np.sign(np.linalg.det(q))
        y[b, :k] = x[b, :k] @ q + 2.0 * rng.standard_normal((k, 3)) - 20.0
    layer = Coords2RMSD()
    r = layer(*(torch.from_numpy(v.reshape(B, 3 * A)).cuda() for v in (x, y)),
              torch.from_numpy(n.astype(np.int32)).cuda()).cpu().numpy()
    ut = layer.UT.cpu().numpy().astype(np.longdouble)
    for b, k in enumerate(n):
        xb, yb = (v[b, :k].astype(np.longdouble) for v in (x, y))
        off = (xb - xb.mean(0)) - (yb - yb.mean(0)) @ ut[b].T
        dev = (off ** 2).sum() + np.longdouble(1e-10)
        # At most 30 roundings on an atom's way into the sums that keep both
        # parts, a third of 2^-53 each on average, over at least 120 of them.
        moments = ((xb - xb[0]) ** 2).sum() + ((yb - yb[0]) ** 2).sum()
        assert abs(r[b] - np.sqrt(dev / k)) <= 2.0 ** -53 * moments / (2 * np.sqrt(dev * k)) + 1e-15 * r[b], (b, k)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("B,A", [(3, 10240), (2, 12001)])
def test_split_does_not_depend_on_the_checks(dtype, B, A, monkeypatch):
    """Native function, Python function and the binding with a status word, with
    checks and without: the same kernels, so the same bits."""
    from torchproteinlibrary_amd._native_rmsd import ext
    from torchproteinlibrary_amd.RMSD.Coords2RMSD.Coords2RMSD import Coords2RMSDFunction
    python = type("PythonRMSD", (Coords2RMSDFunction,), {})
    gen = torch.Generator().manual_seed(A)
    x = torch.randn(B, A, 3, dtype=torch.float64, generator=gen).cumsum(1).reshape(B, 3 * A).to(dtype).cuda()
    y = (x.cpu().double() + torch.randn(B, 3 * A, dtype=torch.float64, generator=gen)).to(dtype).cuda()
    n = torch.tensor([A - k for k in range(B)], dtype=torch.int32).cuda()
    outs = []
    for checks in ("1", "0"):
        monkeypatch.setenv("TPL_A2B_CHECKS", checks)
        for fn in (Coords2RMSDFunction, python):
            xx = x.clone().requires_grad_(True)
            r, ut = fn.apply(xx, y, n)
            outs.append((r.detach(), ut, torch.autograd.grad(r.sum(), xx)[0]))
    for status in (None, torch.zeros(1, dtype=torch.int32, device="cuda")):
        r, ut = x.new_empty(B), x.new_empty(B, 3, 3)
        ext.Coords2RMSDGPU_forward(x, y, r, n, ut, None, status)
        outs.append((r, ut, outs[0][2]))
        assert status is None or int(status) == 0
    for o in outs[1:]:
        assert all(torch.equal(u, v) for u, v in zip(o, outs[0]))
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    ext.Coords2RMSDGPU_forward(x, y, r, n + 1000, ut, None, status)
    assert int(status) == 2


# Shapes that split, at the most workgroups a structure gets: 64 from 65536
# atoms on, 512 / B for 8 < B <= 32, a share per 1024 atoms below; few atoms in a
# long stride (1, 2 and 3 leave most shares empty, and the rotation of 1 and 2
# undetermined: their rmsd is compared).
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("B,A", [(8, 12001), (20, 12001), (20, 30000), (9, 57345), (1, 65535), (2, 65536), (3, 65537), (4, 10240)])
def test_split_shapes_match_one_workgroup(dtype, B, A):
    from torchproteinlibrary_amd.RMSD import Coords2RMSD
    gen = torch.Generator().manual_seed(B * 31 + A)
    counts = ([1, 2, 3, A, A - 1, 1025, 4, 5000] * 4)[:B] if B > 1 else [A]
    n = torch.tensor(counts, dtype=torch.int32).cuda()
    step = torch.randn(B, A, 3, dtype=torch.float64, generator=gen)
    x = (1.5 * step / step.norm(dim=2, keepdim=True)).cumsum(1) + 20.0
    y = x.flip(2) + 2.0 * torch.randn(B, A, 3, dtype=torch.float64, generator=gen)
    x, y = (v.reshape(B, 3 * A).to(dtype).cuda() for v in (x, y))
    got = Coords2RMSD()(x, y, n)
    rep = -(-33 // B)  # more than 32 structures take one workgroup each
    want = Coords2RMSD()(x.repeat(rep, 1), y.repeat(rep, 1), n.repeat(rep))[:B]
    for b, k in enumerate(counts):
        c, d = (v[b, :3 * k].double().view(-1, 3) for v in (x, y))
        r2 = float(((c - c[0]) ** 2).sum() + ((d - d[0]) ** 2).sum())
        rmsd = float(want[b])
        # r^2 n = R2 - 2 lambda + 1e-10 of sums that round, in either order, to
        # within 256 units of 2^-53 of r2; r itself is no more than sqrt of that off
        off = 256 * 2.0 ** -53 * r2
        tol = min(off / (k * rmsd), (off / k) ** 0.5) + 2 * torch.finfo(dtype).eps * rmsd
        assert abs(float(got[b]) - rmsd) <= tol, (b, k)
