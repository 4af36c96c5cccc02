"""The step's own kernels (Angles2BackboneStep with equal chunk sizes in both
directions, and with long chains) against the float64 host path, at the sizes where it can go wrong:
empty and one-residue chains, chunk edges (64 R), chains of 1 to 8 chunks
and of up to 256 in groups of 64 (and one more, which takes the layer's kernels),
batches that fit on the GPU at once and batches packed by length, strides with
every alignment and padding past the chains.  Several runs on changed inputs,
under a capture too."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(B, L, lens, dtype, seed):
    rng = np.random.default_rng(seed)
    a = torch.from_numpy(rng.uniform(-np.pi, np.pi, (B, 3, L)))
    a[:, 2] = np.pi + 0.05 * a[:, 2]  # omega
    a = a.to(dtype).cuda()
    g = torch.from_numpy(rng.standard_normal((B, 9 * L))).to(dtype).cuda()
    return a, torch.tensor(lens, dtype=torch.int32, device="cuda"), g


def _oracle(a, lens, g):
    from torchproteinlibrary_amd import ReducedModel
    ac = a.double().cpu().requires_grad_()
    c = ReducedModel.Angles2Backbone()(ac, lens.cpu())
    # the step's gradients past the chain are not used
    c.backward(g.double().cpu())
    return c.detach(), ac.grad


def _check(step, a, lens, g, dtype):
    c, ga = _oracle(a, lens, g)
    L = a.size(2)
    nmax = max(1, int(lens.max()))
    eps = torch.finfo(dtype).eps
    # The frames are FP64; positions reach 3.8 A a residue, rounded once to the
    # dtype.  The step and the oracle differ by their order of products: 3 n
    # steps of a few units of 2^-53 each, on coordinates and on a gradient that
    # sums 3 n torques of up to 3.8 n times |g| < 6.
    acc = 64 * 3 * nmax * 2.0 ** -53
    tol_c = 3.8 * nmax * (eps + acc)
    scale = ga.abs().amax(dim=(1, 2), keepdim=True)
    tol_g = scale * eps + 3 * nmax * 3.8 * nmax * 6 * acc
    assert (step.coords.double().cpu() - c).abs().max() <= tol_c
    assert ((step.grad_angles.double().cpu() - ga).abs() <= tol_g).all()
    for b, n in enumerate(lens.tolist()):
        assert not step.coords[b, 9 * n:].any()
        assert not step.grad_angles[b, :, n:].any()


def _lengths(B, L, kind, C, rng):
    if kind == "equal":
        return [L] * B
    if kind == "long":  # groups of 64 chunks
        lens = [min(v, L) for v in (64 * C, 64 * C + 1, 64 * C - 1, 65 * C, 128 * C + 1, 192 * C, L, 0, 5 * C)]
        return lens[:B]
    edges = [0, 1, 2, C - 1, C, C + 1, 2 * C - 1, 2 * C, 2 * C + 1, 3 * C, 4 * C, 4 * C + 1, L - 1, L]
    lens = [min(e, L) for e in edges]
    lens += [int(v) for v in np.exp(rng.uniform(np.log(2), np.log(L), max(0, B - len(lens))))]
    rng.shuffle(lens)
    return lens[:B]


@pytest.mark.parametrize("dtype,R", [(torch.float32, 1), (torch.float32, 2), (torch.float32, 4),
                                     (torch.float64, 1), (torch.float64, 2)])
@pytest.mark.parametrize("B,L,kind", [
    (1, 1, "equal"), (3, 5, "equal"), (2, 127, "equal"), (2, 129, "equal"), (5, 512, "equal"),
    (17, 515, "mixed"), (14, 1023, "mixed"), (16, 1024, "mixed"), (18, 2048, "mixed"), (600, 333, "mixed"), (1100, 770, "mixed"),
    (1537, 514, "mixed"), (2050, 101, "mixed"), (4095, 259, "mixed"),
    (3, 2049, "equal"), (19, 4100, "mixed"), (9, 8400, "long"), (9, 16500, "long"),
])
def test_step_matches_oracle(dtype, R, B, L, kind):
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    rng = np.random.default_rng(B * 10007 + L)
    lens = _lengths(B, L, kind, 64 * R, rng)
    a, ln, g = _case(B, L, lens, dtype, B + L)
    step = Angles2BackboneStep(a, ln, config=(R, R))
    step.coords.fill_(float("nan"))
    step.grad_angles.fill_(float("nan"))
    step.grad_coords.copy_(g)
    step.replay()
    _check(step, a, ln, g, dtype)
    # new angles and lengths in the same memory
    a.copy_(a.flip(0))
    ln.copy_(ln.flip(0))
    step.replay()
    _check(step, a, ln, g, dtype)


@pytest.mark.parametrize("B", [5, 1500])
def test_step_under_capture(B):
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    L = 300
    a, ln, g = _case(B, L, _lengths(B, L, "mixed", 128, np.random.default_rng(1)), torch.float32, 1)
    step = Angles2BackboneStep(a, ln, config=(2, 2))
    step.grad_coords.copy_(g)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        step.replay()
    for _ in range(3):
        a.copy_(a.flip(0))
        step.coords.zero_()
        step.grad_angles.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got = step.coords.clone(), step.grad_angles.clone()
        step.replay()
        assert torch.equal(got[0], step.coords) and torch.equal(got[1], step.grad_angles)


@pytest.mark.parametrize("dtype,B,L,R", [
    (torch.float32, 3, 256, 1), (torch.float32, 3, 257, 2), (torch.float32, 3, 513, 4), (torch.float32, 3, 2048, 4),
    (torch.float32, 3, 2049, 1), (torch.float32, 16, 4096, 1), (torch.float32, 17, 4096, 2),
    (torch.float32, 3, 4097, 2), (torch.float32, 32, 4200, 4),
    (torch.float64, 3, 300, 2), (torch.float64, 3, 1024, 2), (torch.float64, 3, 1025, 1), (torch.float64, 20, 4097, 2),
])
def test_step_rule(dtype, B, L, R):
    from torchproteinlibrary_amd import _tuning
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    lens = _lengths(B, L, "mixed", 64 * R, np.random.default_rng(L))
    a, ln, g = _case(B, L, lens, dtype, B + L)
    step = Angles2BackboneStep(a, ln)
    assert step.config == (R, R)
    step.grad_coords.copy_(g)
    step.replay()
    _check(step, a, ln, g, dtype)
    # What a caller pins stays first, for the shape or for one mix of lengths.
    other = (2, 2) if R == 1 else (1, 1)
    try:
        for lengths in (ln, None):
            _tuning.clear()
            _tuning.set_config(a, other, lengths)
            assert _tuning.pinned_config(a, ln) == other
            assert Angles2BackboneStep(a, ln).config == other
    finally:
        _tuning.clear()
    assert _tuning.pinned_config(a, ln) is None


def test_step_of_nothing():
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    for B, L in ((0, 5), (3, 0)):
        step = Angles2BackboneStep(torch.zeros(B, 3, L, device="cuda"), torch.zeros(B, dtype=torch.int32, device="cuda"))
        step.replay()
        assert step.coords.shape == (B, 9 * L) and step.grad_angles.shape == (B, 3, L)


def test_step_on_another_stream_may_go_while_it_runs():
    """The memory that only the step holds is not handed out again before a run
    on another stream than the step's own has ended."""
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    B, L = 16, 8000
    a, ln, g = _case(B, L, _lengths(B, L, "mixed", 128, np.random.default_rng(3)), torch.float32, 3)
    step = Angles2BackboneStep(a, ln)
    step.grad_coords.copy_(g)
    step.replay()
    want = step.coords.clone(), step.grad_angles.clone()
    coords, grad, grad_coords = step.coords, step.grad_angles, step.grad_coords
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(200):
            step.replay()
    del step
    taken = [torch.full((n,), 255, dtype=torch.uint8, device="cuda") for n in (1 << 18, 1 << 20, 1 << 21, 1 << 22)]
    side.synchronize()
    assert torch.equal(coords, want[0]) and torch.equal(grad, want[1])
    del taken, grad_coords


@pytest.mark.parametrize("B,lo,R", [(600, 500, 2), (768, 500, 2), (769, 500, 4), (1536, 200, 2), (3073, 100, 4)])
def test_step_rule_counts_waves(B, lo, R):
    """float32, strides of 257..512 residues: 2 per lane while 3 waves on each of 1024 SIMDs hold all chunks."""
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    a, ln, g = _case(B, 500, [lo] * B, torch.float32, B)
    step = Angles2BackboneStep(a, ln)
    assert step.config == (R, R)
    step.grad_coords.copy_(g)
    step.replay()
    _check(step, a, ln, g, torch.float32)


@pytest.mark.parametrize("L", [500, 8000])
def test_step_alone_on_another_stream_may_go_while_it_runs(L):
    """As above where the caller keeps nothing at all, neither the angles nor the
    outputs: none of that memory is handed out before the runs have ended."""
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    B = 16
    a, ln, g = _case(B, L, [L] * B, torch.float32, 3)
    step = Angles2BackboneStep(a, ln)
    step.grad_coords.copy_(g)
    held = [a, ln, step.grad_coords, step.coords, step.grad_angles, step._state, step._sync]
    held = [(t.data_ptr(), t.nbytes) for t in held if t.nbytes]
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        busy = torch.empty(1 << 30, dtype=torch.uint8, device="cuda")
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(200):  # some 50 ms before the runs begin
            busy.fill_(1)
        for _ in range(20):
            step.replay()
    del step, a, ln
    taken = [torch.empty(size, dtype=torch.uint8, device="cuda") for _, size in held for _ in range(2)]
    assert not side.query()  # still running: nothing may have been given out
    for t in taken:
        assert all(t.data_ptr() + t.nbytes <= p or t.data_ptr() >= p + size for p, size in held)
    side.synchronize()


@pytest.mark.parametrize("dtype,R,L,B", [
    (torch.float32, 1, 64, 768), (torch.float64, 1, 33, 768), (torch.float32, 2, 128, 1536), (torch.float32, 1, 128, 1536),
    (torch.float64, 1, 65, 1536), (torch.float32, 2, 256, 1536), (torch.float64, 2, 129, 3072), (torch.float32, 1, 129, 1280),
    (torch.float32, 1, 256, 1280), (torch.float64, 1, 256, 3072)])
def test_step_kernel_of_few_chunks_up_to_a_batch(dtype, R, L, B):
    """Up to B chains of few chunks the step's own kernel, beyond them the layer's two."""
    from torchproteinlibrary_amd._native import ext
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    f64 = dtype == torch.float64
    assert ext.step_fits(f64, B, L, [R, R]) and not ext.step_fits(f64, B + 1, L, [R, R])
    for batch in (B, B + 1):
        a, ln, g = _case(batch, L, _lengths(batch, L, "mixed", 64 * R, np.random.default_rng(L)), dtype, batch)
        step = Angles2BackboneStep(a, ln, config=(R, R))
        step.grad_coords.copy_(g)
        step.replay()
        _check(step, a, ln, g, dtype)


@pytest.mark.parametrize("R", [1, 2])
@pytest.mark.parametrize("B,L,kind", [(600, 333, "mixed"), (16, 1024, "mixed"), (3, 2049, "equal"), (19, 4100, "mixed"),
                                      (9, 8400, "long"), (9, 16500, "long")])
def test_step_gradients_in_float64(R, B, L, kind):
    """Relative to each chain's largest gradient.  The frame of a residue is a
    product of 3 n steps, which turns with their roundings (3 n of them, some
    2^-53 each), and a torque sum of as many terms as the gradient rounds less:
    8 n 2^-53, 1.5e-11 at the longest; a record or a sum in float32 is 6e-8 off."""
    from torchproteinlibrary_amd.ReducedModel.Angles2Backbone.Angles2Backbone import Angles2BackboneStep
    lens = _lengths(B, L, kind, 64 * R, np.random.default_rng(L + R))
    a, ln, g = _case(B, L, lens, torch.float64, B + L)
    step = Angles2BackboneStep(a, ln, config=(R, R))
    step.grad_coords.copy_(g)
    step.replay()
    c, ga = _oracle(a, ln, g)
    n = ln.double().cpu().clamp_min(1)
    scale = ga.abs().amax(dim=(1, 2))
    off = (step.grad_angles.cpu() - ga).abs().amax(dim=(1, 2))
    assert (off <= 8 * n * 2.0 ** -53 * scale).all(), (off / scale / n * 2.0 ** 53).max()
    reach = c.abs().amax(dim=1)
    assert ((step.coords.cpu() - c).abs().amax(dim=1) <= 8 * n * 2.0 ** -53 * reach).all()
