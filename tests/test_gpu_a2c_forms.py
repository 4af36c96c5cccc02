"""The forms of the Angles2Coords kernels agree: one workgroup per structure,
and the group kernels with a workspace, over the sizes where their blocks (64
residues), groups (256), rounds and staging end, for odd strides, empty and
flagged structures and scheduling orders."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import a2c_oracle as O
from torchproteinlibrary_amd import _build
from torchproteinlibrary_amd.FullAtomModel.Angles2Coords import convertStringList

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
FUSED, GROUPS = 1, 2


def _lib():
    lib = ctypes.CDLL(_build.lib_path("libtpl_a2c.so"))
    lib.tplx_a2c_workspace_bytes.restype = ctypes.c_size_t
    return lib


def _batch(lengths, L, seed, dtype, letters=O.AA20):
    rng = np.random.default_rng(seed)
    seqs = ["".join(rng.choice(list(letters), size=n)) for n in lengths]
    ang = np.zeros((len(lengths), 8, L))
    for b, n in enumerate(lengths):
        ang[b, 0, :n] = rng.normal(-1.1, 0.3, n)
        ang[b, 1, :n] = rng.normal(2.3, 0.4, n)
        ang[b, 2, :n] = np.pi + rng.normal(0, 0.05, n)
        ang[b, 3:, :n] = rng.uniform(-np.pi, np.pi, (5, n))
    return seqs, torch.tensor(ang, dtype=dtype, device=DEV)


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _forward(form, seqs, X, A, order=None, offset=0):
    """(coords, res_names, atom_names, status) of one form; outputs start full
    of other values, `offset` values into their buffers."""
    lib, B, L = _lib(), X.shape[0], X.shape[2]
    S = convertStringList(seqs).to(DEV)
    buf = torch.full((B * 3 * A + offset,), 7.0, dtype=X.dtype, device=DEV)
    coords = buf[offset:].view(B, 3 * A)
    rn = torch.full((B, A, 4), 255, dtype=torch.uint8, device=DEV)
    an = torch.full((B, A, 4), 255, dtype=torch.uint8, device=DEV)
    st = torch.zeros(1, dtype=torch.int32, device=DEV)
    ws = torch.empty(max(lib.tplx_a2c_workspace_bytes(B, L), 1), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    assert lib.tplx_a2c_forward(form, _p(order), 0 if X.dtype == torch.float32 else 1, _p(S), S.shape[1], _p(X), L,
                                _p(coords), _p(rn), _p(an), A, _p(ws), _p(st), None, B, None) == 0
    torch.cuda.synchronize()
    assert offset == 0 or bool((buf[:offset] == 7.0).all())
    return coords, rn, an, int(st.item())


def _tolerance(X, scale):
    """Two products of up to 3L rotations in float64 (8 roundings each), and
    one rounding to float32."""
    return scale * (3 * X.shape[2] * 8 * 2.0 ** -53 + (2.0 ** -23 if X.dtype == torch.float32 else 0.0))


SHAPES = [([1, 64, 65, 63], 65), ([65, 128, 127, 0, 3], 129), ([255, 256, 257, 64, 1], 257),
          ([513, 512, 30, 300], 515), ([1024, 1025, 1, 700], 1025), ([2100, 64, 1500], 2100), ([70] * 2050, 71)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_forward_forms_agree(shape, dtype):
    lengths, L = SHAPES[shape]
    seqs, X = _batch(lengths, L, 100 + shape, dtype)
    natoms = [O.num_atoms(s) for s in seqs]
    A = max(natoms) + (5, 2, 0, 3, 1, 4, 7)[shape]
    print(f"a2c forward forms: {len(lengths)} structures, stride {L}, {dtype}", flush=True)
    outs = [_forward(f, seqs, X, A, offset=shape % 3) for f in (FUSED, GROUPS)]
    assert outs[0][3] == outs[1][3] == 0
    scale = float(outs[0][0].abs().max())
    assert float((outs[0][0] - outs[1][0]).abs().max()) <= _tolerance(X, scale)
    for k in (1, 2):
        assert torch.equal(outs[0][k], outs[1][k])
    for c, rn, an, _ in outs:
        for b in range(0, len(lengths), max(1, len(lengths) // 8)):
            n = natoms[b]
            assert not c[b, 3 * n:].any() and not rn[b, n:].any() and not an[b, n:].any()
            res, atoms = O.names_one(seqs[b])
            assert [bytes(v).rstrip(b"\0").decode() for v in an[b, :n].cpu().numpy()] == atoms
            assert [bytes(v).rstrip(b"\0").decode() for v in rn[b, :n].cpu().numpy()] == res
    b = int(np.argmin([abs(n - 300) for n in lengths]))  # the oracle on one structure
    want = O.forward_one(seqs[b], X[b].double().cpu().numpy())[0]
    for c, *_ in outs:
        assert np.abs(c[b, :3 * natoms[b]].double().cpu().numpy() - want).max() <= _tolerance(X, scale)


@pytest.mark.parametrize("letters", ["W", "G", "P"])
def test_forward_forms_at_the_largest_and_smallest_residues(letters):
    seqs, X = _batch([64, 130, 300, 1], 300, 7, torch.float32, letters)
    A = max(O.num_atoms(s) for s in seqs)
    a, b = _forward(FUSED, seqs, X, A), _forward(GROUPS, seqs, X, A)
    assert float((a[0] - b[0]).abs().max()) <= _tolerance(X, float(a[0].abs().max()))
    assert torch.equal(a[1], b[1]) and torch.equal(a[2], b[2])
    one = _batch([64, 64, 3, 20, 33], 64, 8, torch.float64, letters)  # one block per structure
    n = [O.num_atoms(s) for s in one[0]]
    c = _forward(FUSED, one[0], one[1], max(n))[0]
    for k in range(5):
        want = O.forward_one(one[0][k], one[1][k].cpu().numpy())[0]
        assert np.abs(c[k, :3 * n[k]].cpu().numpy() - want).max() <= 1e-10


@pytest.mark.parametrize("L", [40, 200, 700])
def test_forward_forms_flag_alike(L):
    """A bad letter (in the last block), too many residues, too many atoms: the
    structure is zeros, its bit is set, the others are built."""
    good = "ACDEFGHIKLMNPQRSTVWY" * (L // 20)
    A = O.num_atoms(good)
    for bad, bit in ((good[:-1] + "X", 1), (good + "G", 2), ("W" * L, 4)):
        seqs = [good, bad, "G" * L, good[:30]]
        _, X = _batch([L] * 4, L, 3, torch.float32)
        outs = [_forward(f, seqs, X, A) for f in (FUSED, GROUPS)]
        for c, rn, an, st in outs:
            assert st == bit
            assert not c[1].any() and not rn[1].any() and not an[1].any()
            assert c[0].any() and c[2].any() and c[3].any()
        assert float((outs[0][0] - outs[1][0]).abs().max()) <= _tolerance(X, float(outs[0][0].abs().max()))


def test_forward_forms_take_an_order():
    seqs, X = _batch([300, 20, 500, 64, 257], 500, 11, torch.float32)
    A = max(O.num_atoms(s) for s in seqs)
    for form in (FUSED, GROUPS):
        plain = _forward(form, seqs, X, A)
        turned = _forward(form, seqs, X, A, torch.tensor([2, 0, 4, 3, 1], dtype=torch.int32, device=DEV))
        for k in range(3):
            assert torch.equal(plain[k], turned[k])
        c, rn, an, st = _forward(form, seqs, X, A, torch.tensor([2, 0, 5, 3, 1], dtype=torch.int32, device=DEV))
        assert st == 8
        assert bool((c[4] == 7.0).all()) and bool((rn[4] == 255).all())  # displaced: unwritten
        assert torch.equal(c[:4], plain[0][:4])


@pytest.mark.parametrize("lengths,L", [([21], 21), ([300, 40], 300), ([600] * 300, 600)])
def test_layer_raises_where_the_coordinate_sum_is_nan(lengths, L):
    from torchproteinlibrary_amd.FullAtomModel import Angles2Coords
    seqs, X = _batch(lengths, L, 5, torch.float32)
    Angles2Coords()(X, seqs)
    for value in (float("nan"), float("inf")):
        Y = X.clone()
        Y[-1, 0, lengths[-1] // 2] = value
        with pytest.raises(Exception, match="forward Nan"):
            Angles2Coords()(Y, seqs)
    Y = X.clone()
    Y[0, 7, :] = 1e9  # large, finite: no error
    Angles2Coords()(Y, seqs)


def _backward(form, seqs, coords, g, L, order=None):
    """(grad_angles, status) of one form; the output starts full of others."""
    lib, B, A = _lib(), coords.shape[0], coords.shape[1] // 3
    lib.tplx_a2c_backward_workspace_bytes.restype = ctypes.c_size_t
    S = convertStringList(seqs).to(DEV)
    ga = torch.full((B, 8, L), 7.0, dtype=coords.dtype, device=DEV)
    st = torch.zeros(1, dtype=torch.int32, device=DEV)
    ws = torch.empty(lib.tplx_a2c_backward_workspace_bytes(B, L), dtype=torch.uint8, device=DEV)
    torch.cuda.synchronize()
    assert lib.tplx_a2c_backward(form, _p(order), 0 if coords.dtype == torch.float32 else 1, _p(S), S.shape[1],
                                 _p(coords), _p(g), A, _p(ga), L, _p(ws), _p(st), None, B, None) == 0
    torch.cuda.synchronize()
    return ga, int(st.item())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_backward_forms_agree(shape, dtype):
    """Both forms sum the same float64 terms in other orders: up to 14L terms,
    each bounded by the largest gradient's terms, and one rounding."""
    lengths, L = SHAPES[shape]
    seqs, X = _batch(lengths, L, 200 + shape, dtype)
    natoms = [O.num_atoms(s) for s in seqs]
    coords = _forward(FUSED, seqs, X, max(natoms) + shape % 3)[0]
    g = torch.randn(coords.shape, dtype=dtype, device=DEV, generator=torch.Generator(DEV).manual_seed(shape))
    print(f"a2c backward forms: {len(lengths)} structures, stride {L}, {dtype}", flush=True)
    outs = [_backward(f, seqs, coords, g, L) for f in (FUSED, GROUPS)]
    assert outs[0][1] == outs[1][1] == 0
    tol = 14 * L * 2.0 ** -53 * 8 + (2.0 ** -23 if dtype == torch.float32 else 0.0)
    for b in range(len(lengths)):
        scale = float(outs[0][0][b].abs().max())
        assert float((outs[0][0][b] - outs[1][0][b]).abs().max()) <= tol * scale, b
        for ga, _ in outs:
            assert not ga[b, :, lengths[b]:].any()
    b = int(np.argmin([abs(n - 300) for n in lengths]))  # the oracle on one structure
    want = O.backward_fast(seqs[b], X[b].double().cpu().numpy(), g[b, :3 * natoms[b]].double().cpu().numpy())
    for ga, _ in outs:
        rel = np.abs(ga[b].double().cpu().numpy() - want).max() / np.abs(want).max()
        assert rel <= (1e-9 if dtype == torch.float64 else 1e-4), rel


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("letters", ["W", "G", "P"])
def test_backward_forms_at_the_largest_and_smallest_residues(letters, dtype):
    seqs, X = _batch([64, 130, 300, 1, 0], 301, 17, dtype, letters)
    coords = _forward(FUSED, seqs, X, max(O.num_atoms(s) for s in seqs))[0]
    g = torch.randn(coords.shape, dtype=dtype, device=DEV, generator=torch.Generator(DEV).manual_seed(1))
    for form in (FUSED, GROUPS):
        ga, st = _backward(form, seqs, coords, g, 301)
        assert st == 0 and not ga[4].any()
        for b in (0, 1, 3):
            n = O.num_atoms(seqs[b])
            want = O.backward_fast(seqs[b], X[b].double().cpu().numpy(), g[b, :3 * n].double().cpu().numpy())
            rel = np.abs(ga[b].double().cpu().numpy() - want).max() / max(np.abs(want).max(), 1e-12)
            assert rel <= (1e-9 if dtype == torch.float64 else 1e-4), (form, b, rel)


def test_backward_forms_flag_and_order_alike():
    L = 200
    good = O.AA20 * (L // 20)
    A = O.num_atoms(good)
    _, X = _batch([L] * 4, L, 3, torch.float32)
    g = torch.randn(4, 3 * A, device=DEV)
    for bad, bit in ((good[:-1] + "X", 1), (good + "G", 2), ("W" * L, 4)):
        seqs = [good, bad, "G" * L, good[:30]]
        coords = _forward(FUSED, seqs, X, A)[0]
        outs = [_backward(f, seqs, coords, g, L) for f in (FUSED, GROUPS)]
        for ga, st in outs:
            assert st == bit and not ga[1].any() and ga[0].any() and ga[2].any()
    seqs = [good, good[:70], "G" * L, good[:30]]
    coords = _forward(FUSED, seqs, X, A)[0]
    for form in (FUSED, GROUPS):
        plain = _backward(form, seqs, coords, g, L)[0]
        turned = _backward(form, seqs, coords, g, L, torch.tensor([2, 0, 3, 1], dtype=torch.int32, device=DEV))[0]
        assert torch.equal(plain, turned)
        ga, st = _backward(form, seqs, coords, g, L, torch.tensor([2, 0, -1, 1], dtype=torch.int32, device=DEV))
        assert st == 8 and bool((ga[3] == 7.0).all()) and torch.equal(ga[:3], plain[:3])


@pytest.mark.parametrize("lengths,L", [([21], 21), ([300, 40], 300), ([600] * 300, 600)])
def test_layer_raises_where_the_gradient_sum_is_nan(lengths, L):
    from torchproteinlibrary_amd.FullAtomModel import Angles2Coords
    seqs, X = _batch(lengths, L, 5, torch.float32)
    coords = Angles2Coords()(X.requires_grad_(True), seqs)[0]
    g = torch.zeros_like(coords)
    g[-1, 3 * (O.num_atoms(seqs[-1]) - 1)] = float("nan")
    with pytest.raises(Exception, match="backward Nan"):
        coords.backward(g)


def _through_the_binding(B, L, dtype):
    """A forward and a backward call on buffers that are there beforehand."""
    from torchproteinlibrary_amd._native_xform import ext
    seqs, X = _batch([L] * B, L, B, dtype)
    A = max(O.num_atoms(s) for s in seqs)
    S = convertStringList(seqs).to(DEV)
    coords, g = torch.empty(B, 3 * A, dtype=dtype, device=DEV), torch.randn(B, 3 * A, dtype=dtype, device=DEV)
    rn, an = (torch.empty(B, A, 4, dtype=torch.uint8, device=DEV) for _ in range(2))
    ga = torch.empty_like(X)

    def call():
        assert ext.Angles2Coords_forward_checked(S, X, coords, rn, an) == 0
        assert ext.Angles2Coords_backward_checked(g, ga, S, coords) == 0
    return call, (coords, rn, an, ga)


@pytest.mark.parametrize("B,L", [(512, 300), (32, 350), (256, 1000), (600, 128)])
def test_no_workspace_where_none_is_read(B, L):
    """One workgroup per structure: nothing is allocated beside the outputs."""
    call, outs = _through_the_binding(B, L, torch.float32)
    call()
    want = [t.clone() for t in outs]
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    call()
    assert torch.cuda.max_memory_allocated() == before
    assert all(torch.equal(u, v) for u, v in zip(outs, want))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_no_memory_for_the_workspace(dtype):
    """Where the workspace does not fit, the kernels without one do the call."""
    B, L = 320, 700
    call, outs = _through_the_binding(B, L, dtype)
    call()
    want = [t.clone() for t in outs]
    for t in outs:
        t.fill_(1)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(DEV).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 4096) / total)
    try:
        call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    eps = 2.0 ** -23 if dtype == torch.float32 else 0.0
    scale = float(want[0].abs().max())
    assert float((outs[0] - want[0]).abs().max()) <= scale * (3 * L * 8 * 2.0 ** -53 + eps)
    assert torch.equal(outs[1], want[1]) and torch.equal(outs[2], want[2])
    # the gradients' sums in another order, from coordinates that differ as above
    scale = want[3].abs().amax(dim=(1, 2), keepdim=True)
    assert ((outs[3] - want[3]).abs() <= scale * (14 * L * 8 * 2.0 ** -53 + 1e3 * eps)).all()


RUNS, TILES = 3, 4


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_run_and_tile_forms_agree(shape, dtype):
    """A run of residues per thread, and tiles, against a wave per block."""
    lengths, L = SHAPES[shape]
    seqs, X = _batch(lengths, L, 300 + shape, dtype)
    natoms = [O.num_atoms(s) for s in seqs]
    A = max(natoms) + (5, 2, 0, 3, 1, 4, 7)[shape]
    print(f"a2c run and tile forms: {len(lengths)} structures, stride {L}, {dtype}", flush=True)
    a, b = (_forward(f, seqs, X, A, offset=shape % 3) for f in (FUSED, RUNS))
    assert a[3] == b[3] == 0
    assert float((a[0] - b[0]).abs().max()) <= _tolerance(X, float(a[0].abs().max()))
    assert torch.equal(a[1], b[1]) and torch.equal(a[2], b[2])
    g = torch.randn(a[0].shape, dtype=dtype, device=DEV, generator=torch.Generator(DEV).manual_seed(shape))
    coords = a[0].clone()  # at the start of a buffer of its own
    outs = [_backward(f, seqs, coords, g, L) for f in (FUSED, RUNS) + ((TILES,) if L <= 2048 else ())]
    tol = 14 * L * 2.0 ** -53 * 8 + (2.0 ** -23 if dtype == torch.float32 else 0.0)
    scale = outs[0][0].abs().amax(dim=(1, 2), keepdim=True)
    for ga, st in outs:
        assert st == 0 and ((ga - outs[0][0]).abs() <= tol * scale).all()
        for k in range(len(lengths)):
            assert not ga[k, :, lengths[k]:].any()


@pytest.mark.parametrize("L", [40, 200, 700])
def test_run_and_tile_forms_flag_alike(L):
    good = "ACDEFGHIKLMNPQRSTVWY" * (L // 20)
    A = O.num_atoms(good)
    _, X = _batch([L] * 4, L, 3, torch.float32)
    g = torch.randn(4, 3 * A, device=DEV)
    for bad, bit in ((good[:-1] + "X", 1), (good + "G", 2), ("W" * L, 4)):
        seqs = [good, bad, "G" * L, good[:30]]
        c, rn, an, st = _forward(RUNS, seqs, X, A)
        assert st == bit and not c[1].any() and not rn[1].any() and not an[1].any()
        assert c[0].any() and c[2].any() and c[3].any()
        for form in (RUNS, TILES):
            ga, st = _backward(form, seqs, c, g, L)
            assert st == bit and not ga[1].any() and ga[0].any() and ga[2].any()
    seqs = [good, good[:70], "G" * L, good[:30]]
    turn = torch.tensor([2, 0, 3, 1], dtype=torch.int32, device=DEV)
    beyond = torch.tensor([2, 0, 4, 1], dtype=torch.int32, device=DEV)
    plain = _forward(RUNS, seqs, X, A)
    for k in range(3):
        assert torch.equal(_forward(RUNS, seqs, X, A, turn)[k], plain[k])
    c, _, _, st = _forward(RUNS, seqs, X, A, beyond)
    assert st == 8 and bool((c[3] == 7.0).all()) and torch.equal(c[:3], plain[0][:3])
    for form in (RUNS, TILES):
        ga = _backward(form, seqs, plain[0], g, L)[0]
        assert torch.equal(_backward(form, seqs, plain[0], g, L, turn)[0], ga)
        gb, st = _backward(form, seqs, plain[0], g, L, beyond)
        assert st == 8 and bool((gb[3] == 7.0).all()) and torch.equal(gb[:3], ga[:3])


# Shapes that the layer takes by runs (forward; backward in float64) and tiles (backward).
@pytest.mark.parametrize("B,L,dtype", [(512, 200, torch.float32), (400, 300, torch.float32), (64, 200, torch.float64)])
def test_layer_raises_from_every_form(B, L, dtype):
    from torchproteinlibrary_amd.FullAtomModel import Angles2Coords
    seqs, X = _batch([L] * B, L, 5, dtype)
    Y = X.clone()
    Y[-1, 1, L // 2] = float("nan")
    with pytest.raises(Exception, match="forward Nan"):
        Angles2Coords()(Y, seqs)
    Y = X.clone()
    Y[0, 7, :] = 1e9  # large, finite: no error
    Angles2Coords()(Y, seqs)
    coords = Angles2Coords()(X.requires_grad_(True), seqs)[0]
    g = torch.zeros_like(coords)
    g[-1, 3 * (O.num_atoms(seqs[-1]) - 1)] = float("nan")
    with pytest.raises(Exception, match="backward Nan"):
        coords.backward(g)
