"""The layers' autograd functions in native code against the Python functions
that they stand in for: the same values and gradients bit for bit (both launch
the same kernels), the same errors, and the Python function wherever a call is
not a plain eager one.  A subclass of a Function runs the Python one."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

NAMES = ("backbone", "rmsd", "translate", "rotate", "center", "fullatom")


def _functions(name):
    mod = {"backbone": "ReducedModel.Angles2Backbone.Angles2Backbone", "rmsd": "RMSD.Coords2RMSD.Coords2RMSD",
           "fullatom": "FullAtomModel.Angles2Coords.Angles2Coords"}.get(
               name, "FullAtomModel.CoordsTransform.CoordsTransform")
    m = importlib.import_module("torchproteinlibrary_amd." + mod)
    native = {"backbone": "Angles2BackboneGPUFunction", "rmsd": "Coords2RMSDFunction",
              "translate": "CoordsTranslateFunction", "rotate": "CoordsRotateFunction",
              "center": "Coords2CenterFunction", "fullatom": "Angles2CoordsFunction"}[name]
    native = getattr(m, native)
    return native, type("Python" + native.__name__, (native,), {})


def _args(name, dtype, B=3, L=37, seed=0):
    rng = np.random.default_rng(seed)
    t = lambda *s: torch.from_numpy(rng.standard_normal(s)).to(dtype).cuda()
    n = torch.tensor([L, 1, L // 2][:B], dtype=torch.int32).cuda()
    if name == "backbone":
        return t(B, 3, L), n
    if name == "rmsd":
        return t(B, 3 * L), t(B, 3 * L), n
    if name == "translate":
        return t(B, 3 * L), t(B, 3), n
    if name == "rotate":
        return t(B, 3 * L), t(B, 3, 3), n
    if name == "center":
        return t(B, 3 * L), n
    from torchproteinlibrary_amd.FullAtomModel import convertStringList
    from torchproteinlibrary_amd._native_xform import ext
    seqs = ["".join(rng.choice(list("ACDEFGHIKLMNPQRSTVWY"), k)) for k in n.tolist()]
    atoms = torch.tensor([ext.getSeqNumAtoms(s) for s in seqs], dtype=torch.int32).cuda()
    return t(B, 8, L), convertStringList(seqs).cuda(), atoms


def _outs(r):
    return list(r) if isinstance(r, (tuple, list)) else [r]


def _grads(fn, args, weight):
    x = args[0].detach().clone().requires_grad_(True)
    out = _outs(fn.apply(x, *args[1:]))
    w = weight(out[0])
    g, = torch.autograd.grad(out[0], x, w)
    return out, g


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_same_values(name, dtype):
    native, python = _functions(name)
    args = _args(name, dtype)
    # a gradient that is contiguous, expanded, transposed
    for weight in (torch.ones_like, lambda o: o.new_ones(1).expand_as(o),
                   lambda o: torch.randn(o.t().shape, generator=torch.Generator().manual_seed(1), dtype=o.dtype)
                   .to(o.device).t() if o.dim() == 2 else torch.ones_like(o)):
        a, ga = _grads(native, args, weight)
        b, gb = _grads(python, args, weight)
        assert len(a) == len(b) and torch.equal(ga, gb) and ga.dtype == gb.dtype and ga.stride() == gb.stride()
        for u, v in zip(a, b):
            assert torch.equal(u, v) and u.dtype == v.dtype and u.requires_grad == v.requires_grad
        assert type(a[0].grad_fn).__name__ != type(b[0].grad_fn).__name__
    with torch.no_grad():
        a, b = _outs(native.apply(*args)), _outs(python.apply(*args))
    assert all(torch.equal(u, v) and not u.requires_grad for u, v in zip(a, b))


def _error(call):
    try:
        call()
    except Exception as e:  # noqa: BLE001
        return type(e), str(e).split("\n")[0]
    return None


def _bad_calls(fn, name, dtype):
    """Calls that are refused, and calls with something around them."""
    args = _args(name, dtype)
    x = args[0]

    def grad(y, **kw):
        return torch.autograd.grad(_outs(fn.apply(y, *args[1:]))[0].sum(), y, **kw)

    def leaf():
        return x.detach().clone().requires_grad_(True)

    def twice():
        y = leaf()
        w = torch.ones_like(_outs(fn.apply(y, *args[1:]))[0]).requires_grad_(True)
        g, = torch.autograd.grad(_outs(fn.apply(y, *args[1:]))[0], y, w, create_graph=True)
        g.sum().backward()

    def again():
        y = leaf()
        o = _outs(fn.apply(y, *args[1:]))[0].sum()
        o.backward()
        o.backward()

    def changed():  # saved for the backward, then written (the translation saves only its vector)
        y = leaf()
        a = [t.clone() for t in args[1:]]
        z = y * 1
        o = _outs(fn.apply(z, *a))[0].sum()
        for t in a:
            t.add_(0)
        z.detach().add_(0)
        o.backward()

    def jvp():
        with torch.autograd.forward_ad.dual_level():
            fn.apply(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)), *args[1:])

    def nan():
        y = x.clone()
        y.view(-1)[0] = float("nan")
        fn.apply(y, *args[1:])

    def nan_back():
        y = leaf()
        o = _outs(fn.apply(y, *args[1:]))[0]
        torch.autograd.grad(o, y, torch.full_like(o, float("nan")))

    def long():
        a = list(args)
        if name == "fullatom":
            a[2] = a[2] - 5
        else:
            a[-1] = a[-1] + 1000
        fn.apply(*a)

    return dict(
        twice=twice, again=again, changed=changed, jvp=jvp, nan=nan, nan_back=nan_back, long=long,
        vmap=lambda: torch.func.vmap(lambda v: _outs(fn.apply(v, *args[1:]))[0])(x[None]),
        func_grad=lambda: torch.func.grad(lambda v: _outs(fn.apply(v, *args[1:]))[0].sum())(x),
        cpu=lambda: fn.apply(x.cpu(), *[a.cpu() for a in args[1:]]),
        half=lambda: fn.apply(x.half(), *args[1:]),
        rank=lambda: fn.apply(x[0], *args[1:]),
        strided=lambda: fn.apply(x.transpose(0, -1).contiguous().transpose(0, -1), *args[1:]),
        few=lambda: fn.apply(x),
        batch=lambda: fn.apply(x[:2], *args[1:]),
        other=lambda: fn.apply(x, *[None] * (len(args) - 1)),
        create_graph=lambda: grad(leaf(), create_graph=True),
    )


@pytest.mark.parametrize("name", NAMES)
def test_same_errors(name):
    native, python = _functions(name)
    a, b = (_bad_calls(f, name, torch.float32) for f in (native, python))
    for what in a:
        want = _error(b[what])
        got = _error(a[what])
        assert (got is None) == (want is None), (what, got, want)
        if want is not None:
            # a function says its own name in some of torch's messages
            strip = lambda e: (e[0], e[1].replace(python.__name__, native.__name__))
            assert got[0] is want[0], (what, got, want)
            if want[0] is not TypeError:
                assert strip(got) == strip(want), (what, got, want)


@pytest.mark.parametrize("name", NAMES)
def test_hooks_and_modes(name):
    native, python = _functions(name)
    args = _args(name, torch.float32)
    for fn in (native, python):
        packed = []

        def pack(t):
            packed.append(tuple(t.shape))
            return t.cpu()

        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.cuda()):
            x = args[0].clone().requires_grad_(True)
            out = _outs(fn.apply(x, *args[1:]))[0]
        g, = torch.autograd.grad(out.sum(), x)
        ref, gref = _grads(python, args, torch.ones_like)
        assert torch.equal(g, gref)
        if fn is native:
            first = packed
    assert len(first) == len(packed)

    # a mode sees the call as before: the Python function runs under it
    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, a=(), kw=None):
            return func(*a, **(kw or {}))

    x = args[0].clone().requires_grad_(True)
    with Mode():
        out = _outs(native.apply(x, *args[1:]))[0]
    assert "Backward" in type(out.grad_fn).__name__ and native.__name__ in type(out.grad_fn).__name__


def test_module_sequences():
    """The native preparation of sequences against the Function's inputs."""
    from torchproteinlibrary_amd import FullAtomModel as F
    seqs = ["ACDEFGHIKLMNPQRSTVWY", "", "GG", "W"]
    angles = torch.randn(4, 8, 20, device="cuda")
    layer = F.Angles2Coords()
    out = layer(angles, seqs)
    from torchproteinlibrary_amd._native_xform import ext
    counts = [ext.getSeqNumAtoms(s) if s else 0 for s in seqs]
    assert layer.num_atoms == counts and out[3].tolist() == counts and out[3].dtype == torch.int32
    ref = F.Angles2CoordsFunction.apply(angles, F.convertStringList(seqs).cuda(), out[3])
    assert all(torch.equal(u, v) for u, v in zip(out, ref))
    assert all(torch.equal(u, v) for u, v in zip(layer(angles, tuple(seqs)), ref))
    for bad in (["ACX", "A", "A", "A"], ["A\0C", "A", "A", "A"], ["a", "A", "A", "A"], ["Å", "A", "A", "A"]):
        with pytest.raises(ValueError, match="letter outside"):
            layer(angles, bad)
