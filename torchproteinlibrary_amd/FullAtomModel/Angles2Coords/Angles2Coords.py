"""Full-atom protein coordinates from angles on MI355X.

Drop-in for TorchProteinLibrary/FullAtomModel/Angles2Coords/Angles2Coords.py.
The names (``Angles2Coords``, ``Angles2CoordsFunction``,
``convertStringList``, ``convertString``), the call
``Angles2Coords()(input_angles, sequences)`` and what it returns are the
reference's (:34-87):

* ``input_angles`` ``[B, 8, L]`` (rows phi, psi, omega, xi1..xi5; residue i's
  N hangs on omega of residue i-1), float32 or float64, ``L`` at least the
  longest sequence; ``sequences`` a list of one-letter strings;
* returns ``(coords [B, 3*A], res_names [B, A, 4] uint8, atom_names
  [B, A, 4] uint8, num_atoms [B] int32)`` with ``A`` the largest atom count,
  coordinates and names 0 past each structure's atoms;
* the gradient flows to ``input_angles`` only; angles a structure does not
  use get 0;
* a NaN output raises ``Exception('Angles2CoordsFunction: forward Nan')`` /
  ``backward Nan`` (reference :53-54, 68-69).

What differs, by design: the work runs on the GPU (the angles must be a GPU
tensor; all four outputs are on its device), in FP64 inside whatever the
input dtype; a letter outside the 20 amino acids raises ``ValueError`` (the
reference silently skips the residue but still counts it); the backward is
O(atoms) per structure (the reference's is O(atoms x depth)) and works from
the saved output coordinates (bond axes and origins), so in float32 its
gradient carries the coordinates' rounding (about 1e-5 relative at 1000
residues).
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch
from torch.autograd import Function
from torch.autograd.function import once_differentiable
from torch.nn.modules.module import Module

from ..._native_xform import ext
from ..._plain import is_plain

__all__ = ["Angles2Coords", "Angles2CoordsFunction", "convertStringList", "convertString"]

_STATUS_SEQ, _STATUS_LENGTH, _STATUS_ATOMS, _STATUS_ORDER, _STATUS_RANGE = 1, 2, 4, 8, 16
_LETTERS = set("ACDEFGHIKLMNPQRSTVWY")


def convertStringList(stringList):
    """List of strings -> 0-terminated uint8 tensor [len, longest + 1]
    (reference Angles2Coords.py:12-26)."""
    maxlen = max([len(s) + 1 for s in stringList] + [1])
    ar = np.zeros((len(stringList), maxlen), dtype=np.uint8)
    for i, s in enumerate(stringList):
        b = np.frombuffer(bytes(s, "ascii"), dtype=np.uint8)
        ar[i, :b.shape[0]] = b
    return torch.from_numpy(ar)


def convertString(string):
    """A string -> 0-terminated uint8 tensor (reference :28-30)."""
    return torch.from_numpy(np.frombuffer(bytes(string + "\0", "ascii"), dtype=np.uint8).copy())


def schedule(num_atoms):
    """An order in which a GPU can take the structures, the most atoms first
    (ties in batch order), as an int32 CPU tensor, or None when every
    structure has the same size.  For callers of the C entry points that take
    one, whose kernels build one structure per workgroup; the layer needs
    none, since its kernels spread mixed sizes over the GPU themselves."""
    n = np.asarray(num_atoms, dtype=np.int64)
    if n.size < 2 or (n == n[0]).all():
        return None
    return torch.from_numpy(np.argsort(-n, kind="stable").astype(np.int32))


def _checks_enabled() -> bool:
    return os.environ.get("TPL_A2B_CHECKS", "1") != "0" and not torch.cuda.is_current_stream_capturing()


def _check(s, out, where):
    """Raises on the status bits of a checked call.  The kernels flag outputs
    that are NaN, infinite or huge (1e26); only then is the output summed."""
    if s & _STATUS_SEQ:
        raise ValueError("Angles2CoordsFunction: a sequence holds a letter outside the 20 amino acids")
    if s & _STATUS_LENGTH:
        raise ValueError("Angles2CoordsFunction: a sequence is longer than input_angles.size(2)")
    if s & _STATUS_ATOMS:
        raise ValueError("Angles2CoordsFunction: a structure has more atoms than the output holds")
    if s & _STATUS_ORDER:
        raise RuntimeError("Angles2CoordsFunction: the scheduling order holds an index outside the batch")
    if s & _STATUS_RANGE and math.isnan(out.sum()):
        raise Exception(f"Angles2CoordsFunction: {where} Nan")


def _native(input_angles, sequences, num_atoms, order=None, max_atoms=-1):
    """A plain eager call of the function below, as the same function in native
    code; None if the call is not a plain one."""
    if not is_plain((input_angles, sequences, num_atoms) + (() if order is None else (order,))):
        return None
    out = ext.Angles2Coords_apply(input_angles, sequences, num_atoms, order, max_atoms)
    return None if out is None else out + (num_atoms,)


class Angles2CoordsFunction(Function):
    """Protein angles -> coordinates (reference Angles2Coords.py:34-71).
    ``sequenceTensor`` is the uint8 [B, S] tensor of ``convertStringList`` on
    the angles' device.  ``order`` (optional, int32 [B]) is the order in
    which the GPU takes the structures (a permutation of 0..B-1; the outputs
    do not depend on it).  A plain eager call runs as the same function in
    native code."""

    @classmethod
    def apply(cls, *args, **kwargs):
        if cls is Angles2CoordsFunction and 3 <= len(args) <= 4 and not kwargs:
            out = _native(*args)
            if out is not None:
                return out
        return super().apply(*args, **kwargs)

    @staticmethod
    def forward(ctx, input_angles, sequenceTensor, num_atoms, order=None):
        if input_angles.dim() != 3 or input_angles.size(1) != 8:
            raise ValueError("Angles2CoordsFunction: input_angles must be [batch, 8, length], got "
                             f"{tuple(input_angles.size())}")
        if not input_angles.is_cuda:
            raise RuntimeError("Angles2CoordsFunction: this build runs on the GPU only; "
                               "input_angles must be a GPU tensor")
        input_angles = input_angles.contiguous()
        ctx.angles_shape = input_angles.shape
        dev = input_angles.device
        seqs = sequenceTensor.to(dev).contiguous()
        B = input_angles.size(0)
        max_atoms = int(num_atoms.max()) if num_atoms.numel() else 0
        coords = torch.empty(B, 3 * max_atoms, dtype=input_angles.dtype, device=dev)
        res_names = torch.empty(B, max_atoms, 4, dtype=torch.uint8, device=dev)
        atom_names = torch.empty(B, max_atoms, 4, dtype=torch.uint8, device=dev)
        if order is not None:
            order = order.to(dev).contiguous()
        if _checks_enabled():
            _check(ext.Angles2Coords_forward_checked(seqs, input_angles, coords, res_names, atom_names, order),
                   coords, "forward")
        else:
            ext.Angles2Coords_forward(seqs, input_angles, coords, res_names, atom_names, None, order)
        ctx.save_for_backward(seqs, coords)
        ctx.order = order
        ctx.mark_non_differentiable(res_names, atom_names, num_atoms)
        return coords, res_names, atom_names, num_atoms

    @staticmethod
    @once_differentiable
    def backward(ctx, grad_atoms, *unused):
        seqs, coords = ctx.saved_tensors
        grad_atoms = grad_atoms.contiguous()
        grad_angles = torch.empty(ctx.angles_shape, dtype=coords.dtype, device=coords.device)
        if _checks_enabled():
            _check(ext.Angles2Coords_backward_checked(grad_atoms, grad_angles, seqs, coords, ctx.order), grad_angles,
                   "backward")
        else:
            ext.Angles2Coords_backward_coords(grad_atoms, grad_angles, seqs, coords, None, ctx.order)
        return grad_angles, None, None, None


class Angles2Coords(Module):
    """``Angles2Coords()(input_angles, sequences)`` (reference :73-87); keeps
    the last call's atom counts in ``self.num_atoms``."""

    def __init__(self):
        super().__init__()
        self.num_atoms = None

    def forward(self, input_angles, sequences):
        if is_plain((input_angles,)) and type(sequences) in (list, tuple):
            prepared = ext.Angles2Coords_prepare(list(sequences), input_angles)
            if prepared is not None:
                self.num_atoms, seqs, num_atoms = prepared
                out = _native(input_angles, seqs, num_atoms, None, max(self.num_atoms))
                return Angles2CoordsFunction.apply(input_angles, seqs, num_atoms) if out is None else out
        for s in sequences:
            if not set(s) <= _LETTERS:
                raise ValueError("Angles2Coords: a sequence holds a letter outside the 20 amino acids: "
                                 f"{sorted(set(s) - _LETTERS)}")
        self.num_atoms = [ext.getSeqNumAtoms(s) if s else 0 for s in sequences]
        num_atoms = torch.tensor(self.num_atoms, dtype=torch.int32, device=input_angles.device)
        stringListTensor = convertStringList(sequences)
        return Angles2CoordsFunction.apply(input_angles, stringListTensor, num_atoms)
