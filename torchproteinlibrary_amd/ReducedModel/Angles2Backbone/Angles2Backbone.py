"""Angles2Backbone: backbone dihedral angles -> N/CA/C coordinates, on MI355X.

Drop-in for TorchProteinLibrary/ReducedModel/Angles2Backbone/Angles2Backbone.py.
The names (``Angles2Backbone``, ``Angles2BackboneGPUFunction``), the call
``Angles2Backbone()(input, angles_length)``, the shapes, the output layout and
the error behaviour are the reference's:

* ``input``: ``[B, 3, L_max]`` contiguous, rows phi, psi, omega in radians,
  float32 (the reference GPU dtype) or float64; ``angles_length``: int32
  ``[B]`` on the same device (reference :12-30, angles2backbone_interface.cpp:12-15);
* returns ``[B, 9*L_max]`` coordinates N0, CA0, C0, N1, ... with exact zeros
  past each chain; gradient flows to ``input`` only (reference :52);
* device/contiguity/dtype violations raise ``RuntimeError`` (Math/nUtil.h:49-57),
  a wrong rank raises ``Exception`` (reference :22-23), and a NaN output raises
  ``Exception('Angles2BackboneFunction: forward Nan')`` / ``backward Nan``
  (reference :27-28, :49-50).

What differs, by design:

* the forward is a parallel FP64 prefix scan over per-residue rigid transforms
  and the backward an O(L) reverse-scan adjoint that recomputes the frames
  from the input angles and one FP64 checkpoint frame per 64-256 residues
  saved by the forward (no ``A``/``dr_dangle`` buffers: the reference's ``A``
  is 192 bytes per residue and its ``dr_dangle`` O(B*L^2), 110 GB at B=1024,
  L=1000); the checkpoints are kept only when the input requires grad;
* gradients of psi[len-1] and omega[len-1] are exactly 0 (the reference reads
  frames past the chain there);
* lengths outside [0, L_max] are clamped on the device and reported (the
  reference writes out of bounds);
* the NaN / length checks read status flags that the kernels write into host
  memory (one host sync, like the reference's ``output.sum()``); they are skipped while a
  stream is being captured, and ``TPL_A2B_CHECKS=0`` turns them off;
* the look-back words of the kernels live in one zero-initialised buffer per
  (device, stream), whose tickets, counters and flags every call returns to
  zero;
* CPU tensors (float64, as the reference's CPU path requires) go to a host
  library: the same FP64 recurrence per chain and the O(L) adjoint from the
  forward's coordinates, chains spread over torch.get_num_threads() threads,
  where the reference builds an O(L^2) derivative tensor on one thread.
"""
from __future__ import annotations

import os
import warnings

import torch
from torch.autograd import Function
from torch.autograd.function import once_differentiable
from torch.nn.modules.module import Module

from ... import _tuning
from ..._native import ext
from ..._plain import is_plain

_STATUS_NAN = 1
_STATUS_LENGTH = 2
_STATUS_TIMEOUT = 4
_STATUS_SYNC = 8


def _checks_enabled() -> bool:
    return os.environ.get("TPL_A2B_CHECKS", "1") != "0" and not torch.cuda.is_current_stream_capturing()


def _status_word(device):
    return torch.zeros(1, dtype=torch.int32, device=device) if _checks_enabled() else None


def _run_checked(checked, where: str, sync) -> None:
    """Runs checked(), which returns the call's status bits, and raises on
    them.  A look-back timeout or unclean look-back words make the result
    invalid: the words are cleared and the call is run once more, with a
    RuntimeWarning, and only a second failure raises.  The kernels' waits are
    bounded (a wave that never sees its record gives up and reports TIMEOUT
    instead of hanging), so this is the recovery path for a call that ran out
    of wait time."""
    bits = checked()
    if bits & (_STATUS_TIMEOUT | _STATUS_SYNC):
        ext.sync_clear(sync)  # look-back words may be left set
        _report_lost(bits, where, True)
        bits = checked()
        if bits & (_STATUS_TIMEOUT | _STATUS_SYNC):
            ext.sync_clear(sync)
            _report_lost(bits, where, False)
    _raise_on_bits(bits, where)


def _report_lost(bits: int, where: str, repeated: bool) -> None:
    what = "look-back wait timed out" if bits & _STATUS_TIMEOUT else "look-back words were not clean"
    if not repeated:
        raise RuntimeError("Angles2BackboneFunction: %s %s (result invalid)" % (where, what))
    warnings.warn("Angles2BackboneFunction: %s %s; cleared and repeated" % (where, what), RuntimeWarning)


def _raise_on_status(status, where: str) -> None:
    if status is None:
        return
    bits = int(status.item())
    if bits & (_STATUS_TIMEOUT | _STATUS_SYNC):
        raise RuntimeError("Angles2BackboneFunction: %s look-back failed (result invalid)" % where)
    _raise_on_bits(bits, where)


def _raise_on_bits(bits: int, where: str) -> None:
    if bits & _STATUS_LENGTH:
        raise ValueError("Angles2BackboneFunction: angles_length outside [0, input.size(2)] "
                         "(clamped on the device)")
    if bits & _STATUS_NAN:
        raise Exception("Angles2BackboneFunction: %s Nan" % where)


def _check_rank(input_angles):
    if len(input_angles.size()) != 3:
        raise Exception("Angles2BackboneFunction: ", "Incorrect input size:", input_angles.size())


def _empty_bytes(n, device):
    return torch.empty(int(n), dtype=torch.uint8, device=device)


class Angles2BackboneGPUFunction(Function):
    """Backbone angles -> backbone coordinates (chunk scan forward, O(L)
    adjoint backward from checkpoints).

    Reference: TorchProteinLibrary/ReducedModel/Angles2Backbone/Angles2Backbone.py:8-52.
    A plain eager call runs as the same function in native code.
    """

    @classmethod
    def apply(cls, *args, **kwargs):
        if (cls is Angles2BackboneGPUFunction and len(args) == 2 and not kwargs and is_plain(args)
                and args[0].dim() == 3 and ext.Angles2Backbone_plain(*args)):
            return ext.Angles2Backbone_apply(*args, _tuning.config_for(*args))
        return super().apply(*args, **kwargs)

    @staticmethod
    def forward(ctx, input_angles, angles_length):
        _check_rank(input_angles)
        B, _, L = input_angles.shape
        cfg = _tuning.config_for(input_angles, angles_length)
        dev = input_angles.device
        coords = torch.empty(B, 9 * L, dtype=input_angles.dtype, device=dev)
        st_bytes, sy_bytes = ext.workspace_bytes(input_angles.dtype == torch.float64, B, L,
                                                 list(cfg))
        state = _empty_bytes(st_bytes, dev) if ctx.needs_input_grad[0] else None
        sync = ext.sync_buffer(input_angles, sy_bytes)
        if _checks_enabled():
            _run_checked(lambda: ext.Angles2BackboneGPU_forward_checked(input_angles, coords, angles_length,
                                                                        state, sync, cfg),
                         "forward", sync)
        else:
            ext.Angles2BackboneGPU_forward(input_angles, coords, angles_length, state, sync, None, cfg)
        if state is not None:
            ctx.save_for_backward(input_angles, angles_length, state)
        ctx.cfg = cfg
        return coords

    @staticmethod
    @once_differentiable
    def backward(ctx, gradOutput):
        input_angles, angles_length, state = ctx.saved_tensors
        gradOutput = gradOutput.contiguous()
        if gradOutput.dtype != input_angles.dtype:
            gradOutput = gradOutput.to(input_angles.dtype)
        B, _, L = input_angles.shape
        dev = input_angles.device
        gradInput = torch.empty(B, 3, L, dtype=input_angles.dtype, device=dev)
        _, sy_bytes = ext.workspace_bytes(input_angles.dtype == torch.float64, B, L, list(ctx.cfg))
        sync = ext.sync_buffer(input_angles, sy_bytes)
        if _checks_enabled():
            _run_checked(lambda: ext.Angles2BackboneGPU_backward_checked(gradInput, gradOutput, input_angles,
                                                                         angles_length, state, sync, ctx.cfg),
                         "backward", sync)
        else:
            ext.Angles2BackboneGPU_backward(gradInput, gradOutput, input_angles, angles_length, state, sync,
                                            None, ctx.cfg)
        return gradInput, None


class Angles2BackboneCPUFunction(Function):
    """Backbone angles -> backbone coordinates on the host, float64.

    Reference: TorchProteinLibrary/ReducedModel/Angles2Backbone/Angles2Backbone.py:54-93
    (same names, float64 only, same error strings).
    """

    @staticmethod
    def forward(ctx, input, angles_length):
        _check_rank(input)
        B, _, L = input.shape
        coords = torch.empty(B, 9 * L, dtype=torch.double)
        bits = ext.Angles2BackboneCPU_forward(input, coords, angles_length, torch.get_num_threads())
        if bits & _STATUS_LENGTH:
            raise ValueError("Angles2BackboneFunction: angles_length outside [0, input.size(2)] "
                             "(clamped)")
        if bits & _STATUS_NAN:
            raise Exception('Angles2BackboneFunction: output_coords_cpu forward Nan')
        ctx.save_for_backward(coords, angles_length)
        return coords

    @staticmethod
    @once_differentiable
    def backward(ctx, gradOutput_cpu):
        coords, angles_length = ctx.saved_tensors
        gradOutput_cpu = gradOutput_cpu.contiguous().to(torch.double)
        B, L = coords.shape[0], coords.shape[1] // 9
        gradInput_cpu = torch.empty(B, 3, L, dtype=torch.double)
        bits = ext.Angles2BackboneCPU_backward(gradInput_cpu, gradOutput_cpu, coords, angles_length,
                                               torch.get_num_threads())
        if bits & _STATUS_NAN:
            raise Exception('Angles2BackboneFunction: gradInput_cpu backward Nan')
        return gradInput_cpu, None


class Angles2BackbonePlainGPUFunction(Function):
    """The plain form: one thread per chain runs the serial recurrence.  The
    backward is the O(L^2) per-pair formula with one thread per angle.  It is
    the baseline the scan path is measured against (same API)."""

    @staticmethod
    def forward(ctx, input_angles, angles_length):
        _check_rank(input_angles)
        B, _, L = input_angles.shape
        dev = input_angles.device
        coords = torch.empty(B, 9 * L, dtype=input_angles.dtype, device=dev)
        frames = _empty_bytes(ext.plain_frames_bytes(input_angles.dtype == torch.float64, B, L), dev)
        status = _status_word(dev)
        ext.Angles2BackboneGPU_forward_plain(input_angles, coords, angles_length, frames, status)
        _raise_on_status(status, "forward")
        ctx.save_for_backward(input_angles, angles_length, frames)
        return coords

    @staticmethod
    @once_differentiable
    def backward(ctx, gradOutput):
        input_angles, angles_length, frames = ctx.saved_tensors
        gradOutput = gradOutput.contiguous().to(input_angles.dtype)
        B, _, L = input_angles.shape
        gradInput = torch.empty(B, 3, L, dtype=input_angles.dtype, device=input_angles.device)
        status = _status_word(input_angles.device)
        ext.Angles2BackboneGPU_backward_plain(gradInput, gradOutput, input_angles, angles_length,
                                              frames, status)
        _raise_on_status(status, "backward")
        return gradInput, None


class Angles2Backbone(Module):
    """``Angles2Backbone()(input [B,3,L], angles_length int32 [B]) -> [B, 9L]``.

    Reference: TorchProteinLibrary/ReducedModel/Angles2Backbone/Angles2Backbone.py:96-104:
    GPU tensors go to the chunk kernels, CPU tensors to the host library.
    ``form="plain"`` selects the GPU baseline kernels instead of the scan.
    """

    def __init__(self, form: str = "scan"):
        super(Angles2Backbone, self).__init__()
        if form not in ("scan", "plain"):
            raise ValueError("form must be 'scan' or 'plain'")
        self.form = form

    def forward(self, input, angles_length):
        if not input.is_cuda:
            if self.form == "plain":
                raise RuntimeError("Angles2Backbone: the plain form runs on the GPU only")
            return Angles2BackboneCPUFunction.apply(input, angles_length)
        if self.form == "plain":
            return Angles2BackbonePlainGPUFunction.apply(input, angles_length)
        return Angles2BackboneGPUFunction.apply(input, angles_length)


def _step_residues(dtype, B, L, lengths):
    """Residues per lane of a step, or None where only timing tells.
    ``lengths()`` gives the lengths on the host, or None where they must not be
    read; it is called only where the mix decides.

    The tuner times the layer's two kernels, and the step's own behave
    otherwise: up to 8 chunks a chain (4 of 64 residues) are one kernel (1 to 4
    chunks of few residues per lane only up to a batch; beyond it the layer's
    two, as tuned), more are two, and a wave has both directions' work, so a lane's residues are the
    length of its chain of operations while the GPU is not full.  Steps, us,
    by residues per lane (equal lengths, float32 unless marked):
      one kernel while it can be, with few residues per lane:
        512 x 100      1:  7.8  2:  9.2    1024 x 20..256  1: 11.8  2: 13.7
        32 x 700, f64  1: 13.1  2: 10.2    128 x 1030      2: 19.1  4: 13.9
      but only while all waves of 2 fit, 3 on a SIMD (waves in brackets):
        1024 x 30..512 [1900]  2: 13.1  4: 16.8    800 x 500  [3200]  2: 20.0  4: 15.8
        1500 x 30..500 [2700]  2: 16.5  4: 19.5    1500 x 500 [6000]  2: 30.3  4: 26.6
      and of 1 no line shows (4000 x 200  1: 66.3  2: 59.2, x 10..200  1: 45.5  2: 48.5);
      in two kernels, as many waves as there are SIMDs (1024), in chains of at
      most 64 chunks of 64 (one record per lane to scan):
        16 x 4000      1: 13.6  2: 15.0  4: 17.9
        32 x 4000      1: 18.1  2: 15.3  4: 17.9
        32 x 5000      1: 27.1  2: 20.4  4: 18.4
        1 x 16384      1: 20.0  2: 17.1  4: 17.5
    """
    most = 4 if dtype == torch.float32 else 2
    if L <= 256:
        return 1 if B <= 2048 else None
    if L <= 512:
        if most == 2 or B <= 512:
            return 2
        n = lengths()
        return None if n is None else 2 if int(((n.clamp(0, L) + 127) // 128).sum()) <= 3072 else 4
    if L <= 512 * most:
        return most
    if L <= 4096 and B * -(-L // 64) <= 1024:
        return 1
    return 2 if B * -(-L // 128) <= 1024 else most


class Angles2BackboneStep:
    """Angles2Backbone forward and backward for fixed shapes, laid out once
    and replayed.

    For loops that run the same shapes many times (fitting, serving): one
    ``replay()`` runs the forward (``angles`` -> ``coords``) and the backward
    (``grad_coords`` -> ``grad_angles``) on the current stream, with nothing
    allocated, no host synchronisation and one launch per step, or two: chains
    of at most 8 chunks run in one kernel when both directions have the same
    chunk size (in float64 always) and, with few short chunks, the batch is not
    too large for it, chains of up to 256 chunks in two, other shapes in the
    layer's two.  In the step's own kernels the coordinates are
    those the gradients are computed from, rounded once from float64; they can
    differ from the layer's in the last digits.
    A step reads ``angles``, ``angles_length`` and ``grad_coords`` from their
    memory at every replay, so a loop updates them in place between replays;
    it writes ``coords`` and ``grad_angles``.  A replay under a capture is
    captured.  The chunk sizes are ``config`` (forward, backward residues per
    lane), those pinned for these inputs, those of a rule on the shape
    (``_step_residues``), or the tuned ones (the backward's for both
    directions where the step has kernels of its own).

    Replays do not check for NaN or out-of-range lengths (the checks of the
    layer read a status word on the host); lengths must stay within
    ``[0, angles.size(2)]``.  There is no counterpart in the reference, whose
    layer synchronises the host on every call (Angles2Backbone.py:27,49).
    """

    def __init__(self, angles, angles_length, config=None):
        _check_rank(angles)
        if not angles.is_cuda or not angles_length.is_cuda:
            raise RuntimeError("Angles2BackboneStep: angles and angles_length must be GPU tensors")
        if not angles.is_contiguous() or not angles_length.is_contiguous():
            raise RuntimeError("Angles2BackboneStep: angles and angles_length must be contiguous")
        if angles.dtype not in (torch.float32, torch.float64) or angles_length.dtype != torch.int32:
            raise RuntimeError("Angles2BackboneStep: angles must be float32 or float64, angles_length int32")
        B, _, L = angles.shape
        dev, dt = angles.device, angles.dtype
        if config is not None:
            cfg = tuple(config)
        else:
            cfg = _tuning.pinned_config(angles, angles_length)
            with torch.cuda.device(dev):
                r = cfg[1] if cfg is not None else _step_residues(
                    dt, B, L, lambda: None if torch.cuda.is_current_stream_capturing() else angles_length.cpu())
                if r is None or (cfg is None and not ext.step_fits(dt == torch.float64, B, L, [r, r])):
                    cfg = _tuning.config_for(angles, angles_length)
                    r = cfg[1]
                if ext.step_fits(dt == torch.float64, B, L, [r, r]):
                    cfg = (r, r)
        self.angles = angles
        self.angles_length = angles_length
        self.config = cfg
        self.coords = torch.zeros(B, 9 * L, dtype=dt, device=dev)
        self.grad_coords = torch.zeros(B, 9 * L, dtype=dt, device=dev)
        self.grad_angles = torch.zeros(B, 3, L, dtype=dt, device=dev)
        st_bytes, sy_bytes = ext.workspace_bytes(dt == torch.float64, B, L, list(cfg))
        self._state = _empty_bytes(max(int(st_bytes), 256), dev)
        self._sync = torch.zeros(max(int(sy_bytes), 256), dtype=torch.uint8, device=dev)
        self._step = ext.Step(angles, angles_length, self.grad_coords, self.coords,
                              self.grad_angles, self._state, self._sync, list(cfg))

    def replay(self):
        """Runs one forward+backward step on the current stream."""
        self._step.run()
