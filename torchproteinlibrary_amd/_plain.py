"""Which calls of the layers' autograd functions go to native code."""
from __future__ import annotations

import torch

_PLAIN = (torch.Tensor, torch.nn.Parameter)


def is_plain(args) -> bool:
    """Whether every argument is a plain tensor and nothing is being compiled.
    The native side looks at the rest (tracers, transforms, modes, tangents)."""
    return all(type(a) in _PLAIN for a in args) and not torch.compiler.is_compiling()
