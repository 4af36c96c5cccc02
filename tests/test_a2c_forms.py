"""Which kernels Angles2Coords takes (AUTO), by the type, the batch and the
strides: shapes where both sides were measured, away from the lines between
them, on a GPU of 256 CUs (the number assumed where there is none)."""
import pytest

from tests import abi_a2c

FUSED, GROUPS, RUNS, TILES = 1, 2, 3, 4  # TPLX_A2C_FWD_* and TPLX_A2C_BWD_*
F32, F64 = 0, 1
NB = 8.3  # atoms to a residue of the largest structure


def _lib():
    import torch
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("measured on 256 CUs")
    return abi_a2c.load()


@pytest.mark.parametrize("dtype,B,L,names,workspace,form", [
    # one block, one workgroup per structure, several
    (F32, 4096, 64, 1, 0, FUSED), (F64, 1, 21, 1, 1, FUSED), (F32, 32, 350, 1, 1, FUSED), (F64, 256, 300, 0, 0, FUSED),
    (F32, 512, 300, 1, 1, FUSED), (F64, 400, 300, 0, 0, FUSED), (F32, 64, 600, 1, 1, FUSED), (F32, 256, 1000, 1, 1, FUSED),
    (F64, 256, 600, 1, 1, FUSED),
    # without a workspace: many structures, long ones, no names
    (F32, 1024, 300, 0, 0, RUNS), (F64, 1024, 300, 1, 0, RUNS), (F32, 256, 1000, 0, 0, RUNS), (F64, 64, 1000, 1, 0, RUNS),
    (F32, 8, 3000, 0, 0, RUNS), (F32, 8, 3000, 1, 0, RUNS), (F64, 512, 200, 1, 0, RUNS), (F32, 1024, 1000, 0, 0, RUNS),
    # with one
    (F32, 1024, 1000, 1, 1, GROUPS), (F32, 300, 600, 1, 1, GROUPS), (F64, 300, 600, 1, 1, GROUPS), (F32, 2048, 300, 1, 1, GROUPS),
    (F32, 8, 3000, 1, 1, GROUPS), (F64, 128, 1000, 1, 1, GROUPS), (F64, 200, 800, 1, 1, GROUPS), (F32, 64, 1000, 1, 1, GROUPS),
    (F32, 1024, 200, 1, 1, RUNS), (F32, 512, 450, 1, 1, RUNS), (F64, 512, 200, 1, 1, RUNS), (F64, 2000, 100, 1, 1, RUNS)])
def test_forward_form(dtype, B, L, names, workspace, form):
    assert _lib().tplx_a2c_forward_form(dtype, B, L, int(NB * L), names, workspace) == form


@pytest.mark.parametrize("dtype,B,L,workspace,form", [
    (F32, 1, 21, 0, FUSED), (F32, 1024, 128, 1, FUSED), (F32, 256, 300, 0, FUSED), (F32, 260, 450, 1, FUSED),
    (F32, 256, 1000, 1, FUSED), (F32, 1024, 200, 1, FUSED), (F32, 8, 3000, 0, FUSED), (F64, 512, 450, 1, FUSED),
    (F64, 320, 200, 0, FUSED), (F64, 256, 300, 0, FUSED), (F64, 1, 128, 0, FUSED), (F64, 1024, 30, 0, FUSED),
    (F32, 400, 300, 1, TILES), (F32, 512, 300, 0, TILES), (F32, 512, 600, 1, TILES), (F32, 1024, 300, 0, TILES),
    (F64, 256, 64, 1, RUNS), (F64, 128, 128, 0, RUNS), (F64, 64, 200, 1, RUNS), (F64, 512, 64, 0, RUNS),
    (F32, 1024, 1000, 1, GROUPS), (F32, 2048, 300, 1, GROUPS), (F64, 2048, 300, 1, GROUPS), (F32, 64, 600, 1, GROUPS),
    (F64, 8, 3000, 1, GROUPS), (F32, 700, 300, 1, GROUPS)])
def test_backward_form(dtype, B, L, workspace, form):
    assert _lib().tplx_a2c_backward_form(dtype, B, L, int(NB * L), workspace) == form


def test_short_structures_in_a_long_stride():
    lib = _lib()
    for dtype in (F32, F64):
        assert lib.tplx_a2c_forward_form(dtype, 1024, 1000, int(NB * 125), 1, 1) == RUNS
        assert lib.tplx_a2c_backward_form(dtype, 500, 800, int(NB * 100), 1) == TILES
        assert lib.tplx_a2c_backward_form(dtype, 1024, 1000, int(NB * 125), 1) == GROUPS
        assert lib.tplx_a2c_backward_form(dtype, 1024, 1000, int(NB * 125), 0) == TILES
        assert lib.tplx_a2c_backward_form(dtype, 1024, 16384, int(NB * 125), 0) == FUSED  # more than tiles take
