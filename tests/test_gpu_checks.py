"""The layers' output checks: a call raises exactly where the sum of its
outputs is NaN, wherever the values lie, and reports bad counts."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
INF, NAN = float("inf"), float("nan")

# values put into a zero input: into structure 1, or one into each structure
VALUES = [(NAN,), (INF,), (INF, -INF), (3e37, 3e37), (1e25,)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("atoms", [3, 256, 1021])
@pytest.mark.parametrize("values", VALUES)
def test_transforms_raise_where_the_output_sum_is_nan(dtype, atoms, values):
    from torchproteinlibrary_amd.FullAtomModel.CoordsTransform import Coords2Center, CoordsRotate, CoordsTranslate
    n = torch.tensor([atoms, max(atoms - 2, 1)], dtype=torch.int32, device=DEV)
    T = torch.zeros(2, 3, dtype=dtype, device=DEV)
    R = torch.eye(3, dtype=dtype, device=DEV).repeat(2, 1, 1)

    for first in (0, 3 * (int(n[1]) - 1)):  # the first and the last atom of structure 1
        x = torch.zeros(2, 3 * atoms, dtype=dtype, device=DEV)
        for k, v in enumerate(values):
            x[k if len(values) > 1 else 1, first if k == 0 else 0] = v
        for f, out in ((lambda: CoordsTranslate()(x, T, n), lambda: x.sum()),
                       (lambda: CoordsRotate()(x, R, n), lambda: (x.view(2, -1, 3) @ R.transpose(1, 2)).sum()),
                       (lambda: Coords2Center()(x, n), lambda: (x.view(2, -1, 3).sum(1) / n[:, None]).sum())):
            if torch.isnan(out()):
                with pytest.raises(Exception, match="Nan"):
                    f()
            else:
                f()
    # past num_atoms nothing counts
    if atoms > 3:
        x = torch.zeros(2, 3 * atoms, dtype=dtype, device=DEV)
        x[1, 3 * (atoms - 2):] = values[0]
        CoordsTranslate()(x, T, n), CoordsRotate()(x, R, n), Coords2Center()(x, n)


def test_transforms_report_counts_and_empty_structures():
    from torchproteinlibrary_amd.FullAtomModel.CoordsTransform import Coords2Center, CoordsRotate
    x = torch.zeros(2, 30, device=DEV)
    R = torch.eye(3, device=DEV).repeat(2, 1, 1)
    for bad in (11, -1):
        with pytest.raises(ValueError, match="num_atoms outside"):
            CoordsRotate()(x, R, torch.tensor([10, bad], dtype=torch.int32, device=DEV))
    with pytest.raises(Exception, match="Coords2CenterFunction: forward Nan"):
        Coords2Center()(x, torch.tensor([10, 0], dtype=torch.int32, device=DEV))
    y = torch.ones(2, 30, device=DEV, requires_grad=True)
    out = CoordsRotate()(y, R, torch.tensor([10, 4], dtype=torch.int32, device=DEV))
    with pytest.raises(Exception, match="CoordsRotateFunction: backward Nan"):
        out.backward(torch.full_like(out, NAN))
