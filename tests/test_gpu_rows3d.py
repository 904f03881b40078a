"""Workgroup rows of the 3D two-pass kernels: z sizes on either side of each
row rule (one short row, one full row, equal rows, exact 64-cell rows) with a
last workgroup that is partly outside in y, bit-identical to the split step,
whose shell and interior kernels choose their own workgroups."""
import pytest
import torch

from conftest import has_gpu
from test_gpu_tb3d import _run

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


@pytest.mark.parametrize("nz", [240, 300, 448, 15, 63, 64, 65, 80, 127, 128, 129, 192, 257, 320, 384])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
def test_two_pass_rows_equal_split_step(nz, dtype):
    case = (19, 37, nz, 4, "mask", 7)
    a, oa, _ = _run(case, dtype, 0)
    b, ob, _ = _run(case, dtype, 3)
    for f in a:
        assert torch.equal(a[f], b[f]), f
    for x, y in zip(oa, ob):
        assert torch.equal(torch.view_as_real(x) if x.is_complex() else x,
                           torch.view_as_real(y) if y.is_complex() else y)
