"""The joined passes of the 3D reverse sweep at their edges: calls of one step
(a first and a last pass only), a few and all steps, grids whose shells almost
meet, that have no shell on one side of the workgroup's rows and that end
inside a workgroup, eps varying inside the shells too, and two monitors that
add to E and H cells; FP64 against CPU autograd through the oracle's steps."""
import pytest
import torch

from conftest import has_gpu
from test_gpu_adjoint3d import _rel

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


def _loss(accs):
    return (accs[0][0, 0] ** 2 + accs[0][0, 1] ** 2).sum() + (accs[1][0, 0] ** 2 + 2 * accs[1][0, 1] ** 2).sum()


@pytest.mark.parametrize("shape,npml", [((13, 11, 9), 3), ((8, 9, 70), 2), ((9, 17, 33), 3)])
def test_gradient_at_chunk_and_grid_edges(shape, npml):
    from meep_torch_amd.core.adjoint3d import run_3d_adjoint
    from meep_torch_amd.core.monitors_3d import DFTFieldsMonitor3D, PointSource3D
    from meep_torch_amd.core.sources import GaussianPulse
    from meep_torch_amd.core.stepper_3d import build_3d_coeffs, init_3d_state
    from oracle import yee3d
    nx, ny, nz = shape
    steps, p = 21, nx - npml - 2
    eps0 = 1.0 + 2.0 * torch.rand(shape, generator=torch.Generator().manual_seed(nz), dtype=torch.float64)
    prof = GaussianPulse(0.6, 0.6)
    e = eps0.clone().requires_grad_(True)
    oc = yee3d.coeffs3d(nx, ny, nz, 0.05, e, npml, torch.float64)
    amps = [prof.amplitude((t + 0.5) * oc["dt"]) for t in range(steps)]
    _, oacc = yee3d.run3d(yee3d.state3d(nx, ny, nz, torch.float64), oc, steps, amps, ("Ez", nx // 2, ny // 2, nz // 2),
                          [{"type": "dft", "comp": c, "plane": (0, p), "freq": 0.6} for c in ("Ez", "Hy")])
    want, = torch.autograd.grad(_loss(oacc), e)
    assert float(want.abs().max()) > 0
    for chunk in (1, 5, steps):
        eps = eps0.clone().cuda().requires_grad_(True)
        c = build_3d_coeffs(nx, ny, nz, 0.05, eps=eps, npml=npml, dtype=torch.float64, device="cuda")
        src = PointSource3D(c.dt, "Ez", nx // 2, ny // 2, nz // 2, prof)
        mons = [DFTFieldsMonitor3D(c.dt, [0.6], q, plane=(0, p), dtype=torch.float64) for q in ("Ez", "Hy")]
        st0 = init_3d_state(nx, ny, nz, npml=npml, dtype=torch.float64, device="cuda")
        run_3d_adjoint(c, steps, chunk, src, mons, _loss, st0)
        # FP64 through 21 steps forward and back of a few dozen roundings each
        assert _rel(eps.grad.cpu(), want) <= 1e-12, chunk
