"""TM gradients with monitors that the reverse tiles do not take (averages of
whole fields, terms without a field position) run step by step: equal to a run
in which the step-by-step sweep is forced."""
import pytest
import torch

from conftest import has_gpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


def _case(dtype, which):
    from meep_torch_amd.core.coeffs import build_tm_coeffs
    from meep_torch_amd.core.grid import Grid
    from meep_torch_amd.core.monitors import DFTFieldsMonitor, FluxMonitorTM
    from meep_torch_amd.core.sources import GaussianPulse, LineSource
    from meep_torch_amd.core.stepper_tm import init_tm_state
    nx, ny = 60, 44
    g = Grid(nx=nx, ny=ny, dx=0.05, dtype=dtype, device="cuda")
    gen = torch.Generator().manual_seed(7)
    eps = (1.0 + 3.0 * torch.rand(nx, ny, generator=gen, dtype=torch.float64)).to(dtype).cuda()
    src = LineSource(g, ix=nx // 2, j0=4, j1=ny - 5, profile=GaussianPulse(1.0, 2.0, cutoff=1.0))

    class MeanOfFields(DFTFieldsMonitor):   # a whole-field average
        def engine_terms(self, f):
            kind, ((a, _, half, sem),) = super().engine_terms(f)
            return kind, [(a, f["Dz"].reshape(1, -1), half, sem)]

    class Unplaced(DFTFieldsMonitor):
        def engine_terms(self, f):
            kind, (t,) = super().engine_terms(f)
            return kind, [t[:3]]

    line = FluxMonitorTM(g, [0.8, 0.9], x_normal=True, idx=14, lo=3, hi=ny - 3)
    mons = [line, (MeanOfFields if which == "mean" else Unplaced)(g, [0.7], component="Ez")]
    return build_tm_coeffs(g, eps_inf=eps, npml=5), src, init_tm_state(g), mons


def _grad(c, src, st, mons, ck):
    from meep_torch_amd.core.run import run_tm
    e = c.eps_inf.clone().requires_grad_(True)
    _, acc = run_tm(st, c._replace(eps_inf=e), 30, source=src, monitors=mons, checkpoint_every=ck)
    sum((a ** 2).sum() for a in acc).backward()
    return e.grad


@pytest.mark.parametrize("which", ["mean", "unplaced"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_gradient_steps_back_where_tiles_refuse(dtype, which, monkeypatch):
    from meep_torch_amd import _engine as E
    case = _case(dtype, which)
    monkeypatch.setenv("MEEP_TORCH_AMD_VARIANT", "-1")   # forward runs take these monitors in two passes
    got = _grad(*case, 12)
    assert float(got.abs().max()) > 0
    monkeypatch.setattr(E.lib(), "mt_tm2d_adjoint_tiles_ok", lambda *a: 0, raising=False)
    assert torch.equal(got, _grad(*case, 12))
