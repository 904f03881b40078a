"""The temporally blocked reverse sweep (mt_tm2d_adjoint_tiled) against the
per-step passes (mt_tm2d_adjoint), bit for bit: every cotangent, eps gradient,
x and y lines, whole-field and D monitors, probes, odd and even launch counts,
staging blocks shorter than the sweep, one- and two-step sweeps, tiles of
every shape on grids below, at and above a multiple of the tile, in the common
launch of a one-round grid and in the interior and ring launches of a larger one."""
import ctypes

import pytest
import torch

from conftest import has_gpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


def _sweeps(dtype, size, npml, k, variant, S, y_pmc=False):
    from meep_torch_amd import _engine as E
    from meep_torch_amd.core import adjoint2d, engine2d
    from meep_torch_amd.core.coeffs import build_tm_coeffs
    from meep_torch_amd.core.grid import Grid
    from meep_torch_amd.core.monitors import DFTFieldsMonitor, FluxMonitorTM, PointProbe
    from meep_torch_amd.core.stepper_tm import FIELDS, init_tm_state
    nx, ny = size
    g = Grid(nx=nx, ny=ny, dx=0.05, dtype=dtype, device="cuda")
    gen = torch.Generator().manual_seed(nx * 100 + ny + k)
    rnd = lambda *s: torch.randn(*s, generator=gen, dtype=torch.float64).to(dtype).cuda()
    c = build_tm_coeffs(g, eps_inf=2.0 + rnd(nx, ny).abs(), npml=(npml, 0) if y_pmc else npml, y_pmc=y_pmc)
    st = init_tm_state(g, y_pmc=y_pmc)
    mons = [FluxMonitorTM(g, [0.8, 1.0, 1.1], x_normal=True, idx=nx // 2, lo=1, hi=ny - 1),
            FluxMonitorTM(g, [0.9], x_normal=False, idx=ny // 2, lo=0, hi=nx),
            DFTFieldsMonitor(g, [0.7], component="Dz"), DFTFieldsMonitor(g, [0.7, 0.9], component="Hy"),
            PointProbe(nx // 2, ny // 3)]
    zero = {f: torch.zeros_like(getattr(st, f)) for f in FIELDS}
    gacc = []
    for m in mons:
        kind, terms = m.engine_terms(zero)
        gacc.append(rnd(k) if kind == "probe" else rnd(*m.out_shape(zero)))
    tape = rnd(k, nx, ny)
    init = {f: rnd(*t.shape) if not f.startswith("psi") else torch.zeros_like(t) for f, t in zero.items()}
    L, out = E.lib(), []
    for tiled in (False, True):
        A = {f: t.clone() for f, t in init.items()}
        B = {f: t.clone() for f, t in init.items()}
        eg = torch.zeros(nx, ny, dtype=dtype, device="cuda")
        sc = [torch.empty(nx, ny, dtype=dtype, device="cuda") for _ in range(4)]
        a, b = E.TM2DAdj(), E.TM2DAdj()
        for f in FIELDS:
            setattr(a, "a" + f, A[f].data_ptr())
            setattr(b, "a" + f, B[f].data_ptr())
        for f, t in zip(("gHy", "gHx", "gEx", "gEy"), sc):
            setattr(a, f, t.data_ptr())
        a.eps_grad = eg.data_ptr()
        d, keep = adjoint2d._descriptor(c, A, dtype, "cuda")
        arr, n, kp = adjoint2d._adj_monitors(A, mons, gacc, dtype, "cuda")
        if tiled:
            d.variant = variant
            nb = L.mt_stage_bytes(arr, n, S, E.dtype_code(dtype))
            stage = torch.empty(nb, dtype=torch.uint8, device="cuda")
            rc = L.mt_tm2d_adjoint_tiled(ctypes.byref(d), ctypes.byref(a), ctypes.byref(b), E.ptr(tape), arr, n,
                                         E.ptr(stage), nb, S, 5, k, E.stream_handle())
        else:
            rc = L.mt_tm2d_adjoint(ctypes.byref(d), ctypes.byref(a), E.ptr(tape), arr, n, 5, k, E.stream_handle())
        E.check(rc, "adjoint")
        torch.cuda.synchronize()
        del keep, kp
        out.append({**A, "eps_grad": eg})
    return out


@pytest.mark.parametrize("size,npml,k,S", [((5, 7), 1, 1, 4), ((33, 31), 4, 2, 64), ((64, 96), 6, 19, 7),
                                           ((130, 71), 8, 30, 64), ((210, 190), 7, 9, 3), ((530, 1060), 20, 6, 4)])
@pytest.mark.parametrize("variant", [2, 5, 7, 8, 9])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_tiled_reverse_matches_per_step_passes(dtype, variant, size, npml, k, S):
    ref, got = _sweeps(dtype, size, npml, k, variant, S)
    assert float(ref["eps_grad"].abs().max()) > 0
    for f in ref:
        assert torch.equal(got[f], ref[f]), (f, float((got[f] - ref[f]).abs().max()))


def test_tiled_reverse_y_pmc():
    ref, got = _sweeps(torch.float32, (61, 47), 6, 12, 7, 64, y_pmc=True)
    for f in ref:
        assert torch.equal(got[f], ref[f]), f
