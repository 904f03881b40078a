"""The small tiles of grids that fit the chip in one round (variants 7-9, one
launch over interior and ring tiles) and the D-field taps of every tile
against the two-pass path, bit for bit: grids one cell below, at and above a
multiple of the tile, grids with and without interior tiles, step counts that
end inside a launch, and the smallest grids."""
import pytest
import torch

from conftest import has_gpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


def _run(mode, dtype, variant, size, k, npml):
    from meep_torch_amd.core import engine2d
    from meep_torch_amd.core.coeffs import build_te_coeffs, build_tm_coeffs
    from meep_torch_amd.core.grid import Grid
    from meep_torch_amd.core.monitors import DFTFieldsMonitor, FluxMonitorTE, FluxMonitorTM
    from meep_torch_amd.core.sources import GaussianPulse, LineSource
    from meep_torch_amd.core.stepper_te import FIELDS as TEF, init_te_state
    from meep_torch_amd.core.stepper_tm import FIELDS as TMF, init_tm_state
    nx, ny = size
    g = Grid(nx=nx, ny=ny, dx=0.05, dtype=dtype, device="cuda")
    gen = torch.Generator().manual_seed(nx * 1000 + ny)
    eps = (1.0 + 3.0 * torch.rand(nx, ny, generator=gen, dtype=torch.float64)).to(dtype).cuda()
    src = LineSource(g, ix=nx // 2, j0=1, j1=max(2, ny - 2), profile=GaussianPulse(1.0, 2.0, cutoff=1.0))
    tm = mode == "tm"
    m = (build_tm_coeffs if tm else build_te_coeffs)(g, eps_inf=eps, npml=npml)
    st, names = (init_tm_state(g), TMF) if tm else (init_te_state(g), TEF)
    if tm:
        mons = [FluxMonitorTM(g, [0.9], x_normal=True, idx=nx // 2, lo=0, hi=ny),
                DFTFieldsMonitor(g, [0.8], component="Dz"), DFTFieldsMonitor(g, [0.8], component="Ez")]
    else:
        src.mask = src.mask[:, :-1].contiguous()
        mons = [FluxMonitorTE(g, [0.9], ix=nx // 2, lo=0, hi=ny - 1),
                DFTFieldsMonitor(g, [0.8], component="Dx"), DFTFieldsMonitor(g, [0.8], component="Dy")]
    work = {f: getattr(st, f).clone() for f in names}
    for f in names:   # a running state: every field and psi cell populated where the update reaches
        if not f.startswith("psi"):
            work[f].copy_(torch.randn(work[f].shape, generator=gen, dtype=torch.float64).to(dtype) * 0.1)
    plan = engine2d.source_plan(src, work["Dz" if tm else "Dy"].shape, "cuda", dtype)
    tape = torch.zeros(k, nx, ny, dtype=dtype, device="cuda") if tm else None
    outs = engine2d.run_chunk(mode, work, m, 0, k, plan, mons, tape=tape, variant=variant)
    return [work[f] for f in names] + list(outs) + ([tape] if tm else [])


@pytest.mark.parametrize("size,npml", [((3, 3), 0), ((7, 9), 1), ((33, 31), 4), ((64, 96), 5), ((65, 97), 6),
                                       ((127, 63), 10), ((250, 241), 9)])
@pytest.mark.parametrize("variant", [2, 5, 7, 8, 9])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("mode", ["tm", "te"])
def test_small_tiles_match_two_pass(mode, dtype, variant, size, npml):
    ref = _run(mode, dtype, -1, size, 19, npml)
    got = _run(mode, dtype, variant, size, 19, npml)
    for a, b in zip(got, ref):
        assert torch.equal(a, b), float((a - b).abs().max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("sizes", [[(64, 64)], [(60, 77), (90, 41)], [(150, 140), (131, 160), (170, 120)]])
def test_one_round_batch_matches_run_tm(dtype, sizes):
    """A batch of at most one round of tiles: the common interior + ring
    launch, spectra and eps gradients equal to run_tm of each variant."""
    from meep_torch_amd import tune
    from meep_torch_amd.batch import BatchedTM
    from meep_torch_amd.core.coeffs import build_tm_coeffs
    from meep_torch_amd.core.grid import Grid
    from meep_torch_amd.core.monitors import FluxMonitorTM
    from meep_torch_amd.core.run import run_tm
    from meep_torch_amd.core.sources import GaussianPulse, LineSource
    from meep_torch_amd.core.stepper_tm import init_tm_state
    steps, K = 90, 40
    probs, single = [], []
    for nx, ny in sizes:
        g = Grid(nx=nx, ny=ny, dx=0.05, dtype=dtype, device="cuda")
        gen = torch.Generator().manual_seed(nx + ny)
        eps = (1.0 + 3.0 * torch.rand(nx, ny, generator=gen, dtype=torch.float64)).to(dtype).cuda()
        c = build_tm_coeffs(g, eps_inf=eps, npml=8)
        src = LineSource(g, ix=12, j0=10, j1=ny - 10, profile=GaussianPulse(1.0, 2.0, cutoff=1.5))
        mon = FluxMonitorTM(g, [0.8, 1.0], x_normal=True, idx=nx - 14, lo=10, hi=ny - 10)
        probs.append((c, src, [mon]))
        single.append((g, c, src, mon))
    bt = BatchedTM(probs, steps, checkpoint_every=K)
    assert bt.variant == tune.one_round(dtype, sizes)
    eps = [p[0].eps_inf.clone().requires_grad_(True) for p in probs]
    out = bt.apply(eps)
    sum(m[0].flux(o[0], 0.05).sum() for (_, _, m), o in zip(probs, out)).backward()
    for (g, c, src, mon), o, e in zip(single, out, eps):
        e1 = c.eps_inf.clone().requires_grad_(True)
        _, (acc,) = run_tm(init_tm_state(g), c._replace(eps_inf=e1), steps, source=src, monitors=[mon],
                           checkpoint_every=K)
        assert torch.equal(o[0], acc)
        mon.flux(acc, 0.05).sum().backward()
        # the reverse sweeps add the same cotangents in another order
        assert float((e.grad - e1.grad).norm()) <= (1e-5 if dtype == torch.float32 else 1e-12) * float(e1.grad.norm())
