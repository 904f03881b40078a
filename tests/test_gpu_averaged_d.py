"""Monitors that sample D averaged over two rows or columns, on tile edges
and inside tiles: the tiled steppers against the two-pass path bit for bit,
the batched runner (which has no other path) against single runs, and eps
gradients of the tiled reverse sweep against the per-step passes."""
import pytest
import torch

from conftest import has_gpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


def _monitors(mode, g, xs, ys):
    """Flux lines whose magnetic term is replaced by averaged D."""
    from meep_torch_amd.core.monitors import FluxMonitorTE, FluxMonitorTEY, FluxMonitorTM

    class TMX(FluxMonitorTM):
        def engine_terms(self, f):
            kind, (e, h) = super().engine_terms(f)
            i, lo, hi = self.idx, self.lo, self.hi
            a, b = (f["Dz"][i - 1, lo:hi], f["Dz"][i, lo:hi]) if self.x_normal else (f["Dz"][lo:hi, i - 1],
                                                                                    f["Dz"][lo:hi, i])
            return kind, [e, (a, b, 0, (3,) + h[3][1:])]

    class TEX(FluxMonitorTE):
        def engine_terms(self, f):
            kind, (e, h) = super().engine_terms(f)
            i, lo, hi = self.ix, self.lo, self.hi
            return kind, [e, (f["Dy"][i - 1, lo:hi], f["Dy"][i, lo:hi], 0, (4,) + h[3][1:])]

    class TEY(FluxMonitorTEY):
        def engine_terms(self, f):
            kind, (e, h) = super().engine_terms(f)
            j, lo, hi = self.iy, self.lo, self.hi
            return kind, [e, (f["Dx"][lo:hi, j - 1], f["Dx"][lo:hi, j], 0, (3,) + h[3][1:])]

    nx, ny = g.nx, g.ny
    if mode == "tm":
        return [TMX(g, [0.8, 0.9], x_normal=True, idx=i, lo=1, hi=ny - 2) for i in xs] + \
               [TMX(g, [0.8], x_normal=False, idx=j, lo=0, hi=nx) for j in ys]
    return [TEX(g, [0.8], ix=i, lo=1, hi=ny - 2) for i in xs] + [TEY(g, [0.9], iy=j, lo=0, hi=nx - 1) for j in ys]


def _setup(mode, dtype, nx, ny):
    from meep_torch_amd.core.coeffs import build_te_coeffs, build_tm_coeffs
    from meep_torch_amd.core.grid import Grid
    from meep_torch_amd.core.sources import GaussianPulse, LineSource
    from meep_torch_amd.core.stepper_te import init_te_state
    from meep_torch_amd.core.stepper_tm import init_tm_state
    g = Grid(nx=nx, ny=ny, dx=0.05, dtype=dtype, device="cuda")
    gen = torch.Generator().manual_seed(nx + ny)
    eps = (1.0 + 3.0 * torch.rand(nx, ny, generator=gen, dtype=torch.float64)).to(dtype).cuda()
    src = LineSource(g, ix=nx // 2, j0=4, j1=ny - 5, profile=GaussianPulse(1.0, 2.0, cutoff=1.0))
    if mode == "te":
        src.mask = src.mask[:, :-1].contiguous()
    c = (build_tm_coeffs if mode == "tm" else build_te_coeffs)(g, eps_inf=eps, npml=5)
    return g, c, src, (init_tm_state if mode == "tm" else init_te_state)(g), _monitors(mode, g, (16, 33, 40),
                                                                                      (16, 63, 64))


@pytest.mark.parametrize("variant", [2, 5, 7, 8, 9])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("mode", ["tm", "te"])
def test_tiles_match_two_pass(mode, dtype, variant, monkeypatch):
    from meep_torch_amd.core.run import run_te, run_tm
    g, c, src, st, mons = _setup(mode, dtype, 70, 90)
    out = []
    for v in (-1, variant):
        monkeypatch.setenv("MEEP_TORCH_AMD_VARIANT", str(v))
        out.append((run_tm if mode == "tm" else run_te)(st, c, 45, source=src, monitors=mons))
    assert all(float(a.abs().max()) > 0 for a in out[0][1])
    for a, b in zip([*out[0][0], *out[0][1]], [*out[1][0], *out[1][1]]):
        if torch.is_tensor(a):
            assert torch.equal(a, b)


def test_batch_and_gradient_match_single_runs(monkeypatch):
    from meep_torch_amd.batch import BatchedTM
    from meep_torch_amd.core.run import run_tm
    setups = [_setup("tm", torch.float64, nx, 90) for nx in (70, 61)]
    grads, accs = [], []
    for kw in (dict(), dict(fused_adjoint=False)):
        bt = BatchedTM([(c, src, mons) for _, c, src, _, mons in setups], 45, checkpoint_every=20, **kw)
        eps = [s[1].eps_inf.clone().requires_grad_(True) for s in setups]
        out = bt.apply(eps)
        sum((a ** 2).sum() for o in out for a in o).backward()
        assert bt._adj["fused"] == (not kw)
        grads.append([e.grad for e in eps])
        accs.append([a.detach() for o in out for a in o])
    for a, b in zip(*grads):
        assert float(a.abs().max()) > 0 and torch.equal(a, b)
    i = 0
    for (g, c, src, st, mons), want in zip(setups, grads[0]):
        e = c.eps_inf.clone().requires_grad_(True)
        _, acc = run_tm(st, c._replace(eps_inf=e), 45, source=src, monitors=mons, checkpoint_every=20)
        sum((a ** 2).sum() for a in acc).backward()
        for a in acc:
            assert torch.equal(a.detach(), accs[0][i])
            i += 1
        # the sweeps add the same cotangents in another order
        assert float((e.grad - want).norm()) <= 1e-12 * float(want.norm())
