"""Performance cases: the work that users have this framework do, through its
public entry points (the operators of meep_torch_amd.core, the batched runner
and the surrogate network).

Each case names a kind and its sizes.  `prepare` builds what a program holds
before the call, `run` makes one pass, `exact` gives the same outputs in
float64 from plain torch.  Grid steps are dx = 0.05 or 0.04 throughout, as in
the repository's configurations.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "meep-torch_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

F32, F64 = torch.float32, torch.float64


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # A small 2D cell in double precision: the first runs of a study, a
        # parameter sweep of short simulations.  Launches and host time count.
        dict(name="tm_cell", kind="tm", nx=100, ny=60, dx=0.05, npml=10, steps=400, nfreq=3, fp64=True,
             media=False, resume=False),
        # The repository's first configuration: waveguide, 2000 steps, a
        # 50-frequency flux line.
        dict(name="tm_guide", kind="tm", nx=256, ny=256, dx=0.05, npml=16, steps=2000, nfreq=50, fp64=False,
             media=False, resume=False),
        # Dispersive, Kerr and lossy media on a ragged 2D grid (nonlinear and
        # metal structures).
        dict(name="tm_media", kind="tm", nx=509, ny=387, dx=0.05, npml=20, steps=300, nfreq=20, fp64=False,
             media=True, resume=True),
        # One gradient of a 2D design (forward, checkpoints, reverse sweep):
        # the geometry of the surrogate's design problem.
        dict(name="tm_design", kind="tm_grad", nx=256, ny=256, dx=0.05, npml=24, steps=1000, nfreq=50, ck=250,
             fp64=False),
        # Many design variants of uneven size advanced and differentiated
        # together in captured graphs, as a batched design loop does.
        dict(name="tm_batch", kind="batch", n_var=10, lo=200, hi=900, dx=0.05, npml=24, steps=400, nfreq=20, ck=100,
             fp64=False),
        # A large 2D TE plate with four spectral lines, going on from a saved
        # state: a slice of the second configuration's 10000 steps.
        dict(name="te_plate", kind="te", nx=2048, ny=2048, dx=0.05, npml=32, steps=400, nfreq=100, fp64=False,
             resume=True),
        # TE gradient in double precision on a ragged grid.
        dict(name="te_design", kind="te_grad", nx=331, ny=277, dx=0.05, npml=16, steps=300, nfreq=20, ck=100,
             fp64=True),
        # The repository's headline 3D run: 384^3, two 64-frequency flux
        # planes, going on from a saved state.
        dict(name="yee3d_slab", kind="yee3d", nx=384, ny=384, nz=384, dx=0.05, npml=12, steps=40, nfreq=64,
             fp64=False, media=False, resume=True),
        # A ragged 3D cell with a Lorentz and a Drude pole and conductivity.
        dict(name="yee3d_media", kind="yee3d", nx=141, ny=127, nz=109, dx=0.05, npml=10, steps=100, nfreq=16,
             fp64=False, media=True, resume=True),
        # One gradient of a 3D design through checkpoints and recompute.
        dict(name="yee3d_design", kind="yee3d_grad", nx=96, ny=88, nz=80, dx=0.05, npml=10, steps=240, nfreq=8,
             ck=60, fp64=False),
        # Forward and parameter gradients of one training batch of the
        # surrogate network at its default size.
        dict(name="net_train", kind="net_train", n=128, batch=64),
        # One surrogate step of the design loop: spectrum of one density and
        # the gradient of its mean.
        dict(name="net_design", kind="net_design", n=128, batch=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any kind, sizes spread over the range between the
    smallest and the largest call of that kind."""
    kind = rng.choice(["tm", "tm", "tm_grad", "batch", "te", "te_grad", "yee3d", "yee3d", "yee3d_grad",
                       "net_train", "net_design"])
    dx = rng.choice([0.05, 0.05, 0.04])
    fp64 = rng.random() < 0.25
    media = rng.random() < 0.35
    if kind in ("tm", "te"):
        nx, ny = _log_int(rng, 60, 1600), _log_int(rng, 60, 1600)
        steps = max(40, min(1500, int(4e8 / (nx * ny))))
        c = dict(kind=kind, nx=nx, ny=ny, dx=dx, npml=rng.randint(6, 24), steps=steps, nfreq=rng.randint(1, 100),
                 fp64=fp64, resume=nx * ny > 150 * 150 or rng.random() < 0.5)
        if kind == "tm":
            c["media"] = media
            if media:
                c["steps"] = min(400, steps)
        return c
    if kind in ("tm_grad", "te_grad"):
        nx, ny = _log_int(rng, 140, 500), _log_int(rng, 140, 500)
        return dict(kind=kind, nx=nx, ny=ny, dx=dx, npml=rng.randint(8, 24), steps=rng.randint(300, 500),
                    nfreq=rng.randint(1, 50), ck=rng.choice([60, 100, 200]), fp64=fp64)
    if kind == "batch":
        lo = rng.randint(150, 300)
        return dict(kind=kind, n_var=rng.randint(2, 10), lo=lo, hi=lo + rng.randint(50, 500), dx=dx,
                    npml=rng.randint(12, 24), steps=rng.randint(300, 400), nfreq=rng.randint(2, 20),
                    ck=rng.choice([50, 100]), fp64=False)
    if kind == "yee3d":
        nx, ny, nz = (_log_int(rng, 40, 300) for _ in range(3))
        cost = nx * ny * nz * (2 if fp64 else 1) * (3 if media else 1)
        steps = max(12, min(200, int(1.2e9 / cost)))
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, dx=dx, npml=rng.randint(5, 12), steps=steps,
                    nfreq=rng.randint(1, 64), fp64=fp64, media=media, resume=True)
    if kind == "yee3d_grad":
        nx, ny, nz = (rng.randint(64, 110) for _ in range(3))
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, dx=dx, npml=rng.randint(5, 10), steps=rng.randint(200, 240),
                    nfreq=rng.randint(1, 8), ck=rng.choice([30, 60]), fp64=False)
    if kind == "net_train":
        return dict(kind=kind, n=rng.choice([64, 75, 96, 100, 128]), batch=rng.randint(2, 64))
    return dict(kind="net_design", n=rng.choice([64, 75, 96, 100, 128]), batch=rng.randint(1, 8))


# ----------------------------------------------------------------- shared inputs
def _dtype(case):
    return F64 if case["fp64"] else F32


def _gen(seed):
    return np.random.default_rng(int(seed) + 12345)


def _smooth(g, shape, dtype, waves=3, lo=10.0, hi=60.0):
    """A smooth field: a sum of separable waves of `lo`..`hi` cells with
    random phases, of about unit size (what a run holds mid-way)."""
    out = torch.zeros(shape, dtype=dtype, device="cuda")
    for _ in range(waves):
        term = torch.full((1,) * len(shape), float(g.normal()), dtype=F64, device="cuda")
        for a, n in enumerate(shape):
            v = np.cos(2 * math.pi * np.arange(n) / g.uniform(lo, hi) + g.uniform(0, 2 * math.pi))
            sh = [1] * len(shape)
            sh[a] = n
            term = term * torch.tensor(v, dtype=F64, device="cuda").reshape(sh)
        out += term.to(dtype)
    return out


def _freqs(case, fcen):
    n = case["nfreq"]
    return [fcen] if n == 1 else [fcen * (0.85 + 0.3 * i / (n - 1)) for i in range(n)]


def _pulse(case, dt, frac=0.3, cutoff=2.5):
    """(fcen, fwidth, cutoff) of a pulse that peaks after `frac` of the run,
    with a wavelength of at least ten cells."""
    t0 = frac * case["steps"] * dt
    fw = cutoff / t0
    return min(max(0.5, fw), 0.1 / case["dx"]), fw, cutoff


def _guide_eps(case, g, dtype):
    """eps of about 2.1 with a guide of eps 12.1 along x and a random smooth
    design block in the middle."""
    nx, ny = case["nx"], case["ny"]
    e = 2.1 + 0.2 * torch.sigmoid(_smooth(g, (nx, ny), dtype))
    w = max(2, ny // 26)
    e[:, ny // 2 - w // 2:ny // 2 + (w + 1) // 2] = 12.1
    a, b = nx // 3, ny // 3
    r = torch.sigmoid(4 * _smooth(g, (nx - 2 * a, ny - 2 * b), dtype, lo=6.0, hi=30.0))
    e[a:nx - a, b:ny - b] = 2.1 + 10.0 * r
    return e


def _media2d(case, g, dtype):
    nx, ny = case["nx"], case["ny"]
    blob = lambda: torch.sigmoid(6 * _smooth(g, (nx, ny), dtype, lo=30.0, hi=120.0))
    return dict(poles=[(0.6, 0.02, 0.8), (1e-10, 0.05, 1.0, 0.3)], masks=[blob(), blob()], chi3=0.02 * blob(),
                sigma_d=0.2 * blob())


def _media3d(case, g, dtype):
    sh = (case["nx"], case["ny"], case["nz"])
    blob = lambda: torch.sigmoid(6 * _smooth(g, sh, dtype, lo=30.0, hi=120.0))
    return dict(poles=[(0.6, 0.02, 0.8), (1e-10, 0.05, 1.0, 0.3)], masks=[blob(), blob()], sigma_d=0.2 * blob())


def _lines(case):
    """x lines and y lines of the flux monitors, and their extent."""
    p, nx, ny = case["npml"], case["nx"], case["ny"]
    return [p + (nx - 2 * p) // 3, nx - p - 4], [p + (ny - 2 * p) // 3, ny - p - 4], p, min(nx, ny) - p


def _inputs2d(case, seed):
    """eps, source line, pulse, frequencies, media and (for a resumed run) the
    saved fields, the same for `prepare` and `exact`."""
    g, dtype = _gen(seed), _dtype(case)
    nx, ny, p = case["nx"], case["ny"], case["npml"]
    I = {"eps": _guide_eps(case, g, dtype)}
    dt = 0.5 * case["dx"]
    grad = case["kind"].endswith("_grad")
    I["pulse"] = _pulse(case, dt, *((0.2, 2.0) if grad else ()))
    I["freqs"] = _freqs(case, I["pulse"][0])
    I["src"] = (p + 3, max(p, ny // 2 - ny // 6), min(ny - p, ny // 2 + ny // 6) - 1)
    if case.get("media"):
        I["media"] = _media2d(case, g, dtype)
    if case.get("resume"):
        tm = case["kind"] == "tm"
        shapes = {"Ez": (nx, ny), "Hx": (nx, ny - 1), "Hy": (nx - 1, ny)} if tm else {
            "Ex": (nx - 1, ny), "Ey": (nx, ny - 1), "Hz": (nx - 1, ny - 1)}
        I["fields"] = {k: 0.3 * _smooth(g, s, dtype) for k, s in shapes.items()}
        if tm:
            I["fields"]["Dz"] = I["fields"]["Ez"] * I["eps"]
        else:
            e = I["eps"]
            I["fields"]["Dx"] = I["fields"]["Ex"] * (0.5 * (e[:-1] + e[1:]))
            I["fields"]["Dy"] = I["fields"]["Ey"] * (0.5 * (e[:, :-1] + e[:, 1:]))
    return I


def _batch_cases(case, seed):
    """The single-problem cases of a batch (square grids, uneven sizes over
    the range, not in order)."""
    out = []
    for v in range(case["n_var"]):
        n = int(case["lo"] + (case["hi"] - case["lo"]) * ((v + 1) * 0.6180339887 % 1.0))
        out.append((dict(kind="tm_grad", nx=n, ny=n, dx=case["dx"], npml=case["npml"], steps=case["steps"],
                         nfreq=case["nfreq"], ck=case["ck"], fp64=case["fp64"]), seed + 1000 * (v + 1)))
    return out


def _grad_line(case):
    """x position and extent of the output line of a gradient case: near
    enough that the pulse crosses it within the run."""
    p, nx, ny = case["npml"], case["nx"], case["ny"]
    reach = int(0.5 * case["steps"] * 0.5 / 1.6)
    return min(nx - p - 4, p + 3 + max(8, reach // 2)), p, ny - p


def _inputs3d(case, seed):
    g, dtype = _gen(seed), _dtype(case)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    e = torch.full((nx, ny, nz), 1.0, dtype=dtype, device="cuda")
    z0, w = nz // 2 - max(2, nz // 34), max(3, ny // 15)
    e[:, :, :z0] = 2.1
    e[:, ny // 2 - w:ny // 2 + w, z0:z0 + max(3, nz // 17)] = 12.1
    b = (nx // 4, nx - nx // 4)
    r = torch.sigmoid(4 * _smooth(g, (b[1] - b[0], ny, nz), dtype, lo=8.0, hi=40.0))
    e[b[0]:b[1]] += 0.5 * r
    I = {"eps": e}
    dt = 0.5 * case["dx"] / math.sqrt(3.0)
    I["pulse"] = _pulse(case, dt, 0.25, 2.0)
    I["freqs"] = _freqs(case, I["pulse"][0])
    I["src"] = ("Ez", case["npml"] + 4, ny // 2, nz // 2)
    if case.get("media"):
        I["media"] = _media3d(case, g, dtype)
    if case.get("resume"):
        sh = {"Ex": (nx - 1, ny, nz), "Ey": (nx, ny - 1, nz), "Ez": (nx, ny, nz - 1),
              "Hx": (nx, ny - 1, nz - 1), "Hy": (nx - 1, ny, nz - 1), "Hz": (nx - 1, ny - 1, nz)}
        I["fields"] = {k: 0.3 * _smooth(g, s, dtype, waves=2) for k, s in sh.items()}
    return I


def _planes3d(case):
    p, nx = case["npml"], case["nx"]
    if case["kind"] == "yee3d_grad":
        return [min(nx - p - 3, p + 4 + 12)]
    return [p + (nx - 2 * p) // 4, nx - p - 3]


_NET = dict(width=64, modes=(16, 8), layers=4, n_out=50, head=128, in_ch=3)


def _inputs_net(case, seed):
    """Weights as a trained network holds them (flat, in the order of the
    network's specification), smooth densities in [0, 1] and targets."""
    g = _gen(seed)
    C, Mo, H, L = _NET["width"], _NET["modes"][0] * _NET["modes"][1], _NET["head"], _NET["layers"]
    spec = [("lift_w", (C, 3), 3), ("lift_b", (C,), 3)]
    for l in range(L):
        spec += [(f"s{l}_re", (C, C, Mo), None), (f"s{l}_im", (C, C, Mo), None), (f"w{l}", (C, C), C),
                 (f"b{l}", (C,), C)]
    spec += [("q_w", (H, C), C), ("q_b", (H,), C), ("o_w", (50, H), H), ("o_b", (50,), H)]
    tg = torch.Generator(device="cuda").manual_seed(int(seed) + 5)
    p = {}
    for name, sh, fan in spec:
        if fan is None:
            p[name] = 0.01 * torch.randn(sh, generator=tg, device="cuda")
        else:
            p[name] = (2 * torch.rand(sh, generator=tg, device="cuda") - 1) * math.sqrt(3.0 / fan)
    n, B = case["n"], case["batch"]
    rho = torch.stack([torch.sigmoid(3 * _smooth(g, (n, n), F32, lo=8.0, hi=50.0)) for _ in range(B)])
    T = torch.rand(B, 50, generator=tg, device="cuda")
    return {"spec": spec, "p": p, "rho": rho, "T": T}


# ---------------------------------------------------------------------- prepare
def _tm_problem(case, seed):
    from meep_torch_amd.core.coeffs import build_tm_coeffs
    from meep_torch_amd.core.grid import Grid
    from meep_torch_amd.core.monitors import FluxMonitorTM
    from meep_torch_amd.core.sources import GaussianPulse, LineSource
    from meep_torch_amd.core.stepper_tm import init_tm_state
    I, dtype = _inputs2d(case, seed), _dtype(case)
    grid = Grid(nx=case["nx"], ny=case["ny"], dx=case["dx"], dtype=dtype, device="cuda")
    kw = {}
    if "media" in I:
        m = I["media"]
        kw = dict(poles=m["poles"], pole_masks=m["masks"], chi3=m["chi3"], sigma_d=m["sigma_d"])
    co = build_tm_coeffs(grid, eps_inf=I["eps"], npml=case["npml"], **kw)
    fc, fw, cut = I["pulse"]
    ix, j0, j1 = I["src"]
    src = LineSource(grid, ix=ix, j0=j0, j1=j1, profile=GaussianPulse(fc, fw, cutoff=cut))
    if case["kind"] == "tm_grad":
        ix, lo, hi = _grad_line(case)
        mons = [FluxMonitorTM(grid, I["freqs"], x_normal=True, idx=ix, lo=lo, hi=hi)]
    else:
        lx, ly, lo, hi = _lines(case)
        mons = [FluxMonitorTM(grid, I["freqs"], x_normal=True, idx=lx[1], lo=lo, hi=case["ny"] - lo)]
        if case.get("media"):
            mons.append(FluxMonitorTM(grid, I["freqs"], x_normal=False, idx=ly[0], lo=lo, hi=hi))
    st = init_tm_state(grid, n_poles=len(kw.get("poles", ())))
    if "fields" in I:
        st = st._replace(**I["fields"])
    return dict(case=case, grid=grid, coeffs=co, source=src, monitors=mons, state=st, eps=I["eps"])


def _te_problem(case, seed):
    from meep_torch_amd.core.coeffs import build_te_coeffs
    from meep_torch_amd.core.grid import Grid
    from meep_torch_amd.core.monitors import FluxMonitorTE, FluxMonitorTEY
    from meep_torch_amd.core.sources import GaussianPulse, LineSource
    from meep_torch_amd.core.stepper_te import init_te_state
    I, dtype = _inputs2d(case, seed), _dtype(case)
    grid = Grid(nx=case["nx"], ny=case["ny"], dx=case["dx"], dtype=dtype, device="cuda")
    co = build_te_coeffs(grid, eps_inf=I["eps"], npml=case["npml"])
    fc, fw, cut = I["pulse"]
    ix, j0, j1 = I["src"]
    src = LineSource(grid, ix=ix, j0=j0, j1=j1, profile=GaussianPulse(fc, fw, cutoff=cut))
    src.mask = src.mask[:, :-1].contiguous()
    if case["kind"] == "te_grad":
        ix, lo, hi = _grad_line(case)
        mons = [FluxMonitorTE(grid, I["freqs"], ix=ix, lo=lo, hi=hi)]
    else:
        lx, ly, lo, hi = _lines(case)
        mons = [FluxMonitorTE(grid, I["freqs"], ix=i, lo=lo, hi=hi) for i in lx]
        mons += [FluxMonitorTEY(grid, I["freqs"], iy=j, lo=lo, hi=hi) for j in ly]
    st = init_te_state(grid)
    if "fields" in I:
        st = st._replace(**I["fields"])
    return dict(case=case, grid=grid, coeffs=co, source=src, monitors=mons, state=st, eps=I["eps"])


def _yee3d_problem(case, seed):
    from meep_torch_amd.core.monitors_3d import FluxMonitor3D, PointSource3D
    from meep_torch_amd.core.sources import GaussianPulse
    from meep_torch_amd.core.stepper_3d import build_3d_coeffs, init_3d_state
    I, dtype = _inputs3d(case, seed), _dtype(case)
    nx, ny, nz, p = case["nx"], case["ny"], case["nz"], case["npml"]
    kw = {}
    if "media" in I:
        m = I["media"]
        kw = dict(poles=m["poles"], pole_masks=m["masks"], sigma_d=m["sigma_d"])
    c = build_3d_coeffs(nx, ny, nz, case["dx"], eps=I["eps"], npml=p, dtype=dtype, device="cuda", **kw)
    fc, fw, cut = I["pulse"]
    src = PointSource3D(c.dt, *I["src"], GaussianPulse(fc, fw, cutoff=cut))
    mons = [FluxMonitor3D(c.dt, I["freqs"], normal="x", idx=i, ap=p + 1, dtype=dtype) for i in _planes3d(case)]
    st = init_3d_state(nx, ny, nz, npml=p, n_poles=len(kw.get("poles", ())), dtype=dtype, device="cuda")
    if "fields" in I:
        st = st._replace(**I["fields"])
    return dict(case=case, coeffs=c, source=src, monitors=mons, state=st, eps=I["eps"])


def _batch_problem(case, seed):
    from meep_torch_amd.batch import BatchedTM
    probs = [_tm_problem(c, s) for c, s in _batch_cases(case, seed)]
    bt = BatchedTM([(q["coeffs"], q["source"], q["monitors"]) for q in probs], case["steps"],
                   checkpoint_every=case["ck"])
    eps = [q["eps"] for q in probs]
    bt.set_eps(eps)
    bt.capture()
    bt.capture_adjoint()
    return dict(case=case, runner=bt, eps=eps, monitors=[q["monitors"] for q in probs])


def _net_problem(case, seed):
    from meep_torch_amd.surrogate.fno import SpectralOperator
    I = _inputs_net(case, seed)
    net = SpectralOperator(n=case["n"], device="cuda", **_NET)
    net.load_state_dict({"params": torch.cat([I["p"][n].reshape(-1) for n, _, _ in I["spec"]])})
    return dict(case=case, net=net, rho=I["rho"], T=I["T"])


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("tm", "tm_grad"):
        return _tm_problem(case, seed)
    if kind in ("te", "te_grad"):
        return _te_problem(case, seed)
    if kind in ("yee3d", "yee3d_grad"):
        return _yee3d_problem(case, seed)
    if kind == "batch":
        return _batch_problem(case, seed)
    return _net_problem(case, seed)


# -------------------------------------------------------------------------- run
_TM_OUT = ("Ez", "Hx", "Hy", "Dz", "psi_Ezy", "psi_Ezx", "psi_Hyx", "psi_Hxy")
_TE_OUT = ("Hz", "Ex", "Ey", "Dx", "Dy", "psi_Eyx", "psi_Exy", "psi_Hzy", "psi_Hzx")
_E3_OUT = ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz", "psi_Ez_y", "psi_Ey_z", "psi_Ex_z", "psi_Ez_x", "psi_Ey_x",
           "psi_Ex_y", "psi_Hz_y", "psi_Hy_z", "psi_Hx_z", "psi_Hz_x", "psi_Hy_x", "psi_Hx_y")


def _names(case):
    media = case.get("media")
    if case["kind"] == "tm":
        return _TM_OUT + (("P_cur", "P_prev") if media else ())
    if case["kind"] == "te":
        return _TE_OUT
    return _E3_OUT + (("Px_cur", "Px_prev", "Py_cur", "Py_prev", "Pz_cur", "Pz_prev") if media else ())


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("tm", "te"):
        from meep_torch_amd.core import run as R
        fn = R.run_tm if kind == "tm" else R.run_te
        st, accs = fn(state["state"], state["coeffs"], case["steps"], source=state["source"],
                      monitors=state["monitors"])
        return [getattr(st, f) for f in _names(case)] + list(accs)
    if kind == "tm_grad":
        from meep_torch_amd.core.run import run_tm
        eps = state["eps"].detach().clone().requires_grad_(True)
        _, accs = run_tm(state["state"], state["coeffs"]._replace(eps_inf=eps), case["steps"],
                         source=state["source"], monitors=state["monitors"], checkpoint_every=case["ck"])
        state["monitors"][0].flux(accs[0], case["dx"]).sum().backward()
        return [accs[0].detach(), eps.grad]
    if kind == "te_grad":
        from meep_torch_amd.core.coeffs import build_te_coeffs
        from meep_torch_amd.core.run import run_te
        eps = state["eps"].detach().clone().requires_grad_(True)
        co = build_te_coeffs(state["grid"], eps_inf=eps, npml=case["npml"])
        _, accs = run_te(state["state"], co, case["steps"], source=state["source"], monitors=state["monitors"],
                         checkpoint_every=case["ck"])
        state["monitors"][0].flux(accs[0], case["dx"]).sum().backward()
        return [accs[0].detach(), eps.grad]
    if kind == "batch":
        eps = [e.detach().clone().requires_grad_(True) for e in state["eps"]]
        out = state["runner"].apply(eps)
        fom = sum(m[0].flux(o[0], case["dx"]).sum() for m, o in zip(state["monitors"], out))
        fom.backward()
        return [o[0].detach() for o in out] + [e.grad for e in eps]
    if kind == "yee3d":
        from meep_torch_amd.core.monitors_3d import run_3d
        st, accs = run_3d(state["state"], state["coeffs"], case["steps"], source=state["source"],
                          monitors=state["monitors"])
        return [getattr(st, f) for f in _names(case)] + list(accs)
    if kind == "yee3d_grad":
        from meep_torch_amd.core.adjoint3d import run_3d_adjoint
        eps = state["eps"].detach().clone().requires_grad_(True)
        mon = state["monitors"][0]
        _, accs = run_3d_adjoint(state["coeffs"]._replace(eps=eps), case["steps"], case["ck"], state["source"],
                                 state["monitors"], lambda a: mon.flux(a[0], case["dx"]).sum(), state["state"])
        return [accs[0], eps.grad]
    net = state["net"]
    if kind == "net_train":
        pred = net.forward(state["rho"])
        diff = pred - state["T"]
        net.backward(diff * (2.0 / diff.numel()), param_grads=True, input_grad=False)
        # input_grad=False leaves the lift layer's gradients unformed
        n_lift = _NET["width"] * (_NET["in_ch"] + 1)
        return [pred, net.grads[n_lift:]]
    from meep_torch_amd.surrogate.fno import predict
    rho = state["rho"].detach().clone().requires_grad_(True)
    T = predict(net, rho)
    T.mean(1).sum().backward()
    return [T.detach(), rho.grad]


# ------------------------------------------------------------- work and tolerance
def work(case):
    """Bytes and operations of one pass.  A time step reads and writes its
    fields once and reads eps (and its media maps) once: per cell 28 B (TM),
    29 B (TE) and 58 B (3D) in FP32; a reverse step moves the cotangents the
    same way.  A gradient is a forward and a reverse sweep."""
    kind = case["kind"]
    if kind in ("net_train", "net_design"):
        P, B, C, Mo, H, L = case["n"] ** 2, case["batch"], 64, 128, 128, 4
        f = 2.0 * B * P * (3 * C + L * (2 * C * 2 * Mo + C * C) + C * H) + 2.0 * B * L * Mo * 4 * C * C
        act = 2.0 * B * P * C * (L + 1)                       # layer activations in BF16
        w = 4.0 * (2 * C * C * Mo * L)
        if kind == "net_train":
            return {"bytes": 2 * act * 2 + 2 * w, "flops": 3 * f}
        return {"bytes": 2 * act * 2 + w, "flops": 2 * f}
    if kind == "batch":
        ws = [work(c) for c, _ in _batch_cases(case, 0)]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    sz = 2.0 if case["fp64"] else 1.0
    if kind.startswith("yee3d"):
        cells = case["nx"] * case["ny"] * case["nz"]
        b, f = 58.0, 40.0
        if case.get("media"):
            b, f = b + 4 * (2 * 3 * 4 + 6), f + 3 * 2 * 8
    else:
        cells = case["nx"] * case["ny"]
        b, f = (28.0, 18.0) if kind.startswith("tm") else (29.0, 20.0)
        if case.get("media"):
            b, f = b + 4 * (2 * 4 + 3), f + 40
    n = cells * case["steps"] * (2 if kind.endswith("_grad") else 1)
    return {"bytes": b * sz * n, "flops": f * n}


def tolerance(case):
    """About four times the largest relative distance from `exact` seen over
    the listed and a few dozen drawn cases.  The weak outputs are the CPML
    memories of a nearly silent edge; a Drude pole's recurrence (c1 near 2)
    amplifies its own rounding, hence the wider band for media."""
    kind = case["kind"]
    if kind.startswith("net"):
        return {"rel": 1.5e-2}
    if case["fp64"]:
        return {"rel": 1e-11 if case.get("media") else 1e-12}
    if case.get("media"):
        return {"rel": 5e-3}
    if kind in ("tm", "te"):
        return {"rel": 2e-4}
    return {"rel": 2e-5}


# ------------------------------------------------- the same in float64, plain torch
def _profiles(n, npml, offset, dt, dx):
    pos = torch.arange(n, dtype=F64, device="cuda") + offset
    wall = n - 1 + 2.0 * offset
    ul = torch.clamp((npml - pos) / npml, min=0.0)
    uh = torch.clamp((pos - (wall - npml)) / npml, min=0.0)
    smax = -4.0 * math.log(1e-6) / (2.0 * npml * dx)
    sig = smax * ul ** 3 + smax * uh ** 3
    u = torch.clamp(ul + uh, max=1.0)
    alpha = torch.where(u > 0, 0.05 * (1.0 - u), torch.zeros_like(u))
    b = torch.exp(-(sig + alpha) * dt)
    a = torch.where(sig > 0, sig * (b - 1.0) / (sig + alpha).clamp(min=1e-300), torch.zeros_like(b))
    return b, a


def _amp(pulse, t):
    fc, fw, cut = pulse
    w = 1.0 / fw
    d = t - cut * w
    return math.cos(2 * math.pi * fc * d) * math.exp(-d * d / (2 * w * w))


def _pole(pole, dt):
    fn, gamma, sigma = pole[:3]
    fc = pole[3] if len(pole) > 3 else fn
    w0, wc, G = 2 * math.pi * fn, 2 * math.pi * fc, 2 * math.pi * gamma
    den = 1.0 + G * dt / 2.0
    return (2.0 - w0 * w0 * dt * dt) / den, -(1.0 - G * dt / 2.0) / den, sigma * wc * wc * dt * dt / den


def _pad(v, *p):
    return torch.nn.functional.pad(v, p)


class _Spectra:
    """Running transforms of a list of (E, H) lines: (nfreq, 4, n) each."""

    def __init__(self, freqs, dt, sample, e_half, h_half):
        self.w = 2 * math.pi * torch.tensor(freqs, dtype=F64, device="cuda")
        self.dt, self.sample, self.e_half, self.h_half = dt, sample, e_half, h_half

    def _ph(self, t, half, rank):
        p = self.w * ((t + (0.5 if half else 1.0)) * self.dt)
        sh = (-1,) + (1,) * rank
        return torch.cos(p).reshape(sh), torch.sin(p).reshape(sh)

    def add(self, acc, s, t):
        out = []
        for i, terms in enumerate(self.sample(s)):
            rows = []
            for q, v in enumerate(terms):
                c, sn = self._ph(t, self.e_half if q % 2 == 0 else self.h_half, v.dim())
                rows += [c * v, -sn * v]
            smp = self.dt * torch.stack(rows, 1)
            out.append(smp if acc is None else acc[i] + smp)
        return out


def _tm_exact(case, I, eps, s0=None):
    """step(state, t) of the TM scheme in float64."""
    nx, ny, dx, p = case["nx"], case["ny"], case["dx"], case["npml"]
    dt = 0.5 * dx
    by, ay = _profiles(ny - 1, p, 0.5, dt, dx)
    bx, ax = _profiles(nx - 1, p, 0.5, dt, dx)
    bX, aX = _profiles(nx, p, 0.0, dt, dx)
    bY, aY = _profiles(ny, p, 0.0, dt, dx)
    bx, ax, bX, aX = bx[:, None], ax[:, None], bX[1:-1, None], aX[1:-1, None]
    by, ay, bY, aY = by[None], ay[None], bY[None, 1:-1], aY[None, 1:-1]
    ix, j0, j1 = I["src"]
    mask = torch.zeros(nx, ny, dtype=F64, device="cuda")
    mask[ix, j0:j1] = 1.0 / dx if j1 - j0 > 1 else 1.0 / dx ** 2
    z = lambda *sh: torch.zeros(*sh, dtype=F64, device="cuda")
    s = {"Ez": z(nx, ny), "Hx": z(nx, ny - 1), "Hy": z(nx - 1, ny), "Dz": z(nx, ny), "psi_Ezy": z(nx, ny - 1),
         "psi_Ezx": z(nx - 1, ny), "psi_Hyx": z(nx - 2, ny - 2), "psi_Hxy": z(nx - 2, ny - 2)}
    for k, v in I.get("fields", {}).items():
        s[k] = v.to(F64)
    m = I.get("media")
    if m:
        rec = [_pole(q, dt) for q in m["poles"]]
        c1 = torch.tensor([r[0] for r in rec], dtype=F64, device="cuda")[:, None, None]
        c2 = torch.tensor([r[1] for r in rec], dtype=F64, device="cuda")[:, None, None]
        c3 = torch.stack([r[2] * k.to(F64) for r, k in zip(rec, m["masks"])])
        chi3, sd = m["chi3"].to(F64), m["sigma_d"].to(F64)
        d1, d2 = (1 - sd * dt / 2) / (1 + sd * dt / 2), dt / (1 + sd * dt / 2)
        s["P_cur"], s["P_prev"] = z(len(rec), nx, ny), z(len(rec), nx, ny)

    def step(s, t):
        Ez = s["Ez"]
        g, h = (Ez[:, 1:] - Ez[:, :-1]) / dx, (Ez[1:] - Ez[:-1]) / dx
        o = {"psi_Ezy": by * s["psi_Ezy"] + ay * g, "psi_Ezx": bx * s["psi_Ezx"] + ax * h}
        o["Hx"] = s["Hx"] - dt * (g + o["psi_Ezy"])
        o["Hy"] = s["Hy"] + dt * (h + o["psi_Ezx"])
        dHx = (o["Hx"][1:-1, 1:] - o["Hx"][1:-1, :-1]) / dx
        dHy = (o["Hy"][1:, 1:-1] - o["Hy"][:-1, 1:-1]) / dx
        o["psi_Hyx"] = bX * s["psi_Hyx"] + aX * dHy
        o["psi_Hxy"] = bY * s["psi_Hxy"] + aY * dHx
        curl = _pad(dHy + o["psi_Hyx"] - dHx - o["psi_Hxy"], 1, 1, 1, 1)
        a = _amp(I["pulse"], (t + 0.5) * dt)
        if not m:
            o["Dz"] = s["Dz"] + dt * curl - dt * a * mask
            o["Ez"] = o["Dz"] / eps
            return o
        o["Dz"] = d1 * s["Dz"] + d2 * curl - d2 * a * mask
        o["P_cur"], o["P_prev"] = c1 * s["P_cur"] + c2 * s["P_prev"] + c3 * Ez, s["P_cur"]
        rhs = o["Dz"] - o["P_cur"].sum(0)
        E = rhs / eps
        for _ in range(3):
            E = rhs / (eps + chi3 * E * E)
        o["Ez"] = E
        return o

    return s, step, dt


def _te_exact(case, I, eps):
    nx, ny, dx, p = case["nx"], case["ny"], case["dx"], case["npml"]
    dt = 0.5 * dx
    ex, ey = 0.5 * (eps[:-1] + eps[1:]), 0.5 * (eps[:, :-1] + eps[:, 1:])
    by, ay = _profiles(ny - 1, p, 0.5, dt, dx)
    bx, ax = _profiles(nx - 1, p, 0.5, dt, dx)
    bX, aX = _profiles(nx, p, 0.0, dt, dx)
    bY, aY = _profiles(ny, p, 0.0, dt, dx)
    bx, ax, bX, aX = bx[:, None], ax[:, None], bX[1:-1, None], aX[1:-1, None]
    by, ay, bY, aY = by[None], ay[None], bY[None, 1:-1], aY[None, 1:-1]
    ix, j0, j1 = I["src"]
    mask = torch.zeros(nx, ny - 1, dtype=F64, device="cuda")
    mask[ix, j0:j1] = 1.0 / dx if j1 - j0 > 1 else 1.0 / dx ** 2
    z = lambda *sh: torch.zeros(*sh, dtype=F64, device="cuda")
    s = {"Hz": z(nx - 1, ny - 1), "Ex": z(nx - 1, ny), "Ey": z(nx, ny - 1), "Dx": z(nx - 1, ny),
         "Dy": z(nx, ny - 1), "psi_Eyx": z(nx - 1, ny - 1), "psi_Exy": z(nx - 1, ny - 1),
         "psi_Hzy": z(nx - 1, ny - 2), "psi_Hzx": z(nx - 2, ny - 1)}
    for k, v in I.get("fields", {}).items():
        s[k] = v.to(F64)

    def step(s, t):
        Hz = s["Hz"]
        gy, gx = (Hz[:, 1:] - Hz[:, :-1]) / dx, (Hz[1:] - Hz[:-1]) / dx
        o = {"psi_Hzy": bY * s["psi_Hzy"] + aY * gy, "psi_Hzx": bX * s["psi_Hzx"] + aX * gx}
        o["Dx"] = s["Dx"] + dt * _pad(gy + o["psi_Hzy"], 1, 1)
        o["Dy"] = s["Dy"] - dt * _pad(gx + o["psi_Hzx"], 0, 0, 1, 1) - dt * _amp(I["pulse"], (t + 0.5) * dt) * mask
        o["Ex"], o["Ey"] = o["Dx"] / ex, o["Dy"] / ey
        dEy, dEx = (o["Ey"][1:] - o["Ey"][:-1]) / dx, (o["Ex"][:, 1:] - o["Ex"][:, :-1]) / dx
        o["psi_Eyx"] = bx * s["psi_Eyx"] + ax * dEy
        o["psi_Exy"] = by * s["psi_Exy"] + ay * dEx
        o["Hz"] = Hz - dt * (dEy + o["psi_Eyx"] - dEx - o["psi_Exy"])
        return o

    return s, step, dt


_PSI3 = (("psi_Ez_y", "Ez", 1, "H"), ("psi_Ey_z", "Ey", 2, "H"), ("psi_Ex_z", "Ex", 2, "H"),
         ("psi_Ez_x", "Ez", 0, "H"), ("psi_Ey_x", "Ey", 0, "H"), ("psi_Ex_y", "Ex", 1, "H"),
         ("psi_Hz_y", "Hz", 1, "E"), ("psi_Hy_z", "Hy", 2, "E"), ("psi_Hx_z", "Hx", 2, "E"),
         ("psi_Hz_x", "Hz", 0, "E"), ("psi_Hy_x", "Hy", 0, "E"), ("psi_Hx_y", "Hx", 1, "E"))


def _yee3d_exact(case, I, eps):
    dims, dx, p = (case["nx"], case["ny"], case["nz"]), case["dx"], case["npml"]
    nx, ny, nz = dims
    dt = 0.5 * dx / math.sqrt(3.0)
    avg = lambda v, a: 0.5 * (v.narrow(a, 0, v.shape[a] - 1) + v.narrow(a, 1, v.shape[a] - 1))
    dif = lambda v, a: (v.narrow(a, 1, v.shape[a] - 1) - v.narrow(a, 0, v.shape[a] - 1)) / dx
    pro = {}
    for a, n in enumerate(dims):
        sh = [1, 1, 1]
        sh[a] = -1
        pro["H", a] = [v.reshape(sh) for v in _profiles(n - 1, p, 0.5, dt, dx)]
        pro["E", a] = [v[1:-1].reshape(sh) for v in _profiles(n, p, 0.0, dt, dx)]
    ec = {"E" + c: avg(eps, a) for a, c in enumerate("xyz")}
    z = lambda *sh: torch.zeros(*sh, dtype=F64, device="cuda")
    s = {"Ex": z(nx - 1, ny, nz), "Ey": z(nx, ny - 1, nz), "Ez": z(nx, ny, nz - 1),
         "Hx": z(nx, ny - 1, nz - 1), "Hy": z(nx - 1, ny, nz - 1), "Hz": z(nx - 1, ny - 1, nz)}
    for name, f, a, _ in _PSI3:
        sh = list(s[f].shape)
        sh[a] -= 1
        s[name] = z(*sh)
    for k, v in I.get("fields", {}).items():
        s[k] = v.to(F64)
    m = I.get("media")
    if m:
        rec = [_pole(q, dt) for q in m["poles"]]
        sd = m["sigma_d"].to(F64)
        damp, c3 = {}, {}
        for a, c in enumerate("xyz"):
            q = avg(sd, a)
            damp["E" + c] = ((1 - q * dt / 2) / (1 + q * dt / 2), dt / (1 + q * dt / 2))
            c3["E" + c] = [r[2] * avg(k.to(F64), a) for r, k in zip(rec, m["masks"])]
            s[f"P{c}_cur"] = z(len(rec), *s["E" + c].shape)
            s[f"P{c}_prev"] = z(len(rec), *s["E" + c].shape)
    comp, si, sj, sk = I["src"]
    keep = {}
    for c, cut in (("Ex", (1, 2)), ("Ey", (0, 2)), ("Ez", (0, 1))):
        keep[c] = [slice(1, -1) if a in cut else slice(None) for a in range(3)]

    def step(s, t):
        o = {}

        def term(src, name, f, a, side):
            d = dif(src[f], a)
            b, aa = pro[side, a]
            o[name] = b * s[name] + aa * d
            return d + o[name]

        T = {n: (f, a, sd_) for n, f, a, sd_ in _PSI3}
        cu = lambda src, u, v: term(src, u, *T[u]) - term(src, v, *T[v])
        o["Hx"] = s["Hx"] - dt * cu(s, "psi_Ez_y", "psi_Ey_z")
        o["Hy"] = s["Hy"] - dt * cu(s, "psi_Ex_z", "psi_Ez_x")
        o["Hz"] = s["Hz"] - dt * cu(s, "psi_Ey_x", "psi_Ex_y")
        amp = dt * _amp(I["pulse"], (t + 0.5) * dt)
        for c, (u, fu), (v, fv) in (("Ex", ("psi_Hz_y", 2), ("psi_Hy_z", 1)), ("Ey", ("psi_Hx_z", 0), ("psi_Hz_x", 2)),
                                    ("Ez", ("psi_Hy_x", 1), ("psi_Hx_y", 0))):
            tu, tv = term(o, u, *T[u]), term(o, v, *T[v])
            curl = tu.narrow(fu, 1, tu.shape[fu] - 2) - tv.narrow(fv, 1, tv.shape[fv] - 2)
            pad = [0] * 6
            for a in {"Ex": (1, 2), "Ey": (0, 2), "Ez": (0, 1)}[c]:
                pad[2 * (2 - a)] = pad[2 * (2 - a) + 1] = 1
            curl = _pad(curl, *pad)
            if m:
                d1, d2 = damp[c]
                P, Pp = s[f"P{c[1]}_cur"], s[f"P{c[1]}_prev"]
                Pn = torch.stack([r[0] * P[q] + r[1] * Pp[q] + c3[c][q] * s[c] for q, r in enumerate(rec)])
                o[f"P{c[1]}_cur"], o[f"P{c[1]}_prev"] = Pn, P
                E = (d1 * (s[c] * ec[c] + P.sum(0)) + d2 * curl - Pn.sum(0)) / ec[c]
            else:
                E = s[c] + dt * curl / ec[c]
            if c == comp:
                hot = torch.zeros_like(E)
                hot[si, sj, sk] = amp
                E = E + hot / ec[c]
            o[c] = E
        return o

    return s, step, dt


def _sampler(case):
    kind = case["kind"]
    half = lambda a, b: 0.5 * (a + b)
    if kind == "tm_grad":
        ix, lo, hi = _grad_line(case)
        return lambda s: [[s["Ez"][ix, lo:hi], half(s["Hy"][ix - 1, lo:hi], s["Hy"][ix, lo:hi])]]
    if kind == "te_grad":
        ix, lo, hi = _grad_line(case)
        return lambda s: [[s["Ey"][ix, lo:hi], half(s["Hz"][ix - 1, lo:hi], s["Hz"][ix, lo:hi])]]
    if kind in ("tm", "te"):
        lx, ly, lo, hi = _lines(case)
    if kind == "tm":
        def tm(s):
            i, j, h2 = lx[1], ly[0], case["ny"] - lo
            out = [[s["Ez"][i, lo:h2], half(s["Hy"][i - 1, lo:h2], s["Hy"][i, lo:h2])]]
            if case.get("media"):
                out.append([s["Ez"][lo:hi, j], half(s["Hx"][lo:hi, j - 1], s["Hx"][lo:hi, j])])
            return out
        return tm
    if kind == "te":
        return lambda s: ([[s["Ey"][i, lo:hi], half(s["Hz"][i - 1, lo:hi], s["Hz"][i, lo:hi])] for i in lx] +
                          [[s["Ex"][lo:hi, j], half(s["Hz"][lo:hi, j - 1], s["Hz"][lo:hi, j])] for j in ly])
    ap = case["npml"] + 1
    m0, m1 = case["ny"] - 1 - ap, case["nz"] - 1 - ap
    cr = lambda v: v[ap:m0, ap:m1]
    return lambda s: [[cr(s["Ey"][i]), cr(half(s["Hz"][i - 1], s["Hz"][i])), cr(s["Ez"][i]),
                       cr(half(s["Hy"][i - 1], s["Hy"][i]))] for i in _planes3d(case)]


def _fom(case, acc):
    """Sum of a line's or plane's fluxes over its frequencies."""
    dx = case["dx"]
    if case["kind"] == "yee3d_grad":
        a, b, c, d, e, f, g, h = acc.unbind(1)
        return 0.5 * ((a * c + b * d) - (e * g + f * h)).sum() * dx * dx
    a, b, c, d = acc.unbind(1)
    return (-0.5 if case["kind"] == "tm_grad" else 0.5) * (a * c + b * d).sum() * dx


def _march(case, I, eps, grad):
    maker = {"tm": _tm_exact, "te": _te_exact, "ye": _yee3d_exact}[case["kind"][:2]]
    s, step, dt = maker(case, I, eps)
    te = case["kind"].startswith("te")
    spec = _Spectra(I["freqs"], dt, _sampler(case), te, not te)
    names = list(s)

    def chunk(t0, t1, *flat):
        s, acc = dict(zip(names, flat[:len(names)])), list(flat[len(names):]) or None
        for t in range(t0, t1):
            s = step(s, t)
            acc = spec.add(acc, s, t)
        return (*[s[n] for n in names], *acc)

    flat, n = [s[k] for k in names], case["steps"]
    if not grad:
        flat = chunk(0, n, *flat)
    else:
        from torch.utils.checkpoint import checkpoint
        for t in range(0, n, 20):
            flat = checkpoint(chunk, t, min(n, t + 20), *flat, use_reentrant=False)
    return dict(zip(names, flat)), list(flat[len(names):])


def _net_exact(case, I, need_rho):
    n, B = case["n"], case["batch"]
    C, L, (mx, my) = _NET["width"], _NET["layers"], _NET["modes"]
    p = {k: v.to(F64).requires_grad_(not need_rho) for k, v in I["p"].items()}
    rho = I["rho"].to(F64).requires_grad_(need_rho)
    kx = [a if a < mx // 2 else n - mx + a for a in range(mx)]
    gx = (torch.arange(n, dtype=F64, device="cuda") + 0.5) / n
    x = torch.stack([rho, gx[:, None].expand(n, n).expand(B, n, n), gx[None, :].expand(n, n).expand(B, n, n)], 1)
    x = x.reshape(B, 3, n * n)
    v = torch.matmul(p["lift_w"], x) + p["lift_b"][:, None]
    for l in range(L):
        vh = torch.fft.rfft2(v.reshape(B, C, n, n), norm="ortho")[:, :, kx, :my].reshape(B, C, mx * my)
        w = torch.complex(p[f"s{l}_re"], p[f"s{l}_im"])
        uh = torch.matmul(vh.permute(2, 0, 1).contiguous(), w.permute(2, 0, 1).contiguous()).permute(1, 2, 0)
        full = torch.zeros(B, C, n, n // 2 + 1, dtype=torch.complex128, device="cuda")
        idx = torch.tensor(kx, device="cuda")
        full = full.index_copy(2, idx, _pad(uh.reshape(B, C, mx, my), 0, n // 2 + 1 - my))
        u = torch.fft.irfft2(full, s=(n, n), norm="ortho").reshape(B, C, n * n)
        u = u + torch.matmul(p[f"w{l}"], v) + p[f"b{l}"][:, None]
        v = torch.nn.functional.gelu(u) if l < L - 1 else u
    h = torch.nn.functional.gelu(torch.matmul(p["q_w"], v) + p["q_b"][:, None]).mean(2)
    return p, rho, h @ p["o_w"].t() + p["o_b"]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("tm", "te", "yee3d"):
        I = _inputs3d(case, seed) if kind == "yee3d" else _inputs2d(case, seed)
        with torch.no_grad():
            s, accs = _march(case, I, I["eps"].to(F64), False)
        return [s[n] for n in _names(case)] + accs
    if kind in ("tm_grad", "te_grad", "yee3d_grad"):
        I = _inputs3d(case, seed) if kind == "yee3d_grad" else _inputs2d(case, seed)
        eps = I["eps"].to(F64).requires_grad_(True)
        _, accs = _march(case, I, eps, True)
        _fom(case, accs[0]).backward()
        return [accs[0].detach(), eps.grad]
    if kind == "batch":
        accs, grads = [], []
        for c, s in _batch_cases(case, seed):
            a, g = exact(c, s)
            accs.append(a)
            grads.append(g)
        return accs + grads
    I = _inputs_net(case, seed)
    if kind == "net_train":
        p, _, out = _net_exact(case, I, False)
        ((out - I["T"].to(F64)) ** 2).mean().backward()
        return [out.detach(), torch.cat([p[n].grad.reshape(-1) for n, _, _ in I["spec"][2:]])]
    _, rho, out = _net_exact(case, I, True)
    out.mean(1).sum().backward()
    return [out.detach(), rho.grad]
