"""Tile choice for the temporally blocked 2D steppers.

A grid that fits the chip in one round of workgroups takes the smallest tile
that does (`one_round`): its launch lasts as long as one tile, so fewer cells
per tile and more steps per launch win.  Larger grids time the two large tile
shapes on scratch copies of the real state, sources and monitors, once per
problem signature (mode, grid, dtype, monitor layout), and cache the faster
for the rest of the process; `tune` times any set of variants, the two-pass
per-half-step path (-1) included.  MEEP_TORCH_AMD_VARIANT=<v> forces a variant
(-1 = two-pass), forward and in the TM reverse sweep (-1 = step by step)."""
import os

import torch

from . import _engine as E

_CACHE = {}
TUNE_STEPS = 24
# variants from the smallest tile to the largest (mt_tiled_variants), and the
# two timed on grids of more than one round (of all shapes and the two-pass
# path, ms per 200 steps: TM FP32 520 x 500 2.18 / 1.62 with 2 / 5, next 2.02;
# 1500 x 1400 4.75 / 4.09, next 5.13; TE FP32 1500 x 1400 3.75 / 3.72, next
# 4.47.  FP64 with 4 / 9: TM 520 x 500 3.05 / 2.20, next 2.36; 1500 x 1400 7.27 /
# 7.19, next 8.11; TE 520 x 500 2.80 / 2.05, next 2.22; 2048^2 9.80 / 11.52, next
# 11.35).
LADDER = {torch.float32: (8, 7, 9, 2, 5), torch.float64: (8, 7, 9, 2)}
LARGE = {torch.float32: (2, 5), torch.float64: (4, 9)}
ROUND = 256                  # compute units: tiles that run side by side (kOneRound, schedule.h)


def variants(dtype):
    L = E.lib()
    n = L.mt_tiled_variants(E.dtype_code(dtype), None, None, None)
    steps = (E.c_int * n)()
    tx = (E.c_int * n)()
    ty = (E.c_int * n)()
    L.mt_tiled_variants(E.dtype_code(dtype), steps, tx, ty)
    return [(int(tx[v]), int(ty[v]), int(steps[v])) for v in range(n)]


def one_round(dtype, grids):
    """The smallest tile with which the (nx, ny) grids together make at most
    one round of workgroups; None if none does."""
    shapes = variants(dtype)
    for v in LADDER[dtype]:
        tx, ty, _ = shapes[v]
        if sum(-(-nx // tx) * -(-ny // ty) for nx, ny in grids) <= ROUND:
            return v
    return None


def tile_for(dtype, grids):
    """Variant of a launch over `grids` without timing: the smallest tile of
    one round, else the largest tile (FP32: 32 x 64 with 4 steps, 13% faster on
    64 variants of 514^2 - 1522^2 than 16 x 64; FP64: 8 x 64)."""
    v = one_round(dtype, grids)
    return LADDER[dtype][-1] if v is None else v


def forced_variant():
    """MEEP_TORCH_AMD_VARIANT as a number, None when unset."""
    env = os.environ.get("MEEP_TORCH_AMD_VARIANT")
    return None if env is None else int(env)


def _key(mode, fields, monitors):
    ref = fields["Ez"] if mode == "tm" else fields["Hz"]
    return (mode, tuple(ref.shape), ref.dtype, ref.device.index,
            tuple(type(m).__name__ for m in monitors))


def variant_for(mode, fields, coeffs, plan, monitors, k):
    v = forced_variant()
    if v is not None:
        return v
    ref = fields["Ez"] if mode == "tm" else fields["Hz"]
    if k <= 4:
        # four steps or fewer do not repay the copy into a second buffer set,
        # except the last of them on large FP32 grids (us, two-pass / 16 x 64 x 2
        # tiles: TE 2048^2 k = 2 457 / 473, 3 517 / 482, 4 574 / 486; 1500 x 1400
        # k = 4 437 / 423; TM 2048^2 k = 3 469 / 491, 4 521 / 507, 3000 x 2800
        # k = 4 756 / 742; FP64 two-pass throughout)
        paid = k - (3 if mode == "tm" else 2)
        return 1 if ref.dtype == torch.float32 and paid * ref.numel() >= 2 ** 22 else -1
    v = one_round(ref.dtype, [tuple(ref.shape)])
    if v is not None:
        return v
    if k < 2 * TUNE_STEPS:   # not timed; FP64: 16 x 64 x 2 wins from about 2^20 cells on
        return LARGE[ref.dtype][ref.dtype == torch.float64 and ref.numel() < 2 ** 20]
    key = _key(mode, fields, monitors)
    if key not in _CACHE:
        _CACHE[key] = tune(mode, fields, coeffs, plan, monitors, cands=LARGE[ref.dtype])
    return _CACHE[key]


def tune(mode, fields, coeffs, plan, monitors, steps=TUNE_STEPS, cands=None):
    """Time each candidate (default: every variant and the two-pass path) on
    copies of `fields`; returns the fastest."""
    from .core import engine2d
    ref = fields["Ez"] if mode == "tm" else fields["Hz"]
    if cands is None:
        cands = [-1] + list(range(len(variants(ref.dtype))))
    times = {}
    for v in cands:
        work = {f: t.clone() for f, t in fields.items()}
        alt = {f: t.clone() for f, t in fields.items()} if v >= 0 else None
        engine2d.run_chunk(mode, work, coeffs, 0, 4, plan, monitors, variant=v, alt=alt)
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        engine2d.run_chunk(mode, work, coeffs, 4, steps, plan, monitors, variant=v, alt=alt)
        e1.record()
        torch.cuda.synchronize()
        times[v] = e0.elapsed_time(e1)
    best = min(times, key=times.get)
    tune.last = times
    return best


tune.last = {}
