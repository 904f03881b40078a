"""MEEP_TORCH_AMD_VARIANT reaches the TM reverse sweep: -1 runs it step by
step (and never on tiles), a tile variant runs that tile; same gradient bits
and the same as without the variable."""
import pytest
import torch

from conftest import has_gpu
from test_gpu_reverse_any_monitor import _case, _grad

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


def test_forced_variant_in_the_reverse_sweep(monkeypatch):
    from meep_torch_amd import _engine as E
    c, src, st, mons = _case(torch.float32, "mean")
    L, mons, used = E.lib(), mons[:1], []
    tiled, steps = L.mt_tm2d_adjoint_tiled, L.mt_tm2d_adjoint
    monkeypatch.setattr(L, "mt_tm2d_adjoint_tiled",
                        lambda d, *a: used.append(d._obj.variant) or tiled(d, *a))
    monkeypatch.setattr(L, "mt_tm2d_adjoint", lambda *a: used.append(-1) or steps(*a))
    want = _grad(c, src, st, mons, 12)
    assert float(want.abs().max()) > 0
    for v in (-1, 5, 8):
        monkeypatch.setenv("MEEP_TORCH_AMD_VARIANT", str(v))
        used.clear()
        assert torch.equal(_grad(c, src, st, mons, 12), want), v
        assert used == [v] * 3
