"""Tile choice without timing (tune.variant_for): which variant, or which
candidates, a run takes by its grid, type and step count."""
import pytest
import torch

from meep_torch_amd import tune

F32, F64 = torch.float32, torch.float64


def _choice(monkeypatch, mode, shape, dtype, k):
    """The variant of a run; of a timed one, the candidates."""
    monkeypatch.delenv("MEEP_TORCH_AMD_VARIANT", raising=False)
    monkeypatch.setattr(tune, "_CACHE", {})
    monkeypatch.setattr(tune, "tune", lambda *a, cands=None, **kw: tuple(cands))
    f = torch.empty(shape, dtype=dtype, device="meta")
    return tune.variant_for(mode, {"Ez": f, "Hz": f}, None, None, [], k)


@pytest.mark.parametrize("mode", ["tm", "te"])
def test_large_grids(monkeypatch, mode):
    for shape, short in (((700, 650), 9), ((2048, 2048), 4)):
        assert _choice(monkeypatch, mode, shape, F64, 200) == (4, 9)
        assert _choice(monkeypatch, mode, shape, F64, 40) == short
    assert _choice(monkeypatch, mode, (1500, 1400), F32, 200) == (2, 5)
    assert _choice(monkeypatch, mode, (1500, 1400), F32, 40) == 2


@pytest.mark.parametrize("mode", ["tm", "te"])
def test_grids_of_one_round(monkeypatch, mode):
    for shape, dtype, v in (((100, 60), F64, 8), ((256, 256), F32, 7), ((300, 300), F32, 9), ((500, 500), F32, 2)):
        assert _choice(monkeypatch, mode, shape, dtype, 400) == v


def test_few_steps(monkeypatch):
    c = lambda *a: _choice(monkeypatch, *a)
    for mode in ("tm", "te"):
        for k in (1, 2, 3, 4):
            assert c(mode, (256, 256), F32, k) == c(mode, (2048, 2048), F64, k) == -1
    assert [c("te", (2048, 2048), F32, k) for k in (1, 2, 3, 4)] == [-1, -1, 1, 1]
    assert [c("te", (1500, 1400), F32, k) for k in (2, 3, 4)] == [-1, -1, 1]
    assert [c("tm", (2048, 2048), F32, k) for k in (2, 3, 4)] == [-1, -1, 1]
    assert c("tm", (1500, 1400), F32, 4) == -1
