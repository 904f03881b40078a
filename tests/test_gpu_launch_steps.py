"""Runs of any number of tiled launches are bit-identical to the two-pass path:
step counts that need one launch, an even and an odd number of them, a last
launch of one step, a staging block that ends inside the run, and staging blocks
shorter than a launch.  (That launches come in an even number, so that runs end
in the buffers they began in, is checked in test_schedule_cpu.py.)"""
import pytest
import torch

from conftest import has_gpu
from test_gpu_small_tiles import _run

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


@pytest.mark.parametrize("k", [1, 2, 4, 7, 9, 12, 13, 64, 65, 130])
@pytest.mark.parametrize("variant", [2, 7, 8])
@pytest.mark.parametrize("mode", ["tm", "te"])
def test_any_step_count_matches_two_pass(mode, variant, k):
    for a, b in zip(_run(mode, torch.float32, variant, (65, 50), k, 6),
                    _run(mode, torch.float32, -1, (65, 50), k, 6)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("S", [1, 3, 7])
@pytest.mark.parametrize("variant", [2, 7, 8])
@pytest.mark.parametrize("mode", ["tm", "te"])
def test_short_staging_blocks(mode, variant, S, monkeypatch):
    from meep_torch_amd.core import engine2d
    monkeypatch.setattr(engine2d, "STAGE_STEPS", S)
    for a, b in zip(_run(mode, torch.float32, variant, (65, 50), 23, 6),
                    _run(mode, torch.float32, -1, (65, 50), 23, 6)):
        assert torch.equal(a, b)
