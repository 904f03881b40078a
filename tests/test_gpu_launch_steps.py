"""Runs of tiled launches end in the buffers they began in: step counts that
need one launch, an even and an odd number of them, a last launch of one step
and a staging block that ends inside the run, bit-identical to the two-pass
path."""
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

