"""The BF16 weight copies of the spectral operator: the packed blocks and
their transposes at sizes on either side of the kernel's 32-mode, 64-channel
tiles against mt_pack_spectral, the cast beside its transpose against torch,
and a refresh that allocates nothing."""
import pytest
import torch

from conftest import has_gpu

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


@pytest.mark.parametrize("C,Mo", [(64, 128), (1, 1), (5, 7), (63, 32), (65, 33), (130, 31)])
def test_packed_weights_and_transposes(C, Mo):
    from meep_torch_amd.surrogate import _nn
    g = torch.Generator().manual_seed(C + Mo)
    re, im = (torch.randn(C, C, Mo, generator=g).cuda() for _ in range(2))
    ref, wp, wt = (torch.zeros(Mo, 2 * C, 2 * C, dtype=torch.bfloat16, device="cuda") for _ in range(3))
    _nn.pack_spectral(re, im, ref, C, C, Mo)
    _nn.pack_both(re, im, wp, wt, C, Mo)
    assert torch.equal(wp, ref)
    assert torch.equal(wt, ref.transpose(1, 2))


@pytest.mark.parametrize("R,C", [(64, 64), (128, 64), (3, 17)])
def test_cast_and_transpose(R, C):
    from meep_torch_amd.surrogate import _nn
    x = torch.randn(R, C, generator=torch.Generator().manual_seed(R)).cuda()
    y, yt = (torch.zeros(s, dtype=torch.bfloat16, device="cuda") for s in ((R, C), (C, R)))
    _nn.cast_transpose(x, y, yt, R, C)
    assert torch.equal(y, x.bfloat16()) and torch.equal(yt, x.bfloat16().t())


def test_refresh_allocates_nothing():
    from meep_torch_amd.surrogate.fno import SpectralOperator
    net = SpectralOperator(n=16, n_out=5)
    net.sync_weights()
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    before = count()
    net.sync_weights()
    assert count() == before


def test_general_bases_only_where_used():
    """The row-major bases of the general kernels are made on first use: a
    network on the fused passes holds the bases once and the fragments."""
    from meep_torch_amd.surrogate.fno import SpectralOperator, dft_bases
    net = SpectralOperator(n=16, n_out=5)
    net.backward(torch.ones_like(net.forward(torch.rand(2, 16, 16, device="cuda"))))
    assert net.fused and not any(k in vars(net) for k in ("FT", "GT")) and not net._rows
    F, G = dft_bases(16, 16, 8)
    for got, want in ((net.FT, F), (net.GT, G)):
        assert got.is_contiguous() and torch.equal(got, torch.from_numpy(want.T.copy()).float().bfloat16().cuda())
    assert net.FT is net.FT
