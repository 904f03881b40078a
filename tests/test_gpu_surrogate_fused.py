"""The operator's fused passes (spectral.hip) against the general GEMM and
elementwise kernels on the same weights, both measured against the float64
oracle: outputs, every parameter gradient and the input gradient at the
smallest grid, at point counts that end inside a 128-point tile and inside a
64-point reduction step, and at batches of one, of less and more than a
32-row tile of the mode mixing."""
import pytest
import torch

from conftest import has_gpu
from oracle import fno as O

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not has_gpu(), reason="needs a HIP device")]


def _net(n, fused, seed=5):
    from meep_torch_amd.surrogate.fno import SpectralOperator
    net = SpectralOperator(n=n, n_out=7, seed=seed)
    assert net.fused
    net.fused = fused
    with torch.no_grad():   # spectral weights large enough that their path carries signal
        for l in range(4):
            for part in ("re", "im"):
                t = net.p[f"s{l}_{part}"]
                t.copy_((torch.rand(t.shape, generator=torch.Generator().manual_seed(l)) - 0.5).cuda() * 0.1)
    net.fused = True
    net.sync_weights()
    for l in range(4):      # the general path's packing of the same weights
        from meep_torch_amd.surrogate import _nn
        ref = torch.empty_like(net._wbf[f"wp{l}"])
        _nn.pack_spectral(net.p[f"s{l}_re"], net.p[f"s{l}_im"], ref, 64, 64, 128)
        assert torch.equal(ref, net._wbf[f"wp{l}"])
        assert torch.equal(ref.transpose(1, 2), net._wbf[f"wp{l}T"])
    net.fused = fused
    return net


@pytest.mark.parametrize("n,B", [(16, 1), (20, 3), (36, 33), (100, 2), (128, 5)])
def test_fused_passes_match_general_kernels(n, B):
    g = torch.Generator().manual_seed(n + B)
    rho = torch.rand(B, n, n, generator=g)
    dout = torch.randn(B, 7, generator=g)
    res = []
    for fused in (False, True):
        net = _net(n, fused)
        out = net.forward(rho.cuda())
        drho = net.backward(dout.cuda())
        r = {"out": out, "drho": drho, **net._views(net.grads.clone())}
        res.append({k: v.double().cpu() for k, v in r.items()})
        # without parameter gradients the input gradient is the same bits
        assert torch.equal(net.backward(dout.cuda(), param_grads=False), drho)
    p = {k: v.double().cpu().numpy() for k, v in net.p.items()}
    cfg = dict(n=n, modes=(16, 8), layers=4, in_ch=3)
    out, cache = O.forward(p, rho.double().numpy(), cfg, emulate=False)
    exact, drho = O.backward(p, cache, dout.double().numpy(), cfg)
    exact = {"out": out, "drho": drho, **exact}
    rel = lambda a, b: float((a - b).norm() / b.norm())
    for k, general in res[0].items():
        want = torch.as_tensor(exact[k]).reshape(general.shape)
        # Both paths round FP32 sums to BF16 between the same products, so
        # each lies e from the float64 result and both share most of that
        # error; sums in another order only put some elements on the other
        # side of a rounding step.  The paths then lie within e of each other,
        # and the fused one is no further from float64 than the general one
        # beyond the sampling of those flips (an eighth covers one flip in
        # 64 elements, the size of the smallest tensors; 2^-12 is the floor
        # of one BF16 rounding spread over 256 of them).
        e = rel(general, want)
        assert rel(res[1][k], general) <= e + 2.0 ** -12, (k, e)
        assert rel(res[1][k], want) <= 1.125 * e + 2.0 ** -12, (k, e)


def test_fused_passes_repeat_exactly_and_grow():
    """Same inputs, same bits (no scheduling-dependent sums); buffers follow a
    larger batch and a smaller one after it."""
    net = _net(20, True)
    g = torch.Generator().manual_seed(1)
    rho = torch.rand(9, 20, 20, generator=g).cuda()
    first = []
    for B in (2, 9, 2):
        out = net.forward(rho[:B])
        drho = net.backward(torch.ones(B, 7, device="cuda"))
        first.append((out.clone(), drho.clone(), net.grads.clone()))
    for a, b in zip(first[0], first[2]):
        assert torch.equal(a, b)
