"""The network's head as tensor operations wherever something follows them:
forward mode and batched gradients."""

import pytest
import torch
import torch.autograd.forward_ad as fwd

from ggems_amd import surrogate

pytestmark = pytest.mark.gpu


def _net():
    net = surrogate.UNet(seed=7).cuda()
    x = torch.rand(1, 32, 128, 3, device="cuda", generator=torch.Generator("cuda").manual_seed(2))
    return net, x


@pytest.mark.parametrize("record", [False, True])
def test_forward_mode_over_the_head(record):
    net, x = _net()
    for p in net.parameters():
        p.requires_grad_(record)
    head, bias = net.head.detach(), net.head_bias.detach()
    tangent = torch.linspace(-1, 1, 16, device="cuda")
    del net.head
    with torch.no_grad():  # linear in the head: its value at the tangent, without the bias
        net.head = tangent
        want = net(x) - bias
    with fwd.dual_level():
        net.head = fwd.make_dual(head, tangent)
        got = fwd.unpack_dual(net(x)).tangent
    # the same 16 products, and sums that the bias shifted: a few ulps of their magnitudes
    assert got is not None and (got - want).abs().max() <= 1e-5 * want.abs().max()


def test_batched_gradients_of_the_head():
    net, x = _net()
    out = net(x)
    d = torch.randn(3, *out.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    wanted = (net.head, net.head_bias)
    got = torch.autograd.grad(out, wanted, d, is_grads_batched=True, retain_graph=True)
    for k in range(3):
        one = torch.autograd.grad(out, wanted, d[k], retain_graph=True)
        for a, b in zip(got, one):  # FP32 sums over 4,096 pixels in another order
            assert (a[k] - b).abs().max() <= 1e-4 * b.abs().max() + 1e-3
