"""The U-Net's fused calls against the calls they replace: a layer's three
gradients in one call, inference from the FP32 weights, the padded input and
the head, bit for bit where the order of additions is the same."""

import pytest
import torch

from ggems_amd import surrogate

pytestmark = pytest.mark.gpu


def _rand(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


@pytest.mark.parametrize("relu", [True, False])
@pytest.mark.parametrize("n,h,w,cin,cout,want_dx", [
    (1, 2, 16, 16, 16, True),        # less than a tile, one block
    (2, 10, 32, 8, 32, False),       # the first layer
    (3, 26, 48, 96, 64, True),       # rows past the image in the last tiles
    (1, 32, 32, 128, 128, True),     # split sums
    (9, 64, 64, 48, 16, True),       # blocks that walk several tiles, sums of many blocks
])
def test_layer_backward_equals_the_single_calls(n, h, w, cin, cout, want_dx, relu):
    g = torch.Generator("cuda").manual_seed(cin + cout)
    x = _rand(g, n, h, w, cin).to(torch.bfloat16)
    y = _rand(g, n, h, w, cout).to(torch.bfloat16)
    dy = _rand(g, n, h, w, cout).to(torch.bfloat16)
    wb, wt = surrogate.weights_bf16(_rand(g, cout, 9, cin))
    dx, dw, db = surrogate.conv3x3_backward(x, y if relu else None, dy, wt, want_dx, None)
    masked, want_db = surrogate.relu_bias_backward(dy, y, relu)
    want_dw = surrogate.conv3x3_weight_grad(x, masked)
    assert (dx is None) == (not want_dx)
    if want_dx:
        assert torch.equal(dx, surrogate.conv3x3(masked, wt.view(cin, 9 * cout)))
    # FP32 sums of the same products in another order: 16 ulps of the sum of magnitudes
    size = surrogate.conv3x3_weight_grad(x.abs(), masked.abs())
    assert ((dw - want_dw).abs() <= 1e-6 * size).all()
    assert ((db - want_db).abs() <= 1e-6 * masked.float().abs().sum((0, 1, 2))).all()


def test_layer_backward_leaves_other_shapes_to_the_single_calls():
    g = torch.Generator("cuda").manual_seed(1)
    for h, cin, cout, dtype in ((7, 16, 16, torch.bfloat16), (8, 24, 16, torch.bfloat16), (8, 16, 48, torch.bfloat16),
                                (8, 16, 16, torch.float32)):
        x, dy = _rand(g, 2, h, 16, cin).to(torch.bfloat16), _rand(g, 2, h, 16, cout).to(dtype)
        assert surrogate.conv3x3_backward(x, None, dy, None, False, None) is None


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("cin,cout", [(8, 16), (24, 16), (64, 128), (192, 64)])
def test_inference_layer_equals_the_recorded_one(cin, cout, offset):
    g = torch.Generator("cuda").manual_seed(cin)
    layer = surrogate.Conv3x3(cin, cout).cuda()
    store = _rand(g, cout * 9 * cin + offset)[offset:]  # weights that are not 16-byte aligned
    layer.weight = torch.nn.Parameter(store.view(cout, 9, cin))
    x = _rand(g, 1, 18, 32, cin).to(torch.bfloat16)
    want = layer(x).detach()
    with torch.no_grad():
        assert torch.equal(layer(x), want)


def test_padded_input_and_head_equal_tensor_operations():
    g = torch.Generator("cuda").manual_seed(4)
    net = surrogate.UNet(seed=2).cuda()
    x = _rand(g, 2, 40, 128, 3)
    z = torch.empty(2, 40, 128, 8, device="cuda", dtype=torch.bfloat16)
    surrogate._check(surrogate._lib().ggh_unet_pad(x.data_ptr(), z.data_ptr(), z.numel() // 8, 3, surrogate._stream(x)))
    assert torch.equal(z[..., :3], x.to(torch.bfloat16)) and not z[..., 3:].any()
    z = _rand(g, 2, 40, 128, 16).to(torch.bfloat16)
    far = z.clone()
    far[0, 0, 0, 0] = float("inf")
    with torch.no_grad():
        assert torch.equal(surrogate.head16(far, net.head, net.head_bias),
                           (far.float() * net.head).sum(dim=3) + net.head_bias)
    z.requires_grad_(True)
    out = surrogate._Head.apply(z, net.head, net.head_bias)
    want = (z.float() * net.head).sum(dim=3) + net.head_bias
    assert torch.equal(out, want)
    d = _rand(g, *out.shape)
    got = torch.autograd.grad(out, (z, net.head, net.head_bias), d)
    ref = torch.autograd.grad(want, (z, net.head, net.head_bias), d)
    assert torch.equal(got[0], ref[0])
    size = (d.abs()[..., None] * z.detach().float().abs()).sum((0, 1, 2))
    assert ((got[1] - ref[1]).abs() <= 1e-6 * size).all()
    assert abs(got[2] - ref[2]) <= 1e-6 * d.abs().sum()
    # gradients that are to be differentiated again keep their graph
    again = torch.autograd.grad(surrogate._Head.apply(z, net.head, net.head_bias), z, d, create_graph=True)[0]
    assert torch.equal(again, ref[0])
    second = torch.autograd.grad(again.float().sum(), net.head)[0]
    assert torch.allclose(second, d.sum().expand(16), rtol=1e-3, atol=1e-3 * d.abs().sum().item())


def test_network_without_gradients_equals_the_recorded_one():
    net = surrogate.UNet(seed=5).cuda()
    x = torch.rand(2, 64, 128, 3, device="cuda")
    want = net(x).detach()
    with torch.no_grad():
        assert torch.equal(net(x), want)
        assert torch.equal(net(x.to(torch.bfloat16).float()), want)
        # operations that others record keep their autograd functions
        import torch.autograd.forward_ad as fwd
        with fwd.dual_level(), pytest.raises(Exception):
            net(fwd.make_dual(x, torch.ones_like(x)))
    seen = []
    hook = net.enc[1][0].register_forward_hook(lambda m, i, o: seen.append(o.shape))
    with torch.no_grad():
        net(x)
    hook.remove()
    assert seen == [torch.Size([2, 32, 64, 32])]
