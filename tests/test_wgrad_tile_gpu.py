"""The tile weight gradient against FP64 sums of the same BF16 operands:
every split of the channels over blocks, heights that end inside a tile and
those left to the general kernel, one tile and many, an accumulator that
already holds a gradient, infinities that reach only some weights."""

import pytest
import torch

from ggems_amd import surrogate

pytestmark = pytest.mark.gpu


def _reference(x, dy):
    n, h, w, ci = x.shape
    xp = torch.nn.functional.pad(x.double(), (0, 0, 1, 1, 1, 1))
    d = dy.double().reshape(-1, dy.shape[3]).t().contiguous()
    return torch.stack([d @ xp[:, t // 3:t // 3 + h, t % 3:t % 3 + w, :].reshape(-1, ci) for t in range(9)], dim=1)


def _inputs(n, h, w, cin, cout, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    x = torch.randn(n, h, w, cin, device="cuda", generator=g).to(torch.bfloat16)
    dy = torch.randn(n, h, w, cout, device="cuda", generator=g).to(torch.bfloat16)
    return x, dy


@pytest.mark.parametrize("cin", [8, 16, 24, 32, 48, 64, 80, 192])
@pytest.mark.parametrize("n,h,w,cout", [
    (1, 2, 16, 16),      # one K step
    (2, 10, 32, 32),     # a tile's last rows alone
    (2, 7, 16, 64),      # odd height: the general kernel
    (1, 24, 48, 48),     # three groups of 16 output channels
    (4, 64, 64, 128),    # blocks that walk several tiles, two groups of 64
])
def test_matches_fp64(n, h, w, cin, cout):
    x, dy = _inputs(n, h, w, cin, cout, cin + cout + h)
    before = torch.randn(cout, 9 * cin, device="cuda")
    got = surrogate.conv3x3_weight_grad(x, dy, out=before.clone())
    want = _reference(x, dy).reshape(cout, 9 * cin) + before.double()
    # 16 ulps of FP32 on the sum of magnitudes
    bound = 1e-6 * (_reference(x.abs(), dy.abs()).reshape(cout, 9 * cin) + before.abs().double())
    assert ((got.double() - want).abs() <= bound).all(), ((got.double() - want).abs() / bound).max()


def test_infinity_reaches_the_weights_it_multiplies():
    x, dy = _inputs(1, 10, 16, 16, 16, 3)
    x[0, 9, 4, 5] = float("inf")  # the last image row: no output row below multiplies it by the tap above
    got = surrogate.conv3x3_weight_grad(x, dy).view(16, 9, 16)
    bad = ~got.isfinite()
    assert bad[:, 3:, 5].all() and not bad[:, :3].any() and not bad[:, :, :5].any() and not bad[:, :, 6:].any()
