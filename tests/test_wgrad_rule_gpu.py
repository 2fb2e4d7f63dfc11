"""The weight gradient without a work space, on both sides of the line between
its kernels and at block counts from one tile a block to many, against the
sums that go through a work space."""

import pytest
import torch

from ggems_amd import surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,cin,cout", [
    (1, 8, 16, 16, 16), (4, 64, 64, 64, 16), (4, 64, 80, 64, 16),   # 1, 128 and 160 tiles
    (1, 128, 128, 96, 32), (1, 130, 128, 96, 32),                   # 128 and 136, the last rows past the image
    (1, 64, 64, 16, 64), (2, 32, 32, 128, 128), (3, 40, 48, 256, 128),
    (2, 256, 256, 8, 16), (6, 192, 256, 48, 16),
])
def test_sums_of_blocks_and_of_a_work_space(n, h, w, cin, cout):
    g = torch.Generator("cuda").manual_seed(cin + cout)
    x = torch.randn(n, h, w, cin, device="cuda", generator=g).to(torch.bfloat16)
    dy = torch.randn(n, h, w, cout, device="cuda", generator=g).to(torch.bfloat16)
    _, want, _ = surrogate.conv3x3_backward(x, None, dy, x, False, None)
    got = surrogate.conv3x3_weight_grad(x, dy)
    # FP32 sums of the same products in another order: 16 ulps of the sum of magnitudes
    size = surrogate.conv3x3_weight_grad(x.abs(), dy.abs())
    assert ((got - want).abs() <= 1e-6 * size).all()
    out = torch.ones(cout, 9 * cin, device="cuda")  # added to what is there
    surrogate.conv3x3_weight_grad(x, dy, out=out)
    assert ((out - 1 - got).abs() <= 1e-6 * (size + 1)).all()
