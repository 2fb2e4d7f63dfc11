"""Layers without gradients just below and above the size at which their
weights are rounded beforehand equal the recorded ones."""

import pytest
import torch

from ggems_amd import surrogate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,cout,below,above", [
    (192, 64, (1, 152, 128), (1, 153, 128)),
    (16, 16, (29, 126, 256), (29, 127, 256)),
    (128, 128, (1, 28, 512), (1, 30, 512)),
])
def test_both_sides_of_the_rule(cin, cout, below, above):
    g = torch.Generator("cuda").manual_seed(cin)
    layer = surrogate.Conv3x3(cin, cout).cuda()
    for shape, few in ((below, True), (above, False)):
        assert (shape[0] * shape[1] * shape[2] * cin * cout <= surrogate.F32W_PRODUCTS) == few
        x = torch.randn(*shape, cin, device="cuda", generator=g).to(torch.bfloat16)
        want = layer(x).detach()
        with torch.no_grad():
            assert torch.equal(layer(x), want)
