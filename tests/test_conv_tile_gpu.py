"""The tile convolution against the general kernels, bit for bit: the same
call with an output that is not 8-byte aligned takes the general ones.  Every
channel count the tile kernel has, images whose height ends inside a tile or
is less than one, one pixel tile and many, channel tiles in one block and in
several, with split sums and without, Inf and NaN inputs."""

import pytest
import torch

from ggems_amd import surrogate

pytestmark = pytest.mark.gpu


def _forward(x, w, bias, y, relu):
    n, h, wd, cin = x.shape
    cout = w.shape[0]
    surrogate._check(surrogate._lib().ggh_conv3x3_forward(
        x.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), y.data_ptr(), n, h, wd, cin, cout,
        int(relu), surrogate._stream(x)))


def _both(n, h, wd, cin, cout, bias, relu, special=False):
    g = torch.Generator("cuda").manual_seed(cin * cout + h)
    x = torch.randn(n, h, wd, cin, device="cuda", generator=g).to(torch.bfloat16)
    w = torch.randn(cout, 9 * cin, device="cuda", generator=g).to(torch.bfloat16)
    if special:
        x[0, 0, 0, 0], x[0, h - 1, wd - 1, cin - 1], x[0, 0, wd // 2, cin - 1] = float("inf"), float("nan"), -3e38
    b = torch.randn(cout + 1, device="cuda", generator=g)[1:] if bias else None  # not 16-byte aligned
    got = torch.empty(n, h, wd, cout, device="cuda", dtype=torch.bfloat16)
    store = torch.empty(got.numel() + 1, device="cuda", dtype=torch.bfloat16)
    want = store[1:].view(got.shape)
    assert got.data_ptr() % 8 == 0 and want.data_ptr() % 8 != 0
    _forward(x, w, b, got, relu)
    _forward(x, w, b, want, relu)
    return got, want


@pytest.mark.parametrize("cin", [8, 16, 32, 48, 64, 96, 128, 192])
@pytest.mark.parametrize("n,h,wd,cout,bias,relu", [
    (1, 2, 16, 16, True, True),        # less than a tile
    (2, 9, 32, 48, False, True),       # a tile's last row alone
    (1, 16, 48, 80, True, False),      # five channel tiles
    (3, 23, 32, 64, True, True),
    (16, 64, 80, 96, True, True),      # many tiles: channel tiles in one block
])
def test_tile_equals_general(n, h, wd, cin, cout, bias, relu):
    got, want = _both(n, h, wd, cin, cout, bias, relu)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("cin", [16, 64])
def test_inf_and_nan_stay_where_they_reach(cin):
    got, want = _both(1, 16, 32, cin, 32, True, False, special=True)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert want.isnan().any() and want.isfinite().float().mean() > 0.9
    fine = want.isfinite()
    assert torch.equal(got[fine], want[fine])
