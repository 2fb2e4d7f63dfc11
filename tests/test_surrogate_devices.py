"""A network and an input on different devices are refused before any kernel
is launched: a host pointer would fault the GPU.  So are parameters of another
shape than the kernels read, where tensor operations broadcast or refused
them.  The library is a recorder
and the GPU tensors are stand-ins, so nothing runs on a GPU here."""

import pytest
import torch

from ggems_amd import surrogate as S

GPU = torch.device("cuda", 0)


class OnGpu:
    """what the calls look at of a GPU tensor, over a CPU one"""

    def __init__(self, t):
        self.t, self.device, self.is_cuda = t, GPU, True
        self.shape, self.dtype, self.ndim = t.shape, t.dtype, t.ndim

    def get_device(self):
        return 0

    def contiguous(self):
        return self

    float = detach = contiguous

    def view(self, *shape):
        return OnGpu(self.t.view(*shape))

    def to(self, dtype):
        return OnGpu(self.t.to(dtype))

    def __getattr__(self, name):
        return getattr(self.t, name)


class Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *a: self.calls.append(name) or 0


@pytest.fixture
def launches(monkeypatch):
    lib, empty = Recorder(), torch.empty

    def on_cpu(*shape, device=None, **kw):
        t = empty(*shape, **kw)
        return t if device is None or device.type == "cpu" else OnGpu(t)

    monkeypatch.setattr(S, "_lib", lambda: lib)
    monkeypatch.setattr(S, "_stream", lambda t: 0)
    monkeypatch.setattr(torch, "empty", on_cpu)
    return lib.calls


def _tensors(gpu):
    def put(t):
        return OnGpu(t) if gpu else t
    return dict(w=put(torch.zeros(16, 9, 16)), b=put(torch.zeros(16)), head=put(torch.zeros(16)),
                bias=put(torch.zeros(1)))


CALLS = {
    "layer": lambda x, t: S._conv_layer(x, t["w"], t["b"], True),
    "layer without bias": lambda x, t: S._conv_layer(x, t["w"], None, True),
    "conv3x3": lambda x, t: S.conv3x3(x, t["w"].view(16, 144).to(torch.bfloat16), t["b"], True),
    "head": lambda x, t: S.head16(x, t["head"], t["bias"]),
}


@pytest.mark.parametrize("call", sorted(CALLS))
@pytest.mark.parametrize("here", ["w", "b", "head", "bias", "all"])
def test_host_parameters_are_refused_before_a_launch(launches, call, here):
    x = OnGpu(torch.zeros(1, 16, 16, 16, dtype=torch.bfloat16))
    host, t = _tensors(False), _tensors(True)
    t = host if here == "all" else dict(t, **{here: host[here]})
    used = {"layer": "wb", "layer without bias": "w", "conv3x3": "wb", "head": ("head", "bias")}[call]

    def run():
        CALLS[call](x, t)

    if here == "all" or here in used:
        with pytest.raises((S.EngineError, ValueError)):
            run()
        assert launches == []
    else:
        run()
        assert len(launches) == 1


def test_a_host_tensor_has_no_stream():
    with pytest.raises(ValueError):
        S._stream(torch.zeros(1))


@pytest.mark.parametrize("w,b", [((16, 7, 16), 16), ((16, 9, 16), 12), ((16, 1, 16), 16)])
def test_layers_of_other_shapes_do_not_reach_the_kernel(launches, w, b):
    x = OnGpu(torch.zeros(1, 16, 16, 16, dtype=torch.bfloat16))
    with pytest.raises((S.EngineError, RuntimeError)):
        S._conv_layer(x, OnGpu(torch.zeros(w)), OnGpu(torch.zeros(b)), True)
    assert not [c for c in launches if c.startswith("ggh_conv3x3_forward")]


@pytest.mark.parametrize("head,bias,fits", [((16,), (1,), True), ((1,), (1,), False), ((16,), (), False),
                                            ((16,), (16,), False), ((1, 16), (1,), False)])
def test_head_shapes_that_broadcast_take_the_tensor_operations(launches, head, bias, fits):
    z = OnGpu(torch.zeros(1, 16, 16, 16, dtype=torch.bfloat16))
    head, bias = OnGpu(torch.zeros(head)), OnGpu(torch.zeros(bias))
    assert S._fits_head16(z, head, bias) == fits
    if fits:
        S.head16(z, head, bias)
        return
    with pytest.raises(S.EngineError):
        S.head16(z, head, bias)
    assert launches == []
