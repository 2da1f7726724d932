"""Linear layers of many rows whose caller asks for more than the result: derivatives forward and backward, a map over the call, a dispatch mode, autocast, a subclass. The
tiles' kernel gives none of these, so such calls are the library's."""
from types import SimpleNamespace

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def layer(w, b=None):
    from nano_vllm_amd.layers import LinearBase
    return lambda x: LinearBase.forward(SimpleNamespace(weight=w, bias=b, weight_packed=None), x)


@pytest.fixture
def xw():
    from nano_vllm_amd import ops_seq
    ops_seq.load_library()
    x, w = torch.randn(3000, 256).bfloat16().cuda(), (torch.randn(4096, 256) / 16).bfloat16().cuda()
    with torch.no_grad():
        assert ops_seq.many_rows(x, w)
    return x, w


def both(w):
    from nano_vllm_amd import ops_seq
    return layer(w), lambda x: ops_seq.linear(x, w)


def test_forward_mode_keeps_its_tangent(xw):
    import torch.autograd.forward_ad as fw
    x, w = xw
    t = torch.randn_like(x)
    for f in both(w):
        with torch.no_grad(), fw.dual_level():
            y = fw.unpack_dual(f(fw.make_dual(x, t)))
            assert y.tangent is not None and torch.equal(y.tangent, F.linear(t, w)) and torch.equal(y.primal, F.linear(x, w))
        with torch.no_grad():
            assert torch.equal(torch.func.jvp(f, (x,), (t,))[1], F.linear(t, w))


def test_backward_has_a_gradient(xw):
    x, w = xw
    for f in both(w):
        leaf = x.clone().requires_grad_()
        f(leaf).sum().backward()
        assert leaf.grad is not None


@torch.no_grad()
def test_mapped_calls(xw):
    x, w = xw
    xs = torch.stack([x, x + 1])
    got = torch.func.vmap(layer(w))(xs)
    # the same sums of 256 products in another order, rounded to 8 bits
    assert float((got.double() - F.linear(xs.double(), w.double())).norm() / got.double().norm()) <= 2.0 ** -8


@torch.no_grad()
def test_dispatch_modes_see_the_product(xw):
    from torch.utils._python_dispatch import TorchDispatchMode
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))
    x, w = xw
    for f in both(w):
        seen.clear()
        with Watch():
            f(x)
        assert any(name.startswith(("aten.mm", "aten.linear", "aten.addmm")) for name in seen), seen


@torch.no_grad()
def test_autocast_chooses_the_type(xw):
    x, w = xw
    for f in both(w):
        with torch.autocast("cuda", dtype=torch.float16):
            assert f(x).dtype == torch.float16


@torch.no_grad()
def test_subclasses_stay_themselves(xw):
    class Tagged(torch.Tensor):
        pass
    x, w = xw
    assert isinstance(layer(w)(x.as_subclass(Tagged)), Tagged)


@torch.no_grad()
def test_a_subclass_as_the_bias_is_asked_too(xw):
    class Tagged(torch.Tensor):
        pass
    x, w = xw
    b = torch.randn(w.shape[0]).bfloat16().cuda()
    assert isinstance(layer(w, b.as_subclass(Tagged))(x), Tagged) and type(layer(w, b)(x)) is torch.Tensor


@torch.no_grad()
def test_tensors_of_another_device_than_the_launches(xw, monkeypatch):
    from nano_vllm_amd import ops_seq
    x, w = xw
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert not ops_seq.many_rows(x, w)


def test_plain_calls_are_the_tiles(xw, monkeypatch):
    from nano_vllm_amd import ops_seq
    x, w = xw
    calls, tiles = [], ops_seq.linear_tiles
    monkeypatch.setattr(ops_seq, "linear_tiles", lambda *a: calls.append(a) or tiles(*a))
    for mode in (torch.no_grad, torch.inference_mode):
        with mode():
            for f in both(torch.nn.Parameter(w)):
                f(x)
    assert len(calls) == 4
