"""When a routed layer hands its parts to the norm behind it, and when it is called."""
import torch

from nano_vllm_amd import ops_seq
from nano_vllm_amd.mixers import RoutedExperts, routed_output


def _layer():
    mlp = RoutedExperts(8, 4, 8, 2)
    parts = ("rows", "plan", "weights", "shared", "gate")
    mlp.parts = lambda h, *args: parts
    return mlp, parts


def test_parts_of_a_layer_as_it_is_made():
    mlp, parts = _layer()
    h = torch.zeros(3, 8)
    y = routed_output(mlp, h)
    assert type(y) is ops_seq.ChosenRows and y.h is h and (y.rows, y.plan, y.wts, y.shared, y.gate) == parts


def test_a_layer_that_is_watched_replaced_or_extended_is_called():
    h = torch.zeros(3, 8)
    for watch in ("hook", "pre-hook", "forward", "subclass", "global"):
        mlp, seen = _layer()[0], []
        handle = None
        if watch == "subclass":
            class Mine(RoutedExperts):
                def forward(self, xh, *args):
                    return xh + 1
            mlp = Mine(8, 4, 8, 2)
        else:
            mlp.forward = lambda xh, *args: xh + 1
        if watch != "forward" and watch != "subclass":
            # (the call itself needs a device: a class of its own would not be RoutedExperts, so the replaced call is put where the instance does not show it)
            del mlp.forward
            kept, RoutedExperts.forward = RoutedExperts.forward, lambda self, xh, *args: xh + 1
        try:
            if watch == "hook":
                mlp.register_forward_hook(lambda *a: seen.append(1))
            elif watch == "pre-hook":
                mlp.register_forward_pre_hook(lambda *a: seen.append(1))
            elif watch == "global":
                handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: seen.append(1))
            y = routed_output(mlp, h)
        finally:
            if handle is not None:
                handle.remove()
            if watch != "forward" and watch != "subclass":
                RoutedExperts.forward = kept
        assert torch.equal(y, h + 1) and (watch in ("forward", "subclass") or seen), watch


def test_a_call_that_is_replaced_in_the_class_is_made(monkeypatch):
    h = torch.zeros(3, 8)
    mlp, _ = _layer()
    monkeypatch.setattr(RoutedExperts, "forward", lambda self, xh, *args: xh + 1)
    assert torch.equal(routed_output(mlp, h), h + 1)
    monkeypatch.undo()
    assert type(routed_output(mlp, h)) is ops_seq.ChosenRows
    monkeypatch.setattr(torch.nn.Module, "__call__", lambda self, xh, *args: xh + 2)
    assert torch.equal(routed_output(mlp, h), h + 2)
