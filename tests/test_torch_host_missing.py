"""The extension for torch GPU tensors (csrc/torch_host.cc) is an accelerator, not a condition: host
tensors never ask for it, and without it calls on GPU tensors go through ctypes, with a warning."""
import sys

import pytest
import torch

from atex_amd import nv_norms
from atex_amd.nv_norms import _capi


def _calls():
    x = torch.randn(3, 4, 5, 8, requires_grad=True)
    g, b = torch.ones(8), torch.zeros(8)
    y, m, r = nv_norms.fused_layer_norm_op(x, g, b, axis=[-1])
    nv_norms.fused_layer_norm_grad_op(y, x, g, m, r, axis=[-1])
    y, m, r = nv_norms.fused_instance_norm_op(x, g, b)
    nv_norms.fused_instance_norm_grad_op(y, x, g, m, r)
    for layer in (nv_norms.LayerNormalization(), nv_norms.InstanceNormalization()):
        layer(x).sum().backward()
    assert x.grad is not None


def test_host_tensors_do_not_ask_for_the_extension(monkeypatch):
    def refuse():
        raise AssertionError("a call on host tensors asked for the extension")

    monkeypatch.setattr(_capi, "torch_host", refuse)
    _calls()


def test_a_missing_extension_declines_every_call(monkeypatch):
    monkeypatch.setattr(_capi, "_host", None)
    monkeypatch.delattr(nv_norms, "_torch_host", raising=False)
    monkeypatch.setitem(sys.modules, "atex_amd.nv_norms._torch_host", None)
    with pytest.warns(RuntimeWarning, match="_torch_host.so is missing or does not load"):
        host = _capi.torch_host()
    assert host.layer_norm_fwd(1, 2, 3) is None and host.instance_norm_apply() is None
    assert _capi.torch_host() is host  # warned once


def test_host_tensors_beside_the_extension():
    """Where it is loaded for other calls: it declines these before it leaves a trace in a profile."""
    assert _capi.torch_host().__file__.endswith("_torch_host.so")
    _calls()
    x = torch.randn(6, 8)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as p:
        nv_norms.fused_layer_norm(x, torch.ones(8), torch.zeros(8))
    assert [e.name for e in p.events()].count("_FusedLayerNormFn") == 1
