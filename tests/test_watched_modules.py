"""Launches that stand in for several modules' calls (q, k and v of a prompt, a rotation with its cache update, experts with their weighted sum) leave a module that something
watches or replaces to its own call.  Tensors that say they live on the device stand in for such a device's; nothing here runs a kernel."""
import pytest
import torch
from torch import nn

from gbx_lm_amd import ops
from gbx_lm_amd.models import base, switch_layers
from gbx_lm_amd.models.cache import KVCache
from gbx_lm_amd.models.quantized_linear_gba import QuantizedLinear
from gbx_lm_amd.models.rope_utils import Llama3RoPE, RoPE
from gbx_lm_amd.models.switch_layers import QuantizedSwitchLinear, SwitchGLU


class OnDevice(torch.Tensor):
    """A host tensor that says it is the GPU's (results of operations on it say so too)."""
    is_cuda = property(lambda self: True)


def dev(t):
    return t.as_subclass(OnDevice)


def bf16(*shape):
    return torch.randn(*shape).bfloat16()


def seen_by(watch, module, answer, monkeypatch):
    """Puts ``watch`` over ``module``; the list it returns grows with every call of the module that the watcher sees.  ``answer``: what a forward in the place of the
    module's own returns."""
    calls = []
    note = lambda *a, **k: calls.append(1)
    hooks = {"hook": module.register_forward_hook, "hook before": module.register_forward_pre_hook,
             "hook on all": nn.modules.module.register_module_forward_hook, "hook before all": nn.modules.module.register_module_forward_pre_hook}
    if watch == "forward on the object":
        module.forward = lambda *a, **k: (note(), answer(*a, **k))[1]
    elif watch == "forward on the class":
        monkeypatch.setattr(type(module), "forward", lambda self, *a, **k: (note() if self is module else None, answer(*a, **k))[1])
    else:
        handle = hooks[watch](lambda m, *a: note() if m is module else None)
        monkeypatch.callbacks.append(handle.remove)
    return calls


@pytest.fixture
def patch(monkeypatch):
    monkeypatch.callbacks = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    yield monkeypatch
    for done in monkeypatch.callbacks:
        done()


WATCHES = ["forward on the object", "forward on the class", "hook", "hook before", "hook on all", "hook before all"]


def layer(n=64, k=256):
    m = QuantizedLinear(k, n, False, 64, 4)
    for name, t in dict(qweight=torch.zeros((n, k // 8), dtype=torch.int32), scales=bf16(n, k // 64), zeros=bf16(n, k // 64)).items():
        m._buffers[name] = dev(t)
    return m


@pytest.mark.parametrize("watch", WATCHES + ["compiled", "hook behind"])
@pytest.mark.parametrize("place", [0, 2])
def test_products_of_a_prompt(patch, watch, place):
    patch.setattr(ops, "_dense_image", lambda *a: pytest.fail("an image was asked for"))
    mods = [layer() for _ in range(3)]
    if watch == "compiled":
        mods[place]._compiled_call_impl = lambda x: x
    elif watch == "hook behind":
        mods[place].register_full_backward_hook(lambda *a: None)
    else:
        seen_by(watch, mods[place], lambda x: x, patch)
    assert ops.quantized_matmul_prompt(dev(bf16(1, 300, 256)), mods) is None


def test_products_of_a_prompt_that_nothing_watches_are_one_launch(patch):
    asked = []
    patch.setattr(ops, "_dense_image", lambda *a: asked.append(a))
    assert ops.quantized_matmul_prompt(dev(bf16(1, 300, 256)), [layer(), layer()]) is None and len(asked) == 1


@pytest.mark.parametrize("watch", ["none"] + WATCHES)
@pytest.mark.parametrize("which", ["experts", "down_proj"])
def test_experts_with_their_weighted_sum(patch, watch, which):
    experts = SwitchGLU(256, 256, 4)
    x, idx, scores = dev(bf16(1, 256)), dev(torch.zeros((1, 2), dtype=torch.int32)), bf16(1, 2)
    mixed = []
    patch.setattr(ops, "gather_mix", lambda *a: mixed.append(1) or torch.zeros(1, 256))
    patch.setattr(ops, "moe_combine", lambda y, s, r=None: y)
    patch.setattr(ops, "gather_quantized_matmul", lambda *a, **k: torch.zeros(1, 2, 1, 256))
    experts._activated = lambda x, indices: x
    if watch == "none":
        switch_layers.mixed_experts(experts, x, idx, scores)
        assert mixed == [1]
        return
    module = experts if which == "experts" else experts.down_proj
    assert type(module) in (SwitchGLU, QuantizedSwitchLinear)
    calls = seen_by(watch, module, lambda *a: torch.zeros(1, 2, 1, 256) if which == "down_proj" else torch.zeros(1, 2, 256), patch)
    switch_layers.mixed_experts(experts, x, idx, scores)
    assert calls == [1] and not mixed


@pytest.mark.parametrize("watch", ["none"] + WATCHES)
@pytest.mark.parametrize("kind", ["plain", "llama3"])
def test_rotation_with_its_cache_update(patch, watch, kind):
    rope = RoPE(64) if kind == "plain" else Llama3RoPE(64, scaling_config={"factor": 8.0})
    rope.inv_freq = dev(rope.inv_freq)
    q, k, v = (dev(bf16(1, h, 20, 64)) for h in (4, 2, 2))
    turned = []
    patch.setattr(ops, "rope_qkv", lambda *a: turned.append(1) or a[0])
    patch.setattr(ops, "rope", lambda x, *a: x)
    patch.setattr(ops, "rope_kv_write", lambda *a: None)
    cache = KVCache()
    if watch == "none":
        calls = []
    else:
        calls = seen_by(watch, rope, lambda x, offset=0: x, patch)
    base.rope_and_update_cache(rope, q, k, v, cache, 0)
    assert (calls, turned) == (([], [1]) if watch == "none" else ([1], [])) and cache.offset == 20
