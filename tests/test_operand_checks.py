"""Operands that a kernel cannot take are met before any launch: the call raises, or goes the way on which torch or the general path
refuses it.  Tensors that say they live on the device stand in for such a device's and every launch is a failure, so nothing here runs a kernel."""
import pytest
import torch

from gbx_lm_amd import _lib, mixer_ops as M, ops


class _NoLaunch:
    """A library whose size queries answer and whose launches fail the test."""

    def __getattr__(self, name):
        if name.endswith(("_workspace", "_workspace_bytes")):
            return lambda *a: 1 << 20

        def launch(*a):
            raise AssertionError(f"{name} was reached")
        return launch


@pytest.fixture
def no_launch(monkeypatch):
    lib = _NoLaunch()
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    monkeypatch.setattr(_lib, "mixers", lambda: lib)
    monkeypatch.setattr(ops, "_stream_ptr", lambda device: 0)
    monkeypatch.setattr(M, "_stream", lambda device: 0)


def bf16(*shape):
    return torch.randn(*shape).bfloat16()


def test_only_devices_have_streams(monkeypatch):
    """A host tensor that reaches a launch is refused there, as torch's own lookup of a current stream refuses it."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 7, raising=False)
    for name in ("cpu", torch.device("cpu"), torch.device("meta")):
        for lookup in (ops._stream_ptr, M._stream):
            with pytest.raises(ValueError, match="cuda device"):
                lookup(name)
    for name in ("cuda:0", "cuda", torch.device("cuda", 1)):
        assert ops._stream_ptr(name) == M._stream(name) == 7


@pytest.mark.parametrize("bias", [bf16(47), bf16(49), bf16(1), bf16(48, 1), torch.empty(48, dtype=torch.bfloat16, device="meta")],
                         ids=["short", "long", "one", "column", "other device"])
def test_row_products_leave_other_biases_to_torch(no_launch, bias):
    """A bias that is not one value per output on the rows' device."""
    assert M.linear_rows(bf16(4, 256), bf16(48, 256), bias) is None


@pytest.mark.parametrize("x,w", [((4, 256), (0, 256)), ((4, 0), (48, 0)), ((4, 256), (256,)), ((2, 4, 256), (48, 256)), ((256,), (48, 256)), ((4, 256), (2, 48, 256))])
def test_row_products_leave_other_shapes_to_torch(no_launch, x, w):
    assert M.linear_rows(bf16(*x), bf16(*w), None) is None


class OnDevice(torch.Tensor):
    """A host tensor that says it is the GPU's (results of operations on it say so too)."""
    is_cuda = property(lambda self: True)


def dev(t):
    return t.as_subclass(OnDevice)


ROUTERS = [lambda h, r: M.route_topk(h, r, 2), lambda h, r: M.route_sigmoid_groups(h, r, torch.zeros(8), 2, None, False, 1.0),
           lambda h, r: M.route_groups(h, r, 8, 2, None)]


@pytest.mark.parametrize("route", ROUTERS, ids=["softmax", "sigmoid", "groups"])
def test_routers_on_other_devices_and_rows_of_other_ranks_raise(no_launch, route):
    router = torch.randn(8, 64)
    with pytest.raises((RuntimeError, ValueError)):
        route(dev(torch.randn(4, 64)), router.to("meta"))
    for h in (torch.randn(64), torch.randn(4, 64, 64), torch.randn(4, 32)):
        with pytest.raises((RuntimeError, ValueError, IndexError)):
            route(dev(h), router)


def experts(e=6, n=64, k=256, g=64, bits=4, dt=torch.bfloat16):
    from gbx_lm_amd.models.switch_layers import QuantizedSwitchLinear
    m = QuantizedSwitchLinear(k, n, e, bias=False, group_size=g, bits=bits)
    qw = torch.zeros((e, n, k // 32 * bits), dtype=torch.int32)
    m._buffers["qweight"], m._buffers["scales"], m._buffers["zeros"] = dev(qw), dev(torch.ones(e, n, k // g).to(dt)), dev(torch.zeros(e, n, k // g).to(dt))
    return m


def changed(m, **buffers):
    for name, t in buffers.items():
        m._buffers[name] = dev(t)
    return m


X, IDX = (100, 1, 1, 256), (torch.arange(100) % 6).to(torch.int32)[:, None]
GATED = {
    "rows in 32 bits": lambda: (dev(torch.randn(X)), experts(dt=torch.float32), IDX),
    "other leading sizes": lambda: (dev(bf16(90, 1, 1, 256)), experts(), IDX),
    "one row for all": lambda: (dev(bf16(1, 1, 1, 256)), experts(), IDX),
    "leading sizes in another order": lambda: (dev(bf16(50, 2, 1, 1, 256)), experts(), IDX.view(2, 50, 1)),
    "too few experts": lambda: (dev(bf16(*X)), changed(experts(), qweight=torch.zeros(5, 64, 32, dtype=torch.int32)), IDX),
    "too few outputs": lambda: (dev(bf16(*X)), changed(experts(), qweight=torch.zeros(6, 60, 32, dtype=torch.int32)), IDX),
    "too few groups": lambda: (dev(bf16(*X)), changed(experts(), scales=bf16(6, 64, 2)), IDX),
    "zeros of another shape": lambda: (dev(bf16(*X)), changed(experts(), zeros=bf16(6, 64, 2)), IDX),
    "words of another type": lambda: (dev(bf16(*X)), changed(experts(), qweight=torch.zeros(6, 64, 32)), IDX),
    "indices that are no integers": lambda: (dev(bf16(*X)), experts(), IDX.float()),
    "indices on the host": lambda: (dev(bf16(*X)), experts(), IDX),
    "weights on the host": lambda: (dev(bf16(*X)), experts(), IDX),
}


@pytest.mark.parametrize("name", list(GATED))
def test_gated_experts_leave_what_they_cannot_take_to_the_separate_products(no_launch, name):
    x, m, idx = GATED[name]()
    if name == "weights on the host":
        m._buffers["scales"] = m.scales.as_subclass(torch.Tensor)
    assert ops.gather_swiglu(x, m, m, idx if name == "indices on the host" else dev(idx)) is None


def test_gated_experts_of_fitting_operands_reach_the_launch(no_launch, monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    with pytest.raises(AssertionError, match="gbxm_packed_experts was reached"):
        ops.gather_swiglu(dev(bf16(*X)), experts(), experts(), dev(IDX))


@pytest.mark.parametrize("name", ["too few groups", "zeros of another shape", "words of another type", "short bias", "wide bias", "bias on the host", "indices that are no integers"])
def test_experts_of_many_pairs_leave_what_they_cannot_take_to_one_expert_at_a_time(no_launch, monkeypatch, name):
    """... whose products refuse it."""
    x, m, idx = GATED[name]() if name in GATED else (dev(bf16(*X)), experts(), IDX)
    bias = {"short bias": dev(bf16(6, 32)), "wide bias": dev(bf16(6, 65)), "bias on the host": bf16(6, 64)}.get(name)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    with pytest.raises((ValueError, RuntimeError, TypeError, IndexError)):
        ops.gather_quantized_matmul(x, m.qweight, m.scales, m.zeros, dev(idx), group_size=64, bits=4, bias=bias)


def packed_layer(n=64, k=256, g=64, bits=4, **buffers):
    """A packed layer whose buffers say that they are the GPU's; ``buffers`` take the places of those that fit it."""
    from gbx_lm_amd.models.quantized_linear_gba import QuantizedLinear
    m = QuantizedLinear(k, n, "bias" in buffers, g, bits)
    fits = dict(qweight=torch.zeros((n, k // 32 * bits), dtype=torch.int32), scales=bf16(n, k // g), zeros=bf16(n, k // g))
    for name, t in {**fits, **buffers}.items():
        m._buffers[name] = t if t is None else dev(t)
    return m


MISFITS = {
    "too few outputs": dict(qweight=torch.zeros((60, 32), dtype=torch.int32)),
    "too few words": dict(qweight=torch.zeros((64, 24), dtype=torch.int32)),
    "words of another type": dict(qweight=torch.zeros((64, 32))),
    "words of 64 bits": dict(qweight=torch.zeros((64, 32), dtype=torch.int64)),
    "too few groups": dict(scales=bf16(64, 2)),
    "scales of too few outputs": dict(scales=bf16(32, 4), zeros=bf16(32, 4)),
    "zeros of another shape": dict(zeros=bf16(64, 2)),
    "scales of one rank": dict(scales=bf16(256)),
    "scales of another type": dict(scales=torch.randn(64, 4)),
    "no zeros": dict(zeros=None),
    "words on another device": dict(qweight=torch.zeros((64, 32), dtype=torch.int32, device="meta")),
    "scales on another device": dict(scales=torch.empty((64, 4), dtype=torch.bfloat16, device="meta")),
    "short bias": dict(bias=bf16(32)),
    "long bias": dict(bias=bf16(65)),
    "column as bias": dict(bias=bf16(64, 1)),
    "bias on another device": dict(bias=torch.empty((64,), dtype=torch.bfloat16, device="meta")),
}


@pytest.mark.parametrize("rows", [300, 1024])
@pytest.mark.parametrize("name", list(MISFITS))
def test_products_of_a_prompt_leave_misfits_to_each_layer(no_launch, monkeypatch, name, rows):
    """q, k and v together: a layer that does not hold what its sizes say is left to its own call, which refuses it."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(ops._dense_cache, "get", lambda *a: pytest.fail("an image was asked for") if "bias" not in name else torch.empty(0))
    mods = [packed_layer(**MISFITS[name]), packed_layer(), packed_layer()]
    assert ops.quantized_matmul_prompt(dev(bf16(1, rows, 256)), mods) is None


def test_products_of_a_prompt_of_fitting_layers_ask_for_their_images(no_launch, monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    asked = []
    monkeypatch.setattr(ops._dense_cache, "get", lambda src, key: asked.append(key))
    for mods in ([packed_layer(), packed_layer()], [packed_layer(bias=bf16(64)), packed_layer()], [packed_layer(bits=3), packed_layer()]):
        assert ops.quantized_matmul_prompt(dev(bf16(1, 300, 256)), mods) is None      # nothing is resident
    assert [key[2] for key in asked] == [4, 4, 3]
    with pytest.raises(AssertionError, match="was reached"):
        ops.quantized_matmul_prompt(dev(bf16(1, 1024, 256)), [packed_layer(), packed_layer()])


@pytest.mark.parametrize("rows", [1, 300, 1024])
@pytest.mark.parametrize("dt", [torch.float32, torch.float64, torch.int32])
def test_activations_of_a_packed_product_are_16_bits(no_launch, monkeypatch, rows, dt):
    """... and nothing is converted or allocated for others."""
    monkeypatch.setattr(torch, "empty", lambda *a, **k: pytest.fail("allocated"))
    w, s = dev(torch.zeros(64, 32, dtype=torch.int32)), dev(torch.ones(64, 4).bfloat16())
    with pytest.raises(ValueError, match="float16 or bfloat16"):
        ops.quantized_matmul(dev(torch.ones(rows, 256, dtype=dt)), w, s, s, group_size=64, bits=4)
