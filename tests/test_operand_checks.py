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
