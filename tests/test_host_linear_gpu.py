"""The native call of few packed rows (csrc/host_linear.cpp) against the general path of ops.quantized_matmul, over the forms that both take; what is not plain is left to that path."""
import pytest
import torch

from gbx_lm_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _layer(n, k, bits, group, dtype, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 32 * bits), generator=gen, device="cuda", dtype=torch.int64).to(torch.int32)
    return w, (torch.rand((n, k // group), generator=gen, device="cuda") * 0.02).to(dtype), (torch.randn((n, k // group), generator=gen, device="cuda") * 0.02).to(dtype)


def _general(monkeypatch, *a, **k):
    with monkeypatch.context() as m:
        m.setattr(ops, "_few_rows", lambda *a: None)
        return ops.quantized_matmul(*a, **k)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(256,), (1, 256), (2, 256), (33, 256), (1, 5, 256), (2, 3, 4, 256), (64, 256), (65, 256), (255, 256)])
@pytest.mark.parametrize("bits,group,bias", [(4, 128, False), (3, 64, True), (2, 32, False)])
def test_what_is_plain(monkeypatch, dtype, shape, bits, group, bias):
    w, s, z = _layer(96, 256, bits, group, dtype)
    b = torch.randn((96,), device="cuda").to(dtype) if bias else None
    x = torch.randn(shape, device="cuda").to(dtype)
    native = _lib.host().few_rows(x, w, s, z, group, bits, b)
    assert isinstance(native, torch.Tensor) and not native.requires_grad
    want = _general(monkeypatch, x, w, s, z, group_size=group, bits=bits, bias=b)
    assert native.shape == want.shape == (*shape[:-1], 96) and native.dtype == want.dtype and torch.equal(native, want)
    assert torch.equal(native, ops.quantized_matmul(x, w.view(torch.uint32), s, z, group_size=group, bits=bits, bias=b))


def test_what_is_left_to_the_general_path(monkeypatch):
    dtype, few = torch.bfloat16, _lib.host().few_rows
    w, s, z = _layer(64, 256, 4, 64, dtype)
    x = torch.randn((4, 256), device="cuda", dtype=dtype)
    good = (x, w, s, z, 64, 4, None)
    assert isinstance(few(*good), torch.Tensor)

    class Other(torch.Tensor):
        pass

    wide = torch.randn((4, 512), device="cuda", dtype=dtype)[:, ::2]
    for at, value in ((0, x.float()), (0, x[:, :128].contiguous()), (0, wide), (0, x.cpu()), (0, x[:0]), (0, torch.randn((256, 256), device="cuda", dtype=dtype)), (0, x.as_subclass(Other)),
                      (1, w.float()), (1, w.cpu()), (1, w[:, :-1]), (1, w.reshape(-1)), (1, torch.cat([w, w], 1)[:, ::2]), (2, s.half()), (2, s[:-1]), (2, s.cpu()), (3, z.half()),
                      (3, z[:, :-1]), (4, 48), (4, 0), (4, True), (5, 5), (5, 0), (6, torch.zeros((63,), device="cuda", dtype=dtype)), (6, torch.zeros((64,), device="cuda"))):
        args = list(good)
        args[at] = value
        assert few(*args) is None, (at, value)
    for x_ in (wide, x.as_subclass(Other)):                           # taken there, with the same values
        assert torch.equal(ops.quantized_matmul(x_, w, s, z, group_size=64, bits=4).as_subclass(torch.Tensor), _general(monkeypatch, x_.as_subclass(torch.Tensor).contiguous(), w, s, z, group_size=64, bits=4))
    assert torch.equal(ops.quantized_matmul(x, w, s.half(), z, group_size=64, bits=4), _general(monkeypatch, x, w, s.half(), z, group_size=64, bits=4))
    with pytest.raises(ValueError):
        ops.quantized_matmul(x[:, :128].contiguous(), w, s, z, group_size=64, bits=4)
    from torch.utils._python_dispatch import TorchDispatchMode

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Watch():
        assert few(*good) is None
    seen = []
    torch.vmap(lambda v: seen.append(few(v, w, s, z, 64, 4, None)) or v)(torch.stack([x, x]))
    assert seen == [None]


def test_other_streams():
    w, s, z = _layer(4096, 4096, 4, 128, torch.bfloat16)
    x = torch.randn((1, 4096), device="cuda", dtype=torch.bfloat16)
    want = ops.quantized_matmul(x, w, s, z, group_size=128, bits=4)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        got = ops.quantized_matmul(x, w, s, z, group_size=128, bits=4)
    side.synchronize()
    assert torch.equal(got, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        held = ops.quantized_matmul(x, w, s, z, group_size=128, bits=4)
    for i in range(3):
        x.normal_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(held, ops.quantized_matmul(x, w, s, z, group_size=128, bits=4))


@pytest.mark.parametrize("rows,k", [(1, 256), (16, 4096), (40, 256), (100, 8192)])
def test_other_threads_run_during_a_launch(rows, k):
    """The launch is called without the interpreter's lock: a stand-in answers whether its thread holds it (0: no error, the call's result; 1: an error code)."""
    import ctypes
    L, host = _lib.lib(), _lib.host()
    w, s, z = _layer(64, k, 4, 64, torch.bfloat16)
    x = torch.randn((rows, k), device="cuda", dtype=torch.bfloat16)
    at = lambda f: ctypes.cast(f, ctypes.c_void_p).value
    holds = at(ctypes.pythonapi.PyGILState_Check)
    real = [at(f) for f in (L.gbx_qlinear_forward, L.gbx_qlinear_forward_ws, L.gbx_qlinear_workspace_bytes, L.gbx_qlinear_groups, L.gbx_qlinear_groups_win)]
    try:
        host.bind(holds, holds, real[2], holds, real[4])
        got = host.few_rows(x, w, s, z, 64, 4, None)
    finally:
        host.bind(*real)
    assert isinstance(got, torch.Tensor)
