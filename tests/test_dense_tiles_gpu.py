"""The dense GEMM's tiles of 192 (csrc/mfma_dense.hip: gemm_dense_shape): sizes for which each of the four shapes takes least, their ragged last rows and columns, a bias, and
gate and up.  Reference: float64; tolerance: fp32 sums of K products (K 2^-24 of their magnitudes) and the result's roundings."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(3001, 5120, 64),       # 256 x 256
                                   (2048, 6140, 128),      # 256 x 192, columns off the grid of 16 bytes
                                   (6000, 4090, 192),      # 192 x 256
                                   (3001, 3072, 320), (2900, 3001, 64), (193, 3073, 1024), (1, 200, 64)])       # 192 x 192
def test_every_shape_and_its_edges(dt, m, n, k):
    from gbx_lm_amd import _lib, ops
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    x, w = (torch.randn(s, device=DEV, generator=gen).to(dt) for s in ((m, k), (n, k)))
    bias = torch.randn(n, device=DEV, generator=gen).to(dt)
    want, terms = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    for b in (None, bias):
        y = torch.empty((m, n), dtype=dt, device=DEV)
        _lib.check(_lib.lib().gbx_dense_forward_ws(x.data_ptr(), w.data_ptr(), None if b is None else b.data_ptr(), y.data_ptr(), m, n, k, ops._DT[dt], None, 0,
                                                   torch.cuda.current_stream().cuda_stream))
        full = want if b is None else want + b.double()
        room = EPS[dt] * (full.abs() + (0.0 if b is None else want.abs())) + k * 2.0 ** -24 * terms
        assert bool(((y.double() - full).abs() <= room).all())


@pytest.mark.parametrize("m,n,k", [(1100, 14336, 64), (5000, 2560, 128)])       # 192 x 256 and 256 x 256
def test_gate_and_up(m, n, k):
    from gbx_lm_amd import _lib, ops
    gen = torch.Generator(device=DEV).manual_seed(m)
    dt = torch.bfloat16
    x, gate, up = (torch.randn(s, device=DEV, generator=gen).to(dt) for s in ((m, k), (n, k), (n, k)))
    w = torch.stack([gate.view(-1, 128, k), up.view(-1, 128, k)], 1).reshape(2 * n, k).contiguous()
    y = torch.empty((m, n), dtype=dt, device=DEV)
    _lib.check(_lib.lib().gbx_dense_swiglu_forward(x.data_ptr(), w.data_ptr(), y.data_ptr(), m, n, k, ops._DT[dt], torch.cuda.current_stream().cuda_stream))
    a, b = x.double() @ gate.double().t(), x.double() @ up.double().t()
    s = torch.nn.functional.silu(a)
    room = EPS[dt] * (2 * (s * b).abs() + 1.1 * a.abs() * b.abs() + s.abs() * b.abs()) * 1.02 + 1e-3        # roundings of gate, up, silu (whose slope is at most 1.1) and product
    assert bool(((y.double() - s * b).abs() <= room).all())
