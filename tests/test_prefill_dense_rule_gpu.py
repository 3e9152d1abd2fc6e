"""Prompt chunks of 1024 to 4095 rows whose fused tiles (256 rows x 128 outputs) are just too many for one round over the 256 CUs: they take the
dense GEMM on a dequantised image (csrc/kernels.h: dense_fills_chip).  Tile edges in rows and outputs, contractions of 2 to 20 K tiles, both types, with bias, through
the module path and through the C entry with scratch.  Reference: float64; tolerance: weights and result are rounded to the activation type
once each, 2^-8 (bf16) / 2^-11 (fp16): of the result, and of each of K independent terms."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k,bits,g,bias", [(1025, 6660, 128, 4, 64, False), (2817, 2820, 512, 3, 32, True), (3001, 3072, 1280, 2, 128, True), (4095, 2180, 256, 4, 128, False)])
def test_rows_outputs_and_contractions(dt, m, n, k, bits, g, bias):
    from gbx_lm_amd import _lib, ops
    rows = (m + 255) // 256
    assert rows * ((n + 255) // 256) < 176 and rows * ((n + 127) // 128) > 256 and 31 <= _lib.lib().gbx_qlinear_kernel_id(m, n, k, bits, g, 1) <= 33
    gen = torch.Generator(device=DEV).manual_seed(m + n)
    qw = torch.randint(-2**31, 2**31, (n, k // 32 * bits), device=DEV, generator=gen, dtype=torch.int64).to(torch.int32).view(torch.uint32)
    top = (1 << bits) - 1
    s = (torch.rand((n, k // g), device=DEV, generator=gen) + 0.5) * (0.04 / top)
    z, s = (-s * top / 2 + torch.randn(s.shape, device=DEV, generator=gen) * 0.1 * s).to(dt), s.to(dt)
    x = torch.randn((m, k), device=DEV, generator=gen).to(dt)
    b = (torch.randn(n, device=DEV, generator=gen) * 0.1).to(dt) if bias else None
    w = ops.unpack(qw, bits).double() * s.double().repeat_interleave(g, 1) + z.double().repeat_interleave(g, 1)
    want, spread = x.double() @ w.t(), (x.double() ** 2 @ (w ** 2).t()).sqrt()
    if bias:
        want = want + b.double()
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    room = 3 * eps * (want.abs() + spread + (b.double().abs() if bias else 0.0)) + 1e-6
    y = ops.quantized_matmul(x, qw, s, z, group_size=g, bits=bits, bias=b)
    assert bool(((y.double() - want).abs() <= room).all())
    L, out = _lib.lib(), torch.empty_like(y)
    need = L.gbx_qlinear_workspace_bytes(m, n, k, bits, g)
    ws = torch.empty((need,), dtype=torch.uint8, device=DEV)
    _lib.check(L.gbx_qlinear_forward_ws(x.data_ptr(), qw.data_ptr(), s.data_ptr(), z.data_ptr(), None if b is None else b.data_ptr(), out.data_ptr(), m, n, k, bits, g,
                                        ops._DT[dt], ws.data_ptr(), need, ops._stream_ptr(x.device)))
    assert torch.equal(out, y)
