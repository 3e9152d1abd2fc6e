"""Quantised products of 2 to 32 rows whose rows stay in registers (csrc/mfma_slab_impl.h): one and two row tiles, one to four chunks a wave and waves
without any, workgroups of one tile and of as many as their sums' place holds, more than one round of workgroups, several matrices in a launch.
Reference: float64; tolerance: the result's roundings and fp32 sums of K terms as large as C + q = 143 (bf16) or 1039 (fp16)."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def layer(n, k, bits, g, dt, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    qw = torch.randint(-2**31, 2**31, (n, k // 32 * bits), device=DEV, generator=gen, dtype=torch.int64).to(torch.int32).view(torch.uint32)
    top = (1 << bits) - 1
    s = (torch.rand((n, k // g), device=DEV, generator=gen) + 0.5) * (0.1 / top)
    z = (-s * top / 2 + torch.randn(s.shape, device=DEV, generator=gen) * 0.2 * s).to(dt)
    return SimpleNamespace(qweight=qw, scales=s.to(dt), zeros=z, bias=None, bits=bits, group_size=g, input_dims=k, output_dims=n)


def exact(x, m):
    """(product in float64, sum of the magnitudes of the terms as they are multiplied)"""
    from gbx_lm_amd import ops
    s = m.scales.double().repeat_interleave(m.group_size, 1)
    w = ops.unpack(m.qweight, m.bits).double() * s + m.zeros.double().repeat_interleave(m.group_size, 1)
    return x.double() @ w.t(), x.double().abs() @ (s * (144 if x.dtype == torch.bfloat16 else 1040)).t()


def rows(m, k, dt, seed):
    return torch.randn((m, k), device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed)).to(dt)


def eps_of(dt):
    return 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11


@pytest.mark.parametrize("m,n,k,bits,g,dt", [
    (2, 16, 1024, 4, 128, torch.bfloat16),         # one tile, one chunk a wave
    (16, 17, 1152, 3, 64, torch.float16),          # nine chunks: the fifth wave has one, three have none
    (17, 250, 2944, 2, 32, torch.bfloat16),        # 23 chunks, a last tile of ten outputs
    (32, 4104, 4096, 4, 32, torch.float16),        # four chunks a wave
    (31, 999, 3968, 3, 128, torch.bfloat16),
    (32, 32784, 1024, 2, 64, torch.bfloat16),      # 2049 tiles: eight a workgroup and a second round
    (16, 65541, 1024, 3, 32, torch.bfloat16),      # sixteen a workgroup and a second round
])
def test_tiles_and_chunks(m, n, k, bits, g, dt):
    from gbx_lm_amd import ops
    l, x = layer(n, k, bits, g, dt, n + k), rows(m, k, dt, m)
    y = ops.quantized_matmul(x, l.qweight, l.scales, l.zeros, group_size=g, bits=bits)
    want, terms = exact(x, l)
    assert bool(((y.double() - want).abs() <= eps_of(dt) * want.abs() + 2.0 ** -22 * terms).all())


def test_several_matrices_in_a_launch():
    from gbx_lm_amd import ops
    for m, ns, k, bits in ((17, (4096, 1024, 1024), 2048, 2), (8, (96, 32, 64), 1024, 4), (32, (64, 4128), 3072, 3)):
        ls, x = [layer(n, k, bits, 128, torch.bfloat16, n + i) for i, n in enumerate(ns)], rows(m, k, torch.bfloat16, m)
        for l, y in zip(ls, ops.quantized_matmul_multi(x, ls)):
            want, terms = exact(x, l)
            assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -22 * terms).all())


@pytest.mark.parametrize("m", [33, 34, 49, 64])
@pytest.mark.parametrize("n,k,bits,g", [(24576, 1024, 2, 128), (24592, 2048, 4, 128), (24600, 1024, 2, 32)])
def test_a_row_does_not_depend_on_its_place(m, n, k, bits, g):
    """More than 32 rows of a wide product go in two launches: the last row comes out as it does among the first."""
    from gbx_lm_amd import ops
    l, x = layer(n, k, bits, g, torch.bfloat16, n), rows(m, k, torch.bfloat16, m)
    y = ops.quantized_matmul(x, l.qweight, l.scales, l.zeros, group_size=g, bits=bits)
    want, terms = exact(x, l)
    assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -22 * terms).all())
    assert torch.equal(ops.quantized_matmul(x[m - 32:].contiguous(), l.qweight, l.scales, l.zeros, group_size=g, bits=bits), y[m - 32:])
