"""Experts of a few (token, slot) pairs, rows of one slot a lane (gbx_gather_qlinear_forward, gbx_gather_swiglu_forward): rows of one to 64 slots, row counts that end
inside a wave's share, every bit width, group and type, a bias; against float64, and gate | up against its own three operations."""
import numpy as np
import pytest
import torch

from gbx_lm_amd import ops
from gbx_lm_amd.models.switch_layers import QuantizedSwitchLinear

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(E, N, K, bits, group, dt, seed, bias=False):
    gen = torch.Generator().manual_seed(seed)
    m = QuantizedSwitchLinear(K, N, E, bias=False, group_size=group, bits=bits)
    top = float((1 << bits) - 1)
    s = (torch.rand((E, N, K // group), generator=gen) + 0.5) * (0.04 / top)
    m.qweight = torch.randint(-2 ** 31, 2 ** 31 - 1, (E, N, K // 32 * bits), generator=gen, dtype=torch.int64).to(torch.int32).view(torch.uint32).to(DEV)
    m.scales, m.zeros = s.to(dt).to(DEV), (-s * top / 2).to(dt).to(DEV)
    m.bias = torch.randn((E, N), generator=gen).to(dt).to(DEV) if bias else None
    return m


def _dense(m):
    w = np.pad(m.qweight.cpu().view(torch.int32).numpy().view(np.uint32).astype(np.uint64), ((0, 0), (0, 0), (0, 1)))
    at = np.arange(m.input_dims) * m.bits
    q = ((w[..., at // 32] | (w[..., at // 32 + 1] << np.uint64(32))) >> (at % 32).astype(np.uint64)) & np.uint64((1 << m.bits) - 1)
    s, z = (t.double().cpu().numpy().repeat(m.group_size, -1) for t in (m.scales, m.zeros))
    return torch.from_numpy(q.astype(np.float64) * s + z)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,group,K", [(2, 32, 128), (2, 64, 2048), (2, 128, 2176), (2, 32, 4096), (3, 32, 128), (3, 128, 1024), (3, 64, 1152), (3, 128, 2048),
                                          (4, 32, 128), (4, 64, 1024), (4, 128, 1152), (4, 128, 2048)])
@pytest.mark.parametrize("N,T,top", [(128, 1, 1), (72, 3, 2), (264, 8, 8)])
def test_pairs(dt, bits, group, K, N, T, top):
    E = 5
    m, up = _layer(E, N, K, bits, group, dt, K + N, bias=N == 72), _layer(E, N, K, bits, group, dt, K + N + 1)
    gen = torch.Generator().manual_seed(T)
    idx = torch.randint(0, E, (T, top), generator=gen)
    x = torch.randn((T, 1, 1, K), generator=gen).to(dt)
    own = torch.randn((T, top, 1, K), generator=gen).to(dt)               # a row for each pair
    # one rounding of the result to 16 bits (two with a bias) over fp32 sums; fp16 images of bfloat16 rows lose what lies 2^-24 below a run of 32's largest, far less
    half = 2.0 ** (-9 if dt == torch.bfloat16 else -12)
    w = _dense(m)[idx]                                                    # [T, top, N, K]
    for rows in (x, own):
        y = m(rows.to(DEV), idx.to(DEV)).double().cpu()[..., 0, :]
        exact = torch.matmul(w, rows.double().expand(T, top, 1, K).transpose(-1, -2))[..., 0]
        size = torch.matmul(w.abs(), rows.double().abs().expand(T, top, 1, K).transpose(-1, -2))[..., 0]
        bound = 2 * half * exact.abs() + 1e-5 * size
        if m.bias is not None:
            exact = exact + m.bias.double().cpu()[idx]
            bound = bound + 2 * half * exact.abs()
        assert ((y - exact).abs() <= bound + 1e-7).all()
    m.bias = None
    both = ops.gather_swiglu(x.to(DEV), m, up, idx.to(torch.int32).to(DEV))
    assert both is not None
    g, u = m(x.to(DEV), idx.to(DEV)), up(x.to(DEV), idx.to(DEV))
    # gate and up in the same sums, then the same steps with the same roundings; exp of another library moves silu by a unit in the last place
    three = ((g.float() / (1 + torch.exp(-g.float()))).to(dt) * u).double()
    assert ((both.double() - three).abs() <= 4 * half * three.abs() + 1e-6).all()


def test_bad_index_and_infinity():
    m = _layer(3, 64, 1024, 4, 64, torch.bfloat16, 1)
    x = torch.randn((1, 1, 1, 1024)).bfloat16()
    y = m(x.to(DEV), torch.tensor([[-4, 0, 2, 9]]).to(DEV))
    assert torch.equal(y[0, 0], y[0, 1]) and torch.equal(y[0, 3], y[0, 2])                 # the nearest expert's row
    x[..., 7] = float("inf")
    assert not torch.isfinite(m(x.to(DEV), torch.tensor([[1]]).to(DEV)).float()).any()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,group,K", [(2, 32, 128), (2, 128, 2176), (3, 64, 1152), (3, 128, 768), (4, 32, 1024), (4, 128, 2048)])
@pytest.mark.parametrize("N,T,top", [(128, 1, 1), (76, 3, 2), (264, 8, 8), (2048, 1, 8)])
def test_mixed(dt, bits, group, K, N, T, top):
    """The last products with their weighted sum and residual in one launch: the bits of the two launches."""
    m = _layer(5, N, K, bits, group, dt, K + N)
    gen = torch.Generator().manual_seed(T)
    idx = torch.randint(0, 5, (T, top), generator=gen).to(torch.int32).to(DEV)
    act = torch.randn((T, top, 1, K), generator=gen).to(dt).to(DEV)
    scores = torch.softmax(torch.randn((T, top), generator=gen), -1).to(dt).to(DEV)
    for residual in (None, torch.randn((T, N), generator=gen).to(dt).to(DEV)):
        both = ops.gather_mix(act, m, idx, scores, residual)
        assert both is not None and torch.equal(both, ops.moe_combine(m(act, idx).squeeze(-2), scores, residual))


def test_what_watches_a_module_sees_its_call():
    from gbx_lm_amd.models.switch_layers import SwitchGLU, mixed_experts
    glu = SwitchGLU(256, 128, 4)
    for name, n, k in (("gate_proj", 128, 256), ("up_proj", 128, 256), ("down_proj", 256, 128)):
        src, dst = _layer(4, n, k, 4, 64, torch.bfloat16, n), getattr(glu, name)
        dst.qweight, dst.scales, dst.zeros = src.qweight, src.scales, src.zeros
    x = torch.randn((1, 3, 256), generator=torch.Generator().manual_seed(0)).bfloat16().to(DEV)
    idx = torch.tensor([[[0, 1], [3, 2], [1, 1]]], dtype=torch.int32).to(DEV)
    scores = torch.full((1, 3, 2), 0.5).bfloat16().to(DEV)
    y, seen = mixed_experts(glu, x, idx, scores, x), []
    handle = glu.down_proj.register_forward_hook(lambda *a: seen.append(1))
    assert torch.equal(mixed_experts(glu, x, idx, scores, x), y) and seen == [1]
    handle.remove()
