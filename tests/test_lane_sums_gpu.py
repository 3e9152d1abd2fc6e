"""Sums over the lanes of a wave, a part of it and the waves of a workgroup, at every width where a step of the sum begins or ends."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
EPS = torch.finfo(torch.float32).eps


@pytest.mark.parametrize("dv", [4, 8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("heads", [17, 64])
def test_groups_of_lanes(dv, heads):
    """Each head has a size of its own, so a lane that joins a neighbour's group shows."""
    from gbx_lm_amd import mixer_ops as M
    t, g = 3, torch.Generator().manual_seed(dv)
    o = torch.randn((t, heads, dv), generator=g) * torch.logspace(-2, 2, heads)[None, :, None]
    gate = torch.randn((t, heads * dv), generator=g)
    got = M.head_norm_gate(o.view(t, -1).to(DEV), gate.to(DEV), None, heads, 1e-6, 2).cpu().double()
    x = o.double()
    want = (x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)).view(t, -1) * torch.sigmoid(gate.double())
    # log2(dv) additions and a root: each within EPS of its result; the sigmoid's exponential within a few
    assert ((got - want).abs() <= (16 + dv.bit_length()) * EPS * want.abs() + 1e-12).all()


@pytest.mark.parametrize("width", [4, 60, 252, 256, 260, 512, 1024, 1028, 2304, 3072, 4092, 4096])
def test_waves_of_a_row(width):
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator().manual_seed(width)
    x = torch.randn((2, width), generator=g) * torch.logspace(-1, 1, width)         # a wave left out is a wrong norm
    x[1] = x[1].flip(0)
    w = torch.randn(width, generator=g)
    got = M.stream_rmsnorm(x.to(DEV), w.to(DEV), 1e-6, torch.float32).cpu().double()
    want = x.double() / torch.sqrt((x.double() ** 2).mean(-1, keepdim=True) + 1e-6) * w.double()
    assert ((got - want).abs() <= 32 * EPS * want.abs() + 1e-12).all()               # 4 + 6 + 16 additions, a root, a quotient, two products
