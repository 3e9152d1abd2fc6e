"""Router logits of prompt-sized steps on the matrix cores (csrc/mixers_router.hip) at the edges of their tiles: rows and experts off the grid of 16, each
of the two widths, channels off the block of 32 and fewer blocks than waves, rows that lie apart.  Reference: float64; tolerance: K fp32 roundings of the
terms' magnitudes.  An infinity stays in its row and an infinity."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("t,k,e", [(512, 8, 1), (513, 40, 5), (540, 256, 32), (600, 264, 33), (700, 1024, 63), (1030, 520, 128), (2050, 2048, 129), (2100, 2040, 256), (5000, 288, 64), (2047, 2040, 129), (2048, 2048, 256), (4100, 2048, 65)])
@pytest.mark.parametrize("apart", [False, True])
def test_logits(t, k, e, apart):
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator(device=DEV).manual_seed(t + e)
    h = torch.randn((t, k + 8 * apart), device=DEV, generator=g).to(torch.bfloat16)[:, :k]
    router = torch.randn((e, k), device=DEV, generator=g)
    got = M._router_logits(h, router)
    want, terms = h.double() @ router.double().t(), h.double().abs() @ router.double().abs().t()
    assert got.shape == want.shape and got.dtype == torch.float32
    assert bool(((got.double() - want).abs() <= k * 2.0 ** -24 * terms).all())
    h = h.clone()
    h[t // 2, k - 1], h[3, 0] = torch.inf, torch.nan
    bad = M._router_logits(h, router)
    rows = torch.ones(t, dtype=torch.bool)
    rows[[3, t // 2]] = False
    want = h.float() @ router.t()
    assert bool(torch.isnan(bad[3]).all()) and torch.equal(bad[t // 2], want[t // 2]) and torch.equal(bad[rows], got[rows])


@pytest.mark.parametrize("t,k,e", [(512, 8, 1), (600, 264, 33), (1030, 520, 128), (2047, 2048, 129)])
def test_odd_numbers(t, k, e):
    """Whole workgroups of rows that are no number, infinities of either sign and of both, in rows and in the router; sums past fp32.  Everything else as it was."""
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator(device=DEV).manual_seed(t * e)
    h, router = torch.randn((t, k), device=DEV, generator=g).to(torch.bfloat16), torch.randn((e, k), device=DEV, generator=g)
    plain = M._router_logits(h, router)
    odd = h.clone()
    odd[:64] = torch.nan
    odd[70, 0], odd[71, k - 1], odd[72, 0], odd[72, k - 1], odd[73], odd[74] = torch.inf, -torch.inf, torch.inf, torch.inf, 3e38, 0.0
    got, want = M._router_logits(odd, router), odd[:73].double() @ router.double().t()
    assert torch.equal(torch.isnan(got[:73]), torch.isnan(want))
    assert torch.equal(got[:73][want.isinf()].double(), want[want.isinf()])
    top = 3e38 * router.double().sum(1)                             # row 73: fp32 ends at 3.4e38, whatever the order where every weight has one sign
    one_sign = (router > 0).all(1) | (router < 0).all(1)
    assert torch.equal(got[73][one_sign & (top.abs() > 4e38)].double(), (top.sign() * torch.inf)[one_sign & (top.abs() > 4e38)])
    rows = torch.ones(t, dtype=torch.bool)
    rows[:75] = False
    assert torch.equal(got[rows], plain[rows]) and bool((got[74] == 0).all())
    router[e - 1, k // 2] = torch.inf
    got, x = M._router_logits(h, router), h[:, k // 2].float()
    assert torch.equal(got[:, :e - 1], plain[:, :e - 1])
    assert torch.equal(got[x != 0, e - 1], x[x != 0].sign() * torch.inf) and bool(torch.isnan(got[x == 0, e - 1]).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_a_router_without_experts(dt):
    """Nothing to choose from: no logits, as of any product."""
    from gbx_lm_amd import mixer_ops as M
    got = M._router_logits(torch.ones((600, 64), device=DEV, dtype=dt), torch.ones((0, 64), device=DEV))
    assert got.shape == (600, 0) and got.dtype == torch.float32
