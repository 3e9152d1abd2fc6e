"""Products of few rows (csrc/mixers_rows.hip) against float64: one row to the last row of each tile, contractions of one block to the last one of every
wave count, outputs that end inside a tile or fill several rounds of workgroups, rows with a stride, a bias; and what stays with the library.
Tolerance: K fp32 additions of the terms' magnitudes in the worst case, one rounding to bf16."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def case(t, n, k, bias, pad, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(s, device=DEV, generator=g).bfloat16()
    x = rnd(t, k + pad)[:, pad // 2 // 8 * 8:][:, :k]
    return x, rnd(n, k) * 0.05, (rnd(n) if bias else None)


@pytest.mark.parametrize("t", [1, 2, 15, 16, 17, 31, 32])
@pytest.mark.parametrize("n,k,bias,pad", [(1, 64, False, 0), (15, 448, True, 0), (17, 512, False, 16), (2048, 576, False, 8), (4100, 1024, True, 0),
                                          (33, 1088, False, 0), (8193, 2048, False, 64), (16, 2112, True, 0), (4113, 4096, False, 0)])
def test_rows(t, n, k, bias, pad):
    from gbx_lm_amd import mixer_ops as M
    x, w, b = case(t, n, k, bias, pad, t + n + k)
    y = M.linear_rows(x, w, b)
    if t > 16 and k > 2048:
        assert y is None
        return
    want, room = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    if bias:
        want, room = want + b.double(), room + b.double().abs()
    assert y.shape == (t, n) and bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + (k + 1) * 2.0 ** -24 * room).all())
    if t > 1:                                                  # a row's bits do not depend on the rows beside it
        assert torch.equal(M.linear_rows(x[:1], w, b), y[:1])


def test_what_stays_with_the_library():
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.models.projection import project
    x, w, b = case(4, 48, 256, True, 0, 3)
    for xx, ww, bb in ((x[:0], w, b), (x.float(), w.float(), b.float()), (x[:, :40], w[:, :40].contiguous(), b), (x.half(), w.half(), b.half()),
                       (x.t().contiguous().t(), w, b), (x, w.t().contiguous().t(), b), (x.expand(4, 4, 256).reshape(16, 256)[:1].expand(3, 256), w, b),
                       (torch.cat([x] * 9), w, b), (torch.cat([x] * 17, 1), torch.cat([w] * 17, 1), b)):
        assert M.linear_rows(xx, ww, bb) is None
        assert torch.equal(project(xx, ww, bb), F.linear(xx, ww, bb))
    y = project(x.view(2, 2, 256), w, b)
    assert y.shape == (2, 2, 48) and torch.equal(y.view(4, 48), M.linear_rows(x, w, b))
    wg = w.clone().requires_grad_(True)
    assert project(x, wg, b).requires_grad and not project(x, wg.detach(), b).requires_grad


def test_what_torch_does_around_a_product_stays():
    """Gradients of a bias alone, forward-mode tangents, vmap, autocast, symbolic and recorded traces, dispatch modes: the rows then go through torch."""
    import torch.autograd.forward_ad as fw
    from torch.utils.flop_counter import FlopCounterMode
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.models.projection import RowLinear, project
    x, w, b = case(4, 48, 256, True, 0, 3)
    bg = b.clone().requires_grad_(True)
    project(x, w, bg).float().sum().backward()
    assert torch.equal(bg.grad, torch.full_like(b, 4.0))
    with torch.no_grad(), fw.dual_level():
        t = torch.ones_like(x)
        assert torch.equal(fw.unpack_dual(project(fw.make_dual(x, t), w, b)).tangent, F.linear(t, w))
    xs = torch.stack([x, x + 1])
    with torch.no_grad():
        assert torch.equal(torch.func.vmap(lambda v: project(v, w, b))(xs), torch.func.vmap(lambda v: F.linear(v, w, b))(xs))
        with torch.autocast("cuda", dtype=torch.float16):
            assert project(x, w, b).dtype == torch.float16
        with FlopCounterMode(display=False) as flops:
            project(x, w, b)
        assert flops.get_total_flops() == 2 * 4 * 48 * 256
        layer = RowLinear(256, 48, device=DEV, dtype=torch.bfloat16)
        traced = torch.jit.trace(layer, (x,))
        assert torch.equal(traced(x + 1), F.linear(x + 1, layer.weight, layer.bias))
        symbolic = torch.fx.symbolic_trace(layer)
        assert torch.equal(symbolic(x), F.linear(x, layer.weight, layer.bias))
        compiled = torch.compile(lambda v: project(v, w, b) * 2, backend="eager", fullgraph=True)
        assert torch.equal(compiled(x), F.linear(x, w, b) * 2)
        assert torch.equal(project(x[:, :0], w[:, :0], b), F.linear(x[:, :0], w[:, :0], b))
        assert not torch.equal(project(x, w, b), torch.zeros_like(project(x, w, b))) and torch.equal(project(x, w, b), M.linear_rows(x, w, b))


@pytest.mark.parametrize("t,n,k,taken", [(16, 40000, 4096, True), (17, 32768, 1088, False), (17, 32767, 1088, True), (32, 32768, 1984, False), (32, 40000, 2048, True),
                                         (32, 40000, 1024, True), (32, 16, 2112, False), (33, 16, 64, False)])
def test_the_rule(t, n, k, taken):
    from gbx_lm_amd import mixer_ops as M
    x, w, _ = case(t, n, k, False, 0, t)
    y = M.linear_rows(x, w, None)
    assert (y is not None) == taken == M.rows_win(t, n, k)


@pytest.mark.parametrize("k", [64, 128, 192, 256, 320, 704, 768, 832, 1472, 1536, 1600, 2944, 3072, 3136])
@pytest.mark.parametrize("t", [1, 32])
def test_blocks_of_every_form(t, k):
    """The last contraction of each number of blocks a wave, and those beside it."""
    from gbx_lm_amd import mixer_ops as M
    x, w, b = case(t, 300, k, True, 0, k)
    y = M.linear_rows(x, w, b)
    if y is None:
        assert t > 16 and k > 2048
        return
    want, room = x.double() @ w.double().t() + b.double(), x.double().abs() @ w.double().abs().t() + b.double().abs()
    assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + (k + 1) * 2.0 ** -24 * room).all())
