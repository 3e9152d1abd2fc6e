"""Log-probabilities in one launch (csrc/mixers_ops.hip: log_softmax_kernel): rows shorter than a wave, around the registers a workgroup keeps
(8 pieces of 16 bytes a thread), far beyond them, off the 16-byte grid; masked, infinite and undefined logits.  Reference: float64.  The
logarithm is an fp32 sum of n terms (n 2^-24 relative, so as much absolute in its logarithm, plus its own last place) rounded once to the
rows' type; the difference is rounded once more."""
import pytest
import torch

pytestmark = pytest.mark.gpu
LAST = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


@pytest.mark.parametrize("dt", list(LAST))
@pytest.mark.parametrize("rows,n", [(1, 1), (3, 7), (2, 8), (5, 1000), (2, 32767), (32, 32000), (2, 32800), (1, 65536), (1, 65537), (1, 128256), (3, 151936)])
def test_rows(dt, rows, n):
    from gbx_lm_amd.mixer_ops import log_probabilities
    x = (torch.randn((rows, n), device="cuda", generator=torch.Generator(device="cuda").manual_seed(n)) * 3).to(dt)
    got, want = log_probabilities(x), x.double() - torch.logsumexp(x.double(), -1, keepdim=True)
    assert got.dtype == dt and got.shape == x.shape
    lse = torch.logsumexp(x.double(), -1, keepdim=True).abs()
    room = LAST[dt] * (lse + want.abs()) + n * 2.0 ** -24 + 2.0 ** -22 * (1 + lse)
    assert bool(((got.double() - want).abs() <= room).all())
    off = torch.empty(rows * n + 1, dtype=dt, device="cuda")[1:].view(rows, n).copy_(x)            # rows off the 16-byte grid
    assert bool(((log_probabilities(off).double() - want).abs() <= room).all())


@pytest.mark.parametrize("n", [500, 40000])
@pytest.mark.parametrize("dt", list(LAST))
def test_masked_and_undefined_logits(dt, n):
    from gbx_lm_amd.mixer_ops import log_probabilities
    x = torch.randn((5, n), device="cuda").to(dt)
    x[0, 100:] = float("-inf")
    x[1] = float("-inf")
    x[2, 7] = float("inf")
    x[3, 9] = float("nan")
    x[4] = torch.finfo(dt).min
    got = log_probabilities(x)
    want = x - torch.logsumexp(x.float(), -1, keepdim=True).to(dt)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    ok = torch.isfinite(want)
    assert bool(((got - want).abs()[ok].float() <= 2 * LAST[dt] * (1 + want.abs()[ok].float())).all())


@pytest.mark.parametrize("dt", list(LAST))
def test_slices_without_a_candidate(dt):
    """A few long rows are summed slice by slice: slices in which every logit is masked add nothing, however low the row's maximum lies."""
    from gbx_lm_amd.mixer_ops import log_probabilities
    x = torch.full((4, 40000), float("-inf"), device="cuda", dtype=dt)
    x[0, :100] = -200
    x[1, 39990:] = -30000
    x[2, 20000] = 300
    x[3, :100], x[3, 30000] = -200, float("nan")
    got = log_probabilities(x)
    lse = torch.logsumexp(x.double(), -1, keepdim=True)
    want = x.double() - lse
    assert torch.isnan(got[3]).all()
    for r in range(3):
        ok = torch.isfinite(x[r])
        assert (got[r][~ok] == float("-inf")).all()
        assert bool(((got[r].double() - want[r]).abs()[ok] <= LAST[dt] * (lse[r].abs() + want[r].abs()[ok]) + 2.0 ** -22 * (1 + lse[r].abs())).all())


def test_what_torch_does_around_the_rows_stays():
    """Gradients, forward-mode tangents and vmap of the logits: torch's operations."""
    import torch.autograd.forward_ad as fw
    from gbx_lm_amd.mixer_ops import log_probabilities
    x = torch.randn((3, 500), device="cuda")
    g = x.clone().requires_grad_(True)
    log_probabilities(g)[:, 0].sum().backward()
    want = -torch.softmax(x, -1)
    want[:, 0] += 1
    assert torch.allclose(g.grad, want, atol=1e-6)
    with torch.no_grad(), fw.dual_level():
        t = torch.ones_like(x)
        assert fw.unpack_dual(log_probabilities(fw.make_dual(x, t))).tangent.abs().max() < 1e-5
    assert torch.allclose(torch.func.vmap(log_probabilities)(x[None].expand(2, 3, 500))[1], log_probabilities(x), atol=1e-5)
