"""Grouped matrix-core products of routed experts (csrc/mixers_moe_mfma.hip) at the edges of their tiles: experts that get no pair, one, and
one less / as many / one more than each tile height; output channels and contractions on the 32-grid but off every tile; contractions of
one, two and three pipeline stages; every expert form with and without a factor per pair.  Reference: float64 from the same bf16 numbers.
Tolerance: the hidden row and the result are rounded to bf16 once each (half of the last of 8 bits: at most 2^-8 of their size); a result is a sum over ff hidden values whose
roundings are independent, so its error stays under 2^-8 (|y| + sqrt(ff) rms(terms)) , 3 x for the extremes of half a million values."""
import pytest
import torch

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320, 513]


def reference(h, first, down, idx, kind, limit, scale):
    e64 = lambda t: t.double()
    T, top = idx.shape
    y = torch.zeros((T, top, down.shape[1]), dtype=torch.float64, device=h.device)
    spread = torch.zeros_like(y)
    for e in range(first.shape[0]):
        t, s = torch.nonzero(idx == e, as_tuple=True)
        if not t.numel():
            continue
        z = e64(h[t]) @ e64(first[e]).t()
        if scale is not None:
            z = z * scale[t, s].double()[:, None]
        if kind == "relu2":
            a = z.clamp(min=0) ** 2
        else:
            g, u = z.chunk(2, -1)
            if kind == "clamped_swish":
                g, u = g.clamp(max=limit), u.clamp(-limit, limit) + 1.0
                a = g * torch.sigmoid(1.702 * g) * u
            else:
                a = g * torch.sigmoid(g) * u
        y[t, s] = a @ e64(down[e]).t()
        spread[t, s] = ((a ** 2) @ (e64(down[e]) ** 2).t()).sqrt()
    return y, spread


@pytest.mark.parametrize("kind", ["silu", "clamped_swish", "relu2"])
@pytest.mark.parametrize("width,ff", [(32, 32), (64, 96), (96, 160), (288, 64), (160, 352)])
def test_tiles_of_every_height(kind, width, ff):
    tiles(COUNTS, kind, width, ff)


@pytest.mark.parametrize("kind", ["silu", "clamped_swish", "relu2"])
@pytest.mark.parametrize("width,ff", [(32, 32), (160, 288), (288, 96)])
@pytest.mark.parametrize("counts", [[0, 1, 31, 32, 33, 63, 64, 65, 97, 128], [64], [(13 * i) % 41 for i in range(60)]], ids=["units", "one expert", "runs"])
def test_skinny_tiles(kind, width, ff, counts):
    """Few workgroups in the grouped form: tiles of 32 pairs, both ways of sharing them out among the XCDs."""
    tiles(counts, kind, width, ff)


@pytest.mark.parametrize("pairs", [48, 56, 64])
def test_few_workgroups_of_long_contractions(pairs):
    """Both sides of the rule for steps of few experts: one tile of an expert's pairs, or several that read its weights anew."""
    tiles([pairs + d for d in (-9, 0, 3, 6)] * 2, "relu2", 4096, 2048)


def tiles(counts, kind, width, ff):
    from gbx_lm_amd import mixer_ops as M
    gen = torch.Generator(device="cuda").manual_seed(width + ff)
    E, T = len(counts), sum(counts)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=gen)
    h = rnd(T, width).to(torch.bfloat16)
    first = (rnd(E, ff * (1 if kind == "relu2" else 2), width) * width ** -0.5).to(torch.bfloat16)
    down = (rnd(E, width, ff) * ff ** -0.5).to(torch.bfloat16)
    idx = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])[torch.randperm(T, generator=torch.Generator().manual_seed(1))]
    idx = idx.to(torch.int32).to("cuda")[:, None].contiguous()
    for scale in (None, torch.rand((T, 1), device="cuda", generator=gen) + 0.5):
        got = M.expert_glu(h, first, down, idx, kind, 1.5, scale).double()
        want, spread = reference(h, first, down, idx, kind, 1.5, scale)
        bound = 2.0 ** -8 * (want.abs() + spread) * 3 + 1e-6
        assert bool(((got - want).abs() <= bound).all()), float(((got - want).abs() / bound).max())


def test_choices_share_rows_across_tiles():
    """Several choices per row (a row is then read by tiles of several experts) and one expert far more wanted than the others."""
    from gbx_lm_amd import mixer_ops as M
    gen = torch.Generator(device="cuda").manual_seed(3)
    T, E, top, width, ff = 700, 5, 3, 128, 192
    h = torch.randn((T, width), device="cuda", generator=gen).to(torch.bfloat16)
    first = (torch.randn((E, 2 * ff, width), device="cuda", generator=gen) * width ** -0.5).to(torch.bfloat16)
    down = (torch.randn((E, width, ff), device="cuda", generator=gen) * ff ** -0.5).to(torch.bfloat16)
    score = torch.rand((T, E), device="cuda", generator=gen)
    score[:, 2] += 0.8
    idx = score.topk(top, -1).indices.to(torch.int32).contiguous()
    got = M.expert_glu(h, first, down, idx, "silu", 0.0, None).double()
    want, spread = reference(h, first, down, idx, "silu", 0.0, None)
    assert bool(((got - want).abs() <= 2.0 ** -8 * (want.abs() + spread) * 3 + 1e-6).all())


@pytest.mark.parametrize("experts,pairs", [(8, 2047), (300, 2048), (8, 2049), (8, 32768), (8, 32769), (5, 70000), (300, 40000)])
def test_more_pairs_than_the_sort_keeps(experts, pairs):
    """Either side of the few pairs that go straight to their places, and the pairs beyond those whose places the sort holds in registers; uneven experts."""
    w = torch.arange(1, experts + 1, dtype=torch.float64)
    counts = (w / w.sum() * pairs).long().tolist()
    counts[-1] += pairs - sum(counts)
    tiles(counts, "relu2", 32, 32)


@pytest.mark.parametrize("rows,top", [(40, 2), (700, 2)], ids=["skinny", "grouped"])
@pytest.mark.parametrize("width,ff", [(1056, 736), (512, 1056)])
def test_a_pair_does_not_depend_on_its_neighbours(rows, top, width, ff):
    """Experts start the contraction at places of their own, over whole and odd numbers of chunks: the same bits for a row wherever it stands in the step."""
    from gbx_lm_amd import mixer_ops as M
    gen = torch.Generator(device="cuda").manual_seed(5)
    experts = 9
    first = (torch.randn(experts, 2 * ff, width, generator=gen, device="cuda") / width ** 0.5).bfloat16()
    down = (torch.randn(experts, width, ff, generator=gen, device="cuda") / ff ** 0.5).bfloat16()
    h = torch.randn(rows, width, generator=gen, device="cuda").bfloat16()
    idx = torch.rand(rows, experts, generator=gen, device="cuda").topk(top, -1).indices.to(torch.int32).contiguous()
    got = M.expert_glu(h, first, down, idx, "silu", 1.5, None)
    turned = torch.randperm(rows, generator=gen, device="cuda")
    again = M.expert_glu(h[turned].contiguous(), first, down, idx[turned].contiguous(), "silu", 1.5, None)
    assert torch.equal(got.reshape(rows, -1)[turned], again.reshape(rows, -1))
