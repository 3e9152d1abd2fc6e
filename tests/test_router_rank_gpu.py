"""Router choices of a wave (csrc/mixers_common.h: wave_choose) and of a workgroup against rounds of arg-max on the host: expert counts around a wave, a workgroup and the
limit, ties, experts that a correction of -inf takes out, groups, and steps on both sides of the few-row logits.  Rows of a unit matrix make the
logits exactly the router's entries; weights to a few fp32 roundings."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rounds(score, top):
    """arg-max, take it out, again: of equal scores the lower index first."""
    s, out = score.clone(), []
    for _ in range(top):
        e = int((s == s.max()).nonzero()[0])
        out.append(e)
        s[e] = -2.0 if bool((score >= 0).all()) else -torch.inf
    return out


def setting(e, t, dt):
    g = torch.Generator().manual_seed(7 * e + t)
    router = (torch.randint(-6, 7, (e, 64), generator=g) / 4.0).float()          # many ties
    return torch.eye(64)[torch.arange(t) % 64].to(dt).to(DEV), router, router.t()[torch.arange(t) % 64]


@pytest.mark.parametrize("e,top", [(1, 1), (5, 5), (63, 4), (64, 8), (65, 8), (256, 7), (257, 9), (512, 8), (513, 8)])
@pytest.mark.parametrize("t,dt", [(3, torch.bfloat16), (33, torch.float32)])
@pytest.mark.parametrize("renorm", [False, True])
def test_softmax_choice(e, top, t, dt, renorm):
    from gbx_lm_amd import mixer_ops as M
    h, router, logits = setting(e, t, dt)
    idx, w = M.route_topk(h, router.to(DEV), top, renorm)
    p = torch.softmax(logits.double(), -1)
    want = torch.tensor([rounds(r, top) for r in logits])
    assert torch.equal(idx.cpu().long(), want)
    pw = p.gather(1, want)
    pw = pw / pw.sum(-1, keepdim=True) if renorm else pw
    assert float(((w.cpu().double() - pw).abs() / pw).max()) < (e / 64 + 24) * 2.0 ** -24


@pytest.mark.parametrize("e,top,groups", [(1, 1, None), (5, 2, (5, 3)), (63, 4, (9, 2)), (64, 8, (8, 4)), (66, 6, (3, 1)), (256, 8, None), (260, 8, (4, 2)), (512, 8, (256, 8)), (520, 8, (8, 4))])
@pytest.mark.parametrize("t,dt", [(3, torch.bfloat16), (33, torch.float32)])
@pytest.mark.parametrize("renorm", [False, True])
def test_grouped_sigmoid_choice(e, top, groups, t, dt, renorm):
    from gbx_lm_amd import mixer_ops as M
    h, router, logits = setting(e, t, dt)
    router[0, 1], logits = 30.0, None
    logits = router.t()[torch.arange(t) % 64]
    corr = torch.randint(0, 3, (e,)).float()
    if e > 60:
        corr[5:40] = -torch.inf                                                  # whole groups out, one group left with a single expert
    idx, w = M.route_sigmoid_groups(h, router.to(DEV), corr.to(DEV), top, groups, renorm, 1.5)
    for r in range(t):
        s = torch.sigmoid(logits[r].double())
        got = idx[r].cpu().long()
        c = (1.0 / (1.0 + torch.exp(-logits[r].to(DEV)))).cpu() + corr           # (ties and order as in fp32)
        if groups:
            n, keep = groups
            score = c.view(n, -1).topk(min(2, e // n)).values.sum(-1)
            alive = score.clone()
            for _ in range(keep):
                alive[int((alive == alive.max()).nonzero()[0])] = -torch.inf
            c = torch.where((alive != -torch.inf).repeat_interleave(e // n), torch.tensor(-torch.inf), c)
        assert len(set(got.tolist())) == top
        want = sorted(range(e), key=lambda i: (-c[i].item(), i))[:top]
        assert all(abs(c[a].item() - c[b].item()) < 1e-6 or c[a] == c[b] for a, b in zip(got.tolist(), want))
        sw = s[got] * 1.5 / (s[got].sum() + 1e-20 if renorm else 1.0)
        assert float(((w[r].cpu().double() - sw).abs() / sw).max()) < 32 * 2.0 ** -24


def odd_rows(e):
    """Logit rows with numbers missing here and there or throughout, infinities of both signs, one candidate alone, all equal."""
    rows = torch.randn((8, e), generator=torch.Generator().manual_seed(e))
    rows[0, ::3], rows[1], rows[2, e // 2], rows[3], rows[4, e - 1] = float("nan"), float("nan"), float("inf"), float("-inf"), float("-inf")
    rows[5], rows[5, e - 2], rows[6] = float("-inf"), 1.0, 0.25
    return rows


def choose(rows, top, groups=None, correction=None):
    from gbx_lm_amd import _lib
    t, e = rows.shape
    logits, idx, w = rows.to(DEV).contiguous(), torch.full((t, top), -1, dtype=torch.int32, device=DEV), torch.empty((t, top), device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    if correction is None:
        _lib.check_mixers(_lib.mixers().gbxm_route_topk(logits.data_ptr(), idx.data_ptr(), w.data_ptr(), t, e, top, 0, stream))
    else:
        count, keep = groups or (0, 0)
        c = correction.to(DEV)
        _lib.check_mixers(_lib.mixers().gbxm_route_sigmoid_groups(logits.data_ptr(), c.data_ptr(), idx.data_ptr(), w.data_ptr(), t, e, top, count, keep, 0, 1.0,
                                                                  stream))
    return idx.cpu(), w.cpu()


@pytest.mark.parametrize("e,top", [(8, 8), (32, 2), (33, 2), (128, 8), (129, 8), (256, 16), (257, 3), (520, 8)])
def test_softmax_choice_of_odd_logits(e, top):
    """Always ``top`` different experts; a row without probabilities (a logit that is no number or +inf, none finite) gives the first ones."""
    rows = odd_rows(e)
    idx, _ = choose(rows, top)
    p = torch.softmax(rows.double(), -1)
    for r in range(len(rows)):
        assert idx[r].tolist() == [i for _, i in sorted((-v if v == v else 1.0, i) for i, v in enumerate(p[r].tolist()))[:top]]


@pytest.mark.parametrize("e,top,groups", [(8, 8, None), (22, 2, None), (24, 2, None), (88, 8, None), (89, 8, None), (128, 8, (8, 4)), (136, 8, (8, 4)), (256, 8, (8, 4)),
                                          (256, 8, None), (520, 8, None)])
def test_sigmoid_choice_of_odd_logits(e, top, groups):
    """Always ``top`` different experts, those whose score is no number after all others (in groups: an order of its own, checked for being one)."""
    rows, correction = odd_rows(e), torch.zeros(e)
    idx, _ = choose(rows, top, groups, correction)
    assert all(len(set(r)) == top and min(r) >= 0 and max(r) < e for r in idx.tolist())
    if groups is None:
        c = 1.0 / (1.0 + torch.exp(-rows))
        for r in (0, 1, 2, 3, 4, 5, 6):
            key = sorted((-v if v == v else 1.0, i) for i, v in enumerate(c[r].tolist()))
            got = [c[r, i].item() for i in idx[r].tolist()]
            assert all(a != a if v > 0 else abs(a + v) < 1e-6 for a, (v, _) in zip(got, key))


@pytest.mark.parametrize("e,top", [(16, 16), (32, 26), (32, 27), (64, 46), (64, 47), (64, 64), (128, 64), (128, 65), (129, 70), (256, 64), (256, 65), (256, 256), (300, 70)])
def test_softmax_choice_of_many(e, top):
    """Both sides of the rule between rounds of a wave and ranks, and all experts chosen."""
    for t, renorm in ((3, True), (1030, False)):
        test_softmax_choice(e, top, t, torch.float32, renorm)


@pytest.mark.parametrize("e,top,groups", [(16, 10, None), (16, 11, None), (64, 28, None), (64, 29, None), (130, 70, None), (256, 64, None), (256, 65, None), (256, 200, (4, 4)), (64, 16, (32, 32)),
                                          (64, 17, (32, 32)), (64, 29, (32, 2 * 8)), (128, 8, (128, 40)), (256, 2, (128, 4)), (256, 8, (256, 128)), (300, 70, (100, 50))])
def test_grouped_sigmoid_choice_of_many(e, top, groups):
    """The same, and more groups than a wave has lanes: few of their rounds, and many."""
    test_grouped_sigmoid_choice(e, top, groups, 33, torch.float32, True)


@pytest.mark.parametrize("e,top,keep", [(64, 6, 3), (64, 32, 24), (128, 4, 2)])
def test_a_group_whose_score_is_no_number(e, top, keep):
    """An expert that is always chosen beside one that never is: their group stays and takes no other's place, by rounds and by rank."""
    rows, correction = torch.randn((3, e), generator=torch.Generator().manual_seed(e)), torch.zeros(e)
    correction[10], correction[11] = float("inf"), float("-inf")
    idx, _ = choose(rows, top, (e // 2, keep), correction)
    for r in range(3):
        c = torch.sigmoid(rows[r].double()) + correction
        best = c.view(-1, 2).sum(-1).nan_to_num(-1.0).topk(keep).indices.tolist()
        alive = [i for i in range(e) if i // 2 in best or i // 2 == 5]
        assert idx[r].tolist() == sorted(alive, key=lambda i: (-c[i].item(), i))[:top]


CHOICES = [(1, 1, None), (63, 4, (9, 2)), (64, 64, None), (65, 8, None), (128, 8, (8, 4)), (129, 65, None), (192, 6, (64, 40)), (256, 8, (8, 4)), (256, 64, (128, 64)),
           (260, 8, (4, 2))]


@pytest.mark.parametrize("e,top,groups,form", [c + (f,) for c in CHOICES for f in ("softmax", "gate", "sigmoid") if f != "sigmoid" or not c[2]])
@pytest.mark.parametrize("t", [3, 1030])
def test_choice_on_logits(e, top, groups, t, form):
    """Both forms' limits -- 64 experts a register, 256 of them, 64 choices, 64 groups -- with ties, numbers missing and infinities."""
    from gbx_lm_amd import _lib
    gate = form == "gate"
    rows = (torch.randint(-6, 7, (t, e + gate), generator=torch.Generator().manual_seed(e + t)) / 4.0).float()
    if e > 1:
        rows[0, : e // 2 : 3], rows[1, e - 1] = float("nan"), float("-inf")
    x, idx, w = rows.to(DEV).contiguous(), torch.full((t, top), -1, dtype=torch.int32, device=DEV), torch.zeros((t, top + gate), device=DEV)
    count, keep = groups or (0, 0)
    _lib.check_mixers(_lib.mixers().gbxm_route_groups(x.data_ptr(), e + gate, idx.data_ptr(), w.data_ptr(), top + gate, t, e, top, count, keep, int(gate), int(form == "sigmoid"),
                                                     torch.cuda.current_stream().cuda_stream))
    c = torch.nan_to_num(rows[:, :e], nan=float("-inf"), neginf=float("-inf")).double()
    p = torch.sigmoid(c) if form == "sigmoid" else torch.softmax(c, -1)
    if groups:
        best = torch.sort(c.view(t, count, -1).amax(-1), dim=-1, descending=True, stable=True).indices[:, :keep]
        kept = torch.zeros((t, count), dtype=torch.bool).scatter_(1, best, True).repeat_interleave(e // count, 1)
        c = c.masked_fill(~kept, float("-inf"))
    want = torch.sort(c, dim=-1, descending=True, stable=True).indices[:, :top]
    assert torch.equal(idx.cpu().long(), want)
    pw = torch.where(c.gather(1, want) == float("-inf"), 0.0, p.gather(1, want)) if form != "sigmoid" else p.gather(1, want)
    assert bool(((w.cpu().double()[:, :top] - pw).abs() <= (e / 64 + 24) * 2.0 ** -24 * pw).all())
    if gate:
        assert bool(((w.cpu().double()[:, top] - torch.sigmoid(rows[:, e].double())).abs() <= 8 * 2.0 ** -24).all())


@pytest.mark.parametrize("t,e,k", [(4, 1024, 2048), (5, 1024, 2048), (32, 1023, 2048), (32, 1024, 2048), (1, 1025, 8190), (33, 64, 100)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_logits_on_both_sides_of_the_rule(t, e, k, dt):
    """K fp32 additions of the terms' magnitudes."""
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator(device=DEV).manual_seed(t + e)
    h, router = torch.randn((t, k), device=DEV, generator=g).to(dt), torch.randn((e, k), device=DEV, generator=g)
    want, room = h.double() @ router.double().t(), h.double().abs() @ router.double().abs().t()
    assert bool(((M._router_logits(h, router).double() - want).abs() <= k * 2.0 ** -24 * room).all())
