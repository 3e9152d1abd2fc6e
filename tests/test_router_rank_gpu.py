"""Router choices by rank (csrc/mixers_common.h: RANK_EXPERTS) against rounds of arg-max on the host: expert counts around a wave, a workgroup and the
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
