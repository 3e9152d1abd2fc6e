"""The decayed scans' staging in groups of four (csrc/mixers_state.hip: V) beside the one that goes element by element: sizes where groups end inside the
16-lane grid, rows and strides that are or are not in groups, tokens around a staged chunk's end, both launch shapes.  Reference: float64 token by
token; tolerance: fp32 sums over the key channels and the tokens that a decay of at most 0.9 keeps."""
import pytest
import torch

from gbx_lm_amd.batching import StepBatch
from gbx_lm_amd.models import recurrent_mixers as RM
from gbx_lm_amd.models.cache import SequenceSlots, SlotStateCache

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("dk,dv,H", [(4, 4, 4), (60, 20, 4), (64, 16, 2), (68, 12, 4), (128, 36, 4), (132, 8, 4), (192, 4, 4), (196, 4, 3), (256, 20, 4), (62, 20, 4), (64, 18, 4)])
@pytest.mark.parametrize("counts", [(33, 15), (1, 2), (7, 8)])
def test_scan(dk, dv, H, counts, delta):
    scan(dk, dv, H, counts, delta)


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("dk,dv,H", [(1, 3, 2), (4, 20, 4), (15, 4, 3), (16, 36, 4), (17, 5, 3), (20, 8, 4), (31, 18, 4), (32, 16, 4), (33, 4, 3), (66, 18, 4), (95, 7, 3), (96, 6, 4), (97, 4, 3)])
@pytest.mark.parametrize("counts", [(33, 15), (1, 2)])
def test_heads_of_few_channels(dk, dv, H, counts, delta):
    """Lanes of one, two and four channels: the first and last sizes of each."""
    scan(dk, dv, H, counts, delta)


def scan(dk, dv, H, counts, delta):
    G, g = 1, torch.Generator().manual_seed(dk + dv + counts[0])
    lay = RM.RecurrentLayout(H, G, dk, dv, 0, G * dk, 2 * G * dk, 2 * G * dk + H * dv if delta else -1)
    T = sum(counts)
    q, k = torch.randn((T, G * dk), generator=g), torch.nn.functional.normalize(torch.randn((T, G * dk), generator=g), dim=-1)
    v, d = torch.randn((T, H * dv), generator=g), torch.rand((T, H * dk), generator=g) * 0.4 + 0.5
    beta = torch.rand((T, H), generator=g)
    r = torch.cat([q, k, v, d] + ([beta] if delta else []), 1)
    cache = SlotStateCache(H, dk, dv, 0, 0, SequenceSlots(2))
    cache.reserve(torch.float32, DEV)
    start = torch.randn(cache.state.shape, generator=g)
    cache.state.copy_(start)
    out = RM.decayed_state_scan(r.to(DEV), lay, cache, StepBatch.build([1, 0], [5, 0], list(counts), DEV), delta)
    r0 = 0
    for slot, pos0, n in ((1, 5, counts[0]), (0, 0, counts[1])):
        S = start[slot].double().clone() if pos0 else torch.zeros_like(start[slot].double())          # [H, dv, dk]
        for t in range(r0, r0 + n):
            S = S * d[t].double().view(H, 1, dk)
            u = v[t].double().view(H, dv)
            if delta:
                u = beta[t].double().view(H, 1) * (u - (S * k[t].double()).sum(-1))
            S = S + u.unsqueeze(-1) * k[t].double()
            want, room = (S * q[t].double()).sum(-1), (S.abs() * q[t].double().abs()).sum(-1).amax()
            assert float((out[t].cpu().double().view(H, dv) - want).abs().max()) < (dk + 40) * 2.0 ** -24 * float(room) * 4
        assert float((cache.state[slot].cpu().double() - S).abs().max()) < (dk + 40) * 2.0 ** -24 * float(S.abs().max()) * 4
        r0 += n
