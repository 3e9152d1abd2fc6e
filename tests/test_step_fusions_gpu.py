"""Launches of a decode step that stand for two (or a copy beside one): two short products, the embedding in every stream, the
convolution's inputs moved on by the preparation.  Each against the launches that it stands for, bit for bit."""
import pytest
import torch

from gbx_lm_amd import mixer_ops as M
from gbx_lm_amd.batching import StepBatch
from gbx_lm_amd.models import recurrent_mixers as RM
from gbx_lm_amd.models.cache import SequenceSlots

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T", [1, 16, 17, 32])
@pytest.mark.parametrize("K", [64, 128, 192, 256, 320, 512])
@pytest.mark.parametrize("N0,N1", [(512, 1024), (16, 8), (1, 33), (9000, 24)])
def test_pair(T, K, N0, N1):
    gen = torch.Generator(device=DEV).manual_seed(K)
    rows = torch.randn((T, 2 * K + 24), device=DEV, generator=gen).bfloat16()
    x0, x1 = rows[:, 8:8 + K], rows[:, K + 16:2 * K + 16]
    w0, w1 = (torch.randn((n, K), device=DEV, generator=gen).bfloat16() for n in (N0, N1))
    y = M.linear_rows_pair(x0, w0, x1, w1)
    assert y is not None and torch.equal(y[0], M.linear_rows(x0, w0, None)) and torch.equal(y[1], M.linear_rows(x1, w1, None))


def test_pair_leaves_others_alone():
    b = lambda *s: torch.randn(s, device=DEV).bfloat16()
    for x0, w0, x1, w1 in ((b(1, 64), b(8, 64), b(1, 128), b(8, 128)), (b(33, 64), b(8, 64), b(33, 64), b(8, 64)), (b(1, 576), b(8, 576), b(1, 576), b(8, 576)),
                           (b(1, 72), b(8, 72), b(1, 72), b(8, 72)), (b(1, 64).float(), b(8, 64), b(1, 64), b(8, 64)), (b(1, 65)[:, 1:], b(8, 64), b(1, 64), b(8, 64)),
                           (b(1, 64), b(64, 8).t(), b(1, 64), b(8, 64))):
        assert M.linear_rows_pair(x0, w0, x1, w1) is None


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,streams", [(1, 1024, 4), (5, 1026, 3), (3, 7, 1), (2, 4100, 64)])
def test_streams(dt, T, W, streams):
    table, tokens = torch.randn((50, W), device=DEV).to(dt), torch.randint(0, 50, (T,), device=DEV)
    assert torch.equal(M.embed_streams(table, tokens, streams), table[tokens].float()[:, None].repeat(1, streams, 1))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("first", [[0], [4, 0, 9, 1, 2, 3], [i % 5 for i in range(70)]])
@pytest.mark.parametrize("taps,G,H,dk,dv,grid", [(4, 2, 4, 64, 32, True), (4, 16, 32, 128, 128, True), (4, 3, 3, 4, 8, True), (3, 2, 4, 64, 32, True), (4, 2, 4, 64, 32, False), (2, 1, 2, 20, 6, True)])
def test_tails_move_on(dt, first, taps, G, H, dk, dv, grid):
    """Vectors of four channels, layouts that go number by number (other taps, rows off the grid of their loads), sequences at and behind their start."""
    B, nq, nv = len(first), G * dk, H * dv
    C = 2 * nq + nv
    batch = StepBatch.build([B - i for i in range(B)], first, [1] * B, DEV)
    lay = RM.RecurrentLayout(H, G, dk, dv, 0, nq, 2 * nq, C)
    gen = torch.Generator(device=DEV).manual_seed(B + dk)
    y = torch.randn((B, C + H + -(C + H) % 4 + (0 if grid else 1)), device=DEV, generator=gen).to(dt)
    a = torch.randn((B, H * dk), device=DEV, generator=gen).to(dt)
    bias, rate = torch.randn(H * dk, device=DEV, generator=gen), torch.rand(H, device=DEV, generator=gen) + 0.1
    conv = torch.randn((C, taps), device=DEV, generator=gen).to(dt)
    one, two = (RM.SlotStateCache(H, dk, dv, C, taps, SequenceSlots(B + 1)) for _ in range(2))
    for c in (one, two):
        c.reserve(dt, DEV)
    one.tail.normal_(generator=gen)
    two.tail.copy_(one.tail)
    for _ in range(3):                                                    # (a tail that was moved on is read by the next step)
        got = M.recurrent_prepare(y, a, lay, bias, rate, 1.0, conv, one, batch, True, 0.3, keep_tail=True)
        want = M.recurrent_prepare(y, a, lay, bias, rate, 1.0, conv, two, batch, True, 0.3)
        M.conv_tail_update(y, C, two, batch)
        assert torch.equal(got, want) and torch.equal(one.tail, two.tail)
        first = [p + 1 for p in first]
        batch = StepBatch.build([B - i for i in range(B)], first, [1] * B, DEV)
