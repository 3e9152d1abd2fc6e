"""Attention that leaves the step's rows in the table (gbxm_sink_attention_append) against the two calls apart: the same rows, the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dk,dv,H,G,values,window,keep", [(64, 64, 8, 2, True, None, 0), (128, 128, 16, 4, True, 33, 5), (576, 512, 16, 1, False, None, 0), (50, 34, 6, 3, True, 40, 0),
                                                          (96, 96, 8, 1, False, 33, 0)])
@pytest.mark.parametrize("first,lens", [([0], [1]), ([500], [1]), ([31, 200, 0], [1, 1, 1]), ([0, 90], [70, 3]), ([100, 7], [40, 1]), ([60] * 70, [1] * 70)])
def test_both_in_one_call(dt, dk, dv, H, G, values, window, keep, first, lens):
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.batching import StepBatch
    from gbx_lm_amd.models.cache import SequenceSlots, SlotKVCache
    gen = torch.Generator(device=DEV).manual_seed(dk + len(first))
    n, T = len(first), sum(lens)
    caches = []
    for _ in range(2):
        c = SlotKVCache(G * dk, G * dv if values else 0, window, keep, SequenceSlots(n))
        c.reserve(max(f + m for f, m in zip(first, lens)), dt, torch.device(DEV))
        caches.append(c)
    caches[0].keys.normal_(generator=gen)
    caches[1].keys.copy_(caches[0].keys)
    if values:
        caches[0].values.normal_(generator=gen)
        caches[1].values.copy_(caches[0].values)
    rows = torch.randn((T, H * dk + G * (dk + dv) + 7), device=DEV, generator=gen).to(dt)
    q = rows[:, :H * dk].unflatten(1, (H, dk))
    kr = rows[:, H * dk:H * dk + G * dk]
    k = kr.unflatten(1, (G, dk))
    vr = rows[:, H * dk + G * dk:H * dk + G * (dk + dv)] if values else None
    v = vr.unflatten(1, (G, dv)) if values else k[..., :dv]
    gate = torch.randn((T, H * dv), device=DEV, generator=gen).to(dt)
    batch = StepBatch.build(list(range(n)), first, lens, DEV)
    args = (batch, dk ** -0.5, window, keep, torch.randn(H, device=DEV, generator=gen), gate)
    apart = M.sink_attention(q, k, v, caches[0], *args)
    M.slot_append(caches[0], kr, vr, batch)
    joined = M.sink_attention(q, k, v, caches[1], *args, append=(kr, vr))
    assert torch.equal(apart, joined)
    assert torch.equal(caches[0].keys, caches[1].keys) and torch.equal(caches[0].values, caches[1].values)
