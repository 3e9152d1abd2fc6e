"""RoPE of queries and keys with the cache update of a prompt chunk in one launch (gbx_rope_qkv, models.base.rope_and_update_cache): the bits of the separate steps over head
sizes and counts, chunks behind a filled cache, views of one projection, both pairings; what it does not take goes step by step."""
import pytest
import torch

from gbx_lm_amd import ops
from gbx_lm_amd.models.base import rope_and_update_cache
from gbx_lm_amd.models.cache import KVCache
from gbx_lm_amd.models.rope_utils import RoPE

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("traditional", [False, True])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,H,D", [(1, 32, 8, 128), (2, 3, 1, 64), (1, 4, 4, 16), (3, 2, 2, 256), (1, 5, 5, 48)])
def test_chunks(monkeypatch, traditional, dt, B, Hq, H, D):
    rope = RoPE(D, traditional=traditional, base=10000.0).to(DEV)
    one, steps, start, launches, launch = KVCache(step=64), KVCache(step=64), 0, [], ops.rope_qkv
    monkeypatch.setattr(ops, "rope_qkv", lambda *a, **k: launches.append(1) or launch(*a, **k))
    for L in (17, 16, 300, 3):
        qkv = torch.randn((B, L, (Hq + 2 * H) * D), generator=torch.Generator().manual_seed(L)).to(dt).to(DEV)
        q, k, v = (t.reshape(B, L, -1, D).permute(0, 2, 1, 3) for t in torch.split(qkv, [Hq * D, H * D, H * D], -1))
        if L == 300:                                                      # projections of their own
            q, k, v = (t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for t in (q, k, v))
        got = rope_and_update_cache(rope, q, k, v, one, start)
        want = (rope(q, offset=start), *steps.update_and_fetch(rope(k, offset=start), v))
        start += L
        assert one.offset == steps.offset == start and all(a.shape == b.shape and torch.equal(a, b) for a, b in zip(got, want))
    assert len(launches) == 3                                             # (three tokens are too few)


def test_cache_of_another_geometry_still_raises():
    rope = RoPE(64).to(DEV)
    cache = KVCache()
    q, k, v = (torch.randn((1, h, 20, 64), device=DEV).bfloat16() for h in (4, 2, 2))
    rope_and_update_cache(rope, q, k, v, cache, 0)
    with pytest.raises(RuntimeError):
        rope_and_update_cache(rope, q, k[:, :1].contiguous().expand(1, 3, 20, 64).contiguous(), v[:, :1].expand(1, 3, 20, 64).contiguous(), cache, 20)
    assert cache.offset in (20, 40)


def test_what_watches_the_embedding_sees_its_calls():
    rope, seen = RoPE(64).to(DEV), []
    q, k, v = (torch.randn((1, h, 20, 64), device=DEV).bfloat16() for h in (4, 2, 2))
    rope.register_forward_hook(lambda *a: seen.append(1))
    rope_and_update_cache(rope, q, k, v, KVCache(), 0)
    assert seen == [1]
