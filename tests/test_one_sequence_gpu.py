"""Decoding one sequence: the context of grouped attention split from short caches on (csrc/decode_ops.hip: attn_splits), and log-probabilities of few rows at the
lengths around which they take two launches (csrc/mixers_ops.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("hd,nh,nkv", [(128, 32, 4), (64, 8, 2), (128, 6, 2), (128, 7, 1)])
@pytest.mark.parametrize("cap", [64, 256, 768, 1536])
def test_split_context_against_a_batch_of_the_same_sequence_twice(hd, nh, nkv, cap):
    """Batches are not split at these sizes.  The two sums run over the same products in another order (fp32), their result is rounded once."""
    from gbx_lm_amd import _lib, ops
    from gbx_lm_amd.models.rope_utils import RoPE
    assert _lib.lib().gbx_attn_workspace_bytes(1, nh, nkv, hd, cap) > 0
    gen = torch.Generator(device=DEV).manual_seed(cap + nh)
    q, k, v = (torch.randn((1, n * hd), device=DEV, generator=gen).to(torch.bfloat16) for n in (nh, nkv, nkv))
    kc, vc = (torch.randn((1, nkv, cap, hd), device=DEV, generator=gen).to(torch.bfloat16) for _ in range(2))
    qw, kw = ((torch.rand(hd, device=DEV, generator=gen) + 0.5).to(torch.bfloat16) for _ in range(2))
    inv = RoPE(hd, traditional=False, base=1000000.0).inv_freq.to(DEV)
    for pos in (0, 1, 15, 31, 32, 47, 63, cap - 1):
        p = torch.tensor([pos], device=DEV)
        got = []
        for b in (1, 2):
            caches = [t.expand(b, -1, -1, -1).contiguous() for t in (kc, vc)]
            out = torch.zeros((b, nh * hd), dtype=torch.bfloat16, device=DEV)
            ops.attn_decode_batched(*(t.expand(b, -1).contiguous() for t in (q, k, v)), *caches, inv, p, out, nh, nkv, hd, 1.0, hd ** -0.5, False, qw, kw, 1e-6)
            got.append((out[0].float(), caches[0][0], caches[1][0]))
        (one, k1, v1), (two, k2, v2) = got
        assert torch.equal(k1, k2) and torch.equal(v1, v2)
        assert bool(((one - two).abs() <= 2.0 ** -7 * two.abs() + 2.0 ** -16 * vc.float().abs().max()).all())


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,n", [(1, 24576), (1, 24577), (15, 24584), (16, 24584), (2, 26623)])
def test_log_probabilities_around_the_second_launch(dt, rows, n):
    """The logarithm: an fp32 sum of n terms rounded to the rows' type; the difference is rounded once more."""
    from gbx_lm_amd.mixer_ops import log_probabilities
    x = (torch.randn((rows, n), device=DEV, generator=torch.Generator(device=DEV).manual_seed(n)) * 3).to(dt)
    x[0, :9000] = float("-inf")                                    # slices without a candidate
    got, lse = log_probabilities(x), torch.logsumexp(x.double(), -1, keepdim=True)
    want, last = x.double() - lse, 2.0 ** -24 if dt == torch.float32 else 2.0 ** -8
    seen = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), seen)
    room = last * (lse.abs() + want.abs()) + n * 2.0 ** -24 + 2.0 ** -22 * (1 + lse.abs())
    assert bool(((got.double() - want).abs() <= room)[seen].all())


@pytest.mark.parametrize("kv,heads", [(1, 8), (2, 8), (4, 8), (4, 16)])
def test_short_caches_keep_the_fused_block(kv, heads):
    """What the attention launch of its own does with a short cache does not take the block's fused launch away: only a long one does."""
    from gbx_lm_amd import synthetic as S
    from gbx_lm_amd.decode import FusedDecodeRunner
    from gbx_lm_amd.models.cache import KVCache
    cfg = dict(S.TINY, hidden_size=1024, intermediate_size=2048, num_attention_heads=heads, num_key_value_heads=kv, num_hidden_layers=1)
    model = S.build_model(cfg, S.make_strategy("S22", 1, 128), device=DEV, seed=3)
    at = model.model.layers[0].self_attn
    for capacity, long in ((256, False), (8192, True)):
        c = KVCache(step=capacity)
        like = torch.empty((1, at.n_kv_heads, 1, at.head_dim), dtype=torch.bfloat16, device=DEV)
        c.reserve(1, like, like)
        r = FusedDecodeRunner(model, [c], use_graph=False)
        assert r.long_cache == long and (r.attn_ws is None) == (not long)


@pytest.mark.parametrize("normed,cap", [(False, 256), (False, 768), (False, 4096), (True, 512)])
def test_scratch_only_where_the_context_is_split(normed, cap):
    """A launch that reads its context in one piece is given none."""
    from gbx_lm_amd import _lib, ops
    from gbx_lm_amd.models.rope_utils import RoPE
    nh, nkv, hd = 32, 4, 128
    q, k, v = (torch.randn((1, n * hd), device=DEV).to(torch.bfloat16) for n in (nh, nkv, nkv))
    kc, vc = (torch.zeros((1, nkv, cap, hd), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    w = torch.ones(hd, dtype=torch.bfloat16, device=DEV) if normed else None
    inv, p, out = RoPE(hd, traditional=False, base=10000.0).inv_freq.to(DEV), torch.tensor([9], device=DEV), torch.zeros((1, nh * hd), dtype=torch.bfloat16, device=DEV)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    ops.attn_decode_batched(q, k, v, kc, vc, inv, p, out, nh, nkv, hd, 1.0, hd ** -0.5, False, w, w, 1e-6)
    split = _lib.lib().gbx_attn_splits(1, nh, nkv, cap, int(normed)) > 1
    assert split == (normed or cap == 4096) and (torch.cuda.max_memory_allocated() > before) == split
