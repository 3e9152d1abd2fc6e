"""Decoding one sequence: the context of grouped attention split from caches of 256 positions on (csrc/decode_ops.hip: attn_splits), and log-probabilities of few rows at the
lengths around which they take two launches (csrc/mixers_ops.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


HEADS = [(128, 32, 4), (64, 8, 2), (128, 6, 2), (128, 32, 8), (64, 24, 4), (128, 7, 1), (128, 16, 8)]


def operands(hd, nh, nkv, cap):
    from gbx_lm_amd.models.rope_utils import RoPE
    gen = torch.Generator(device=DEV).manual_seed(cap + nh)
    q, k, v = (torch.randn((1, n * hd), device=DEV, generator=gen).to(torch.bfloat16) for n in (nh, nkv, nkv))
    kc, vc = (torch.randn((1, nkv, cap, hd), device=DEV, generator=gen).to(torch.bfloat16) for _ in range(2))
    qw, kw = ((torch.rand(hd, device=DEV, generator=gen) + 0.5).to(torch.bfloat16) for _ in range(2))
    return q, k, v, kc, vc, qw, kw, RoPE(hd, traditional=False, base=1000000.0).inv_freq.to(DEV)


def attend(q, k, v, kc, vc, qw, kw, inv, pos, nh, nkv, hd, batch=1):
    from gbx_lm_amd import ops
    caches = [t.expand(batch, -1, -1, -1).contiguous() for t in (kc, vc)]
    out = torch.zeros((batch, nh * hd), dtype=torch.bfloat16, device=DEV)
    ops.attn_decode_batched(*(t.expand(batch, -1).contiguous() for t in (q, k, v)), *caches, inv, torch.tensor([pos], device=DEV), out, nh, nkv, hd, 1.0, hd ** -0.5, False,
                            qw, kw, 1e-6)
    return out[0], caches[0][0], caches[1][0]


@pytest.mark.parametrize("hd,nh,nkv", HEADS)
@pytest.mark.parametrize("cap", [64, 256, 768, 1023, 1024, 1536])
def test_split_context_against_float64(hd, nh, nkv, cap):
    """Query and key are rounded to bf16 after the norm and after the rotation, as the launch rounds them: where its fp32 steps fall on the other side of a tie an
    element is one step (2^-8) off.  Tolerance: three standard deviations of the scores for such steps in every element, twice (numerator and sum), and the
    result's rounding."""
    from gbx_lm_amd import _lib
    rep = nh // nkv
    expect = cap >= 1024 or (cap >= 256 and (rep % 4 == 0 or rep % 3 == 0))
    assert (_lib.lib().gbx_attn_workspace_bytes(-1, nh, nkv, hd, cap) > 0) == expect and (_lib.lib().gbx_attn_workspace_bytes(1, nh, nkv, hd, cap) > 0) == (cap >= 1024)
    q, k, v, kc, vc, qw, kw, inv = operands(hd, nh, nkv, cap)

    def turned(x, w, pos):
        x = x.double().view(-1, hd)
        x = (x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * w.double()).to(torch.bfloat16).double()
        a, (x1, x2) = pos * inv.double(), x.chunk(2, -1)
        return torch.cat([x1 * a.cos() - x2 * a.sin(), x1 * a.sin() + x2 * a.cos()], -1).to(torch.bfloat16).double()

    for pos in sorted({0, 1, 15, 31, 32, 47, 63, cap // 2, cap - 1}):
        got, k1, v1 = attend(q, k, v, kc, vc, qw, kw, inv, pos, nh, nkv, hd)
        qr, kr = turned(q, qw, pos), turned(k, kw, pos)
        assert torch.equal(v1[:, pos], v.view(nkv, hd)) and bool(((k1[:, pos].double() - kr).abs() <= 2.0 ** -7 * kr.abs() + 2.0 ** -9).all())
        rest = [i for i in (pos - 1, pos + 1) if 0 <= i < cap]
        assert torch.equal(k1[:, rest], kc[0][:, rest]) and torch.equal(v1[:, rest], vc[0][:, rest])
        ks, vs = (t[:, :pos + 1].double().repeat_interleave(rep, 0) for t in (k1, v1))
        p = torch.softmax((ks @ qr.unsqueeze(-1)).squeeze(-1) * hd ** -0.5, -1)
        want = (p.unsqueeze(1) @ vs).squeeze(1)
        off = 3 * 2.0 ** -8 * hd ** -0.5 * (ks.square() @ qr.square().unsqueeze(-1)).sqrt().amax(1)
        room = 2.0 ** -8 * want.abs() + 2 * off * (p.unsqueeze(1) @ vs.abs()).squeeze(1)
        assert bool(((got.view(nh, hd).double() - want).abs() <= room).all())


@pytest.mark.parametrize("hd,nh,nkv", HEADS[:5])
@pytest.mark.parametrize("cap", [256, 768, 1023])
def test_split_context_against_a_batch_of_the_same_sequence_twice(hd, nh, nkv, cap):
    """Batches are not split at these sizes.  The two sums run over the same products in another order (fp32), their result is rounded once."""
    from gbx_lm_amd import _lib
    assert _lib.lib().gbx_attn_workspace_bytes(-1, nh, nkv, hd, cap) > 0 and _lib.lib().gbx_attn_workspace_bytes(-2, nh, nkv, hd, cap) == 0
    q, k, v, kc, vc, qw, kw, inv = operands(hd, nh, nkv, cap)
    for pos in (0, 1, 15, 31, 32, 47, 63, cap - 1):
        (one, k1, v1), (two, k2, v2) = (attend(q, k, v, kc, vc, qw, kw, inv, pos, nh, nkv, hd, b) for b in (1, 2))
        assert torch.equal(k1, k2) and torch.equal(v1, v2)
        one, two = one.float(), two.float()
        assert bool(((one - two).abs() <= 2.0 ** -7 * two.abs() + 2.0 ** -16 * vc.float().abs().max()).all())


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,n", [(1, 24576), (1, 24577), (15, 24584), (16, 24584), (2, 26623), (1, 28672), (1, 28673), (3, 50257)])
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


@pytest.mark.parametrize("normed,cap", [(False, 256), (False, 768), (False, 4096), (True, 128), (True, 512)])
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
    split = _lib.lib().gbx_attn_workspace_bytes(-1 if normed else 1, nh, nkv, hd, cap) > 0
    assert split == (normed and cap >= 256 or cap == 4096) and (torch.cuda.max_memory_allocated() > before) == split
