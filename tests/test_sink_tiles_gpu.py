"""Softmax attention of prompt portions (csrc/mixers_sink_mfma.hip) on both sides of the rule that gives a query tile one or two groups of waves,
at lengths around 32, 64 and 128 keys, with windows that end inside a tile, sinks, and head factors of either sign and zero.  Reference:
float64 from the same bf16 rows.  Tolerance: weights are rounded to bf16 for the value product, 2^-8 of each, independent of each other; the
result is rounded once: 2^-8 (|y| + the root of the sum of squared terms), 3 x for the extremes; 2^-16 of the terms' absolute sum for the
fp32 scores and exponentials (scores of up to 2^5)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FEW = [1, 33, 64, 65, 129, 300]
MANY = [1 + (37 * i) % 170 for i in range(140)]


@pytest.mark.parametrize("lens", [FEW, MANY], ids=["two-groups", "one-group"])
@pytest.mark.parametrize("dk,dv", [(32, 32), (128, 128), (192, 128), (72, 40)])
@pytest.mark.parametrize("window", [None, 1, 65])
def test_portions(lens, dk, dv, window):
    assert (len(lens) > 100) == (sum((n + 127) // 128 for n in lens) * 8 > 960)
    portions(lens, dk, dv, window)


@pytest.mark.parametrize("lens", [[7], [1, 31, 32, 33, 64], [48 - (7 * i) % 48 for i in range(130)], [128 - (37 * i) % 128 for i in range(200)]],
                         ids=["one", "few up to 64", "many up to 48", "many up to 128"])
@pytest.mark.parametrize("dk,dv", [(32, 32), (128, 128), (72, 40)])
@pytest.mark.parametrize("window", [None, 33])
def test_sequences_of_a_tile_and_less(lens, dk, dv, window):
    """The form for short sequences and, of the last list, heads on either side of its rule."""
    portions(lens, dk, dv, window)


def portions(lens, dk, dv, window):
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.batching import StepBatch
    gen = torch.Generator(device=DEV).manual_seed(dk + len(lens))
    H, G, T = 8, 2, sum(lens)
    batch = StepBatch.build(list(range(len(lens))), [0] * len(lens), lens, DEV)
    q, k, v = (torch.randn((T, n, d), device=DEV, generator=gen).to(torch.bfloat16) for n, d in ((H, dk), (G, dk), (G, dv)))
    sink = torch.randn(H, device=DEV, generator=gen)
    factor = torch.tensor([1.0, -1.0, 0.5, 0.0, 1.3, 2.0, -0.7, 1.0], device=DEV)
    got = M.sink_attention(q, k, v, None, batch, dk ** -0.5, window, 0, sink, head_scale=factor).double().view(T, H, dv)
    r0 = 0
    for n in lens:
        i = torch.arange(n, device=DEV)
        hidden = (i[None] > i[:, None]) | ((i[:, None] - i[None] >= window) if window else False)
        for h in range(H):
            qq, kk, vv = (t[r0:r0 + n].double() for t in (q[:, h], k[:, h // 4], v[:, h // 4]))
            s = (qq @ kk.t() * (dk ** -0.5 * factor[h].double())).masked_fill(hidden, float("-inf"))
            den = torch.logaddexp(torch.logsumexp(s, -1, keepdim=True), sink[h].double())
            p = torch.exp(s - den)
            want, spread, total = p @ vv, (p ** 2 @ vv ** 2).sqrt(), p @ vv.abs()
            err = (got[r0:r0 + n, h] - want).abs()
            assert bool((err <= 3 * 2.0 ** -8 * (want.abs() + spread) + 2.0 ** -16 * total + 1e-6).all()), (n, h, float(err.max()))
        r0 += n


@pytest.mark.parametrize("count,rows,dk,dv", [(128, 120, 128, 128), (113, 128, 192, 128), (61, 250, 72, 64), (43, 257, 64, 64), (40, 300, 32, 32), (30, 1000, 32, 32), (63, 128, 256, 256),
                                              (13, 1100, 96, 96), (12, 1200, 96, 96)])
def test_sequences_of_one_length(count, rows, dk, dv):
    """Two tiles a workgroup -- odd and even numbers of them, one and several a sequence -- and the forms that small heads take instead."""
    portions([rows] * (count - 1) + [rows - 7], dk, dv, None)


@pytest.mark.parametrize("window,keep", [(None, 0), (256, 0), (200, 5), (96, 70), (33, 0)])
@pytest.mark.parametrize("dk,dv,H", [(64, 64, 8), (192, 128, 8), (128, 120, 8), (128, 128, 48)])
def test_portions_behind_a_history(window, keep, dk, dv, H):
    """Key tiles that lie whole in the table or in the step's rows, and those that the kept rows, the ring's seam or the first new row cuts; rows
    further apart than a head.  The last shape takes the form of one group."""
    behind([0, 1, 64, 130, 515, 1000], [300, 129, 64, 200, 33, 140], window, keep, dk, dv, H, 2)


@pytest.mark.parametrize("window,keep", [(None, 0), (200, 5), (33, 0)])
@pytest.mark.parametrize("dk,dv,H,G,values", [(64, 64, 8, 2, True), (128, 128, 16, 4, True), (128, 104, 16, 4, True), (96, 96, 40, 1, True), (256, 256, 8, 2, True), (576, 512, 16, 1, False),
                                              (512, 512, 16, 1, False), (256, 256, 8, 1, False), (560, 512, 16, 1, False), (320, 256, 8, 1, False), (96, 96, 36, 1, False)])
@pytest.mark.parametrize("rows", [1, 7, 300])
def test_single_rows_behind_a_history(window, keep, dk, dv, H, G, values, rows):
    """One row a sequence: heads that fill their capacity and heads that do not, groups of more than 32, values of their own and values that are the
    keys', key tiles shared out over many workgroups and one workgroup for all."""
    first = [(37 * i * i + 11 * i) % (700 if rows < 300 else 90) for i in range(rows)]
    first[0] = 650 if rows < 300 else 89
    behind(first, [1] * rows, window, keep, dk, dv, H, G, values)


@pytest.mark.parametrize("dk,dv,H,G", [(64, 64, 8, 2), (128, 104, 16, 4), (128, 128, 16, 4), (256, 256, 8, 2)])
@pytest.mark.parametrize("first", [[0], [40, 3, 31], [700] + [32 * i + 5 for i in range(20)]])
def test_an_infinite_value_of_the_newest_row(dk, dv, H, G, first):
    """The last tile of keys is not full: what lies behind the newest row adds nothing to its infinity."""
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.batching import StepBatch
    from gbx_lm_amd.models.cache import SequenceSlots, SlotKVCache
    gen, n = torch.Generator(device=DEV).manual_seed(dk + len(first)), len(first)
    cache = SlotKVCache(G * dk, G * dv, None, 0, SequenceSlots(n))
    cache.reserve(max(first) + 1, torch.bfloat16, torch.device(DEV))
    cache.keys.normal_(generator=gen)
    cache.values.normal_(generator=gen)
    q, k, v = (torch.randn((n, h, d), device=DEV, generator=gen).to(torch.bfloat16) for h, d in ((H, dk), (G, dk), (G, dv)))
    v[:, :, 3], v[:, :, dv - 2] = float("inf"), float("-inf")
    got = M.sink_attention(q, k, v, cache, StepBatch.build(list(range(n)), first, [1] * n, DEV), dk ** -0.5, None, 0, None).float().view(n, H, dv)
    assert bool((got[..., 3] == float("inf")).all()) and bool((got[..., dv - 2] == float("-inf")).all())
    got[..., 3] = got[..., dv - 2] = 0
    assert bool(got.isfinite().all())


@pytest.mark.parametrize("lens,dk,dv,H", [([130], 64, 64, 8), ([300], 128, 128, 2), ([300], 192, 128, 2), ([300] * 8, 64, 64, 32), ([300] * 8, 128, 128, 32), ([300], 256, 256, 2),
                                          ([300] * 3, 96, 96, 4)])
@pytest.mark.parametrize("sink", [False, True])
def test_values_near_the_end_of_the_range(lens, dk, dv, H, sink):
    """A key of a later tile outweighs those before it by 2^4.3 .. 2^7.9: its value of 2e38 stays finite.  Weights round to bf16 (2^-8), the result
    once more."""
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.batching import StepBatch
    T = sum(lens)
    for score in (3.0, 4.85, 5.5):
        q, k, v = (torch.zeros((T, H, d), device=DEV, dtype=torch.bfloat16) for d in (dk, dk, dv))
        q[..., 0] = 1.0
        rows = [sum(lens[:b]) + 128 for b in range(len(lens))]
        k[rows, :, 0], v[rows] = score, 2e38
        score = float(k[rows[0], 0, 0])
        got = M.sink_attention(q, k, v, None, StepBatch.build(list(range(len(lens))), [0] * len(lens), lens, DEV), 1.0, None, 0,
                               torch.zeros(H, device=DEV) if sink else None).double().view(T, H, dv)
        for r, n in zip(rows, lens):
            i = torch.arange(128, n, device=DEV, dtype=torch.float64)
            e = torch.exp(torch.tensor(score, dtype=torch.float64, device=DEV))
            want = (float(v[r, 0, 0]) * e / (i + sink + e))[:, None, None]
            assert bool(((got[r:r + n - 128] - want).abs() <= 2.0 ** -6 * want).all()), (score, n)


def behind(first, lens, window, keep, dk, dv, H, G, values=True):
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.batching import StepBatch
    from gbx_lm_amd.models.cache import SequenceSlots, SlotKVCache
    gen = torch.Generator(device=DEV).manual_seed(dk + dv + H)
    T, n = sum(lens), len(lens)

    def rows(count, heads, d):
        return torch.randn((count, heads * d + 24), device=DEV, generator=gen).to(torch.bfloat16)[:, 8:8 + heads * d].view(count, heads, d)

    cache = SlotKVCache(G * dk, G * dv if values else 0, window, keep, SequenceSlots(n))
    cache.reserve(max(f + c for f, c in zip(first, lens)), torch.bfloat16, torch.device(DEV))
    past = []
    for b, f in enumerate(first):
        k = rows(f, G, dk)
        past.append((k, rows(f, G, dv) if values else k[..., :dv]))
        p = torch.arange(f, device=DEV)
        p = p[(p < cache.keep) | (p >= f - cache.ring)]            # (later positions of a ring take the places of earlier ones)
        at = cache.row_of(p)
        cache.keys[b, at] = k[p].reshape(-1, G * dk)
        if values:
            cache.values[b, at] = past[b][1][p].reshape(-1, G * dv)
    batch = StepBatch.build(list(range(n)), first, lens, DEV)
    q, k = rows(T, H, dk), rows(T, G, dk)
    v = rows(T, G, dv) if values else k[..., :dv]
    sink = torch.randn(H, device=DEV, generator=gen)
    got = M.sink_attention(q, k, v, cache, batch, dk ** -0.5, window, keep, sink).double().view(T, H, dv)
    r0 = 0
    for b, (f, c) in enumerate(zip(first, lens)):
        i, j = torch.arange(f, f + c, device=DEV)[:, None], torch.arange(f + c, device=DEV)[None]
        hidden = (j > i) | ((i - j >= window) & (j >= keep) if window else torch.zeros_like(j, dtype=torch.bool))
        kk, vv = (torch.cat([old, new[r0:r0 + c]]).double().repeat_interleave(H // G, 1).transpose(0, 1) for old, new in zip(past[b], (k, v)))
        s = torch.matmul(q[r0:r0 + c].double().transpose(0, 1), kk.transpose(1, 2).contiguous()) * dk ** -0.5
        s = s.masked_fill(hidden, float("-inf"))
        p = torch.exp(s - torch.logaddexp(torch.logsumexp(s, -1, keepdim=True), sink.double()[:, None, None]))
        want, spread, total = (x.transpose(0, 1) for x in (torch.matmul(p, vv.contiguous()), torch.matmul(p ** 2, vv.contiguous() ** 2).sqrt(), torch.matmul(p, vv.contiguous().abs())))
        err = (got[r0:r0 + c] - want).abs()
        assert bool((err <= 3 * 2.0 ** -8 * (want.abs() + spread) + 2.0 ** -16 * total + 1e-6).all()), (b, float(err.max()))
        r0 += c
