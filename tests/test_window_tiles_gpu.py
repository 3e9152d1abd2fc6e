"""Gated window attention of prompt portions (csrc/mixers_attn_mfma.hip) at the edges of its tiles: portions and windows around 32, 64 and 128 keys
and rounds of two key tiles, with and without history in the ring, with and without a soft cap, head sizes of both tile shapes.
Reference: float64 from the same bf16 rows.  Tolerance: gates (up to 1) are rounded to bf16 for the value product, 2^-8 of each, independent
of each other; the result is rounded once: 2^-8 (|y| + the root of the sum of squared terms), 3 x for the extremes, plus what four
approximate transcendentals of 2^-21 each move a gate by, 2^-18 of the terms' absolute sum."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 128), (192, 128), (32, 64)])
@pytest.mark.parametrize("cap", [0.0, 5.0])
@pytest.mark.parametrize("window", [1, 63, 64, 65, 129, 300])
def test_portions(dk, dv, cap, window):
    portions([1, 31, 33, 64, 65, 127, 129, 191, 257, 320], [0, 7, 0, 64, 200, 0, 33, 0, 130, 0], dk, dv, cap, window)


@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 128), (32, 64)])
@pytest.mark.parametrize("cap,window", [(0.0, 33), (5.0, 300)])
def test_more_tiles_than_compute_units(dk, dv, cap, window):
    """One group of waves a tile, tiles of 32 keys: edges of both, beside prompts of a few rows with and without history."""
    portions([1, 31, 32, 33, 63, 65, 129, 257] + [1 + (11 * i) % 40 for i in range(200)], [0, 7, 33, 0, 64, 300, 31, 0] + [(5 * i) % 47 for i in range(200)],
             dk, dv, cap, window)


@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 128), (192, 128), (96, 96)])
@pytest.mark.parametrize("cap,window", [(0.0, 300), (5.0, 9)])
def test_short_sequences_only(dk, dv, cap, window):
    """Up to 48 keys a tile: one buffer of 32 keys."""
    portions([1, 31, 32, 33, 40, 7, 17], [0, 0, 0, 0, 8, 41, 31] if window == 300 else [0, 3, 0, 0, 100, 9, 31], dk, dv, cap, window)


@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 64), (192, 128)])
def test_long_sequences(dk, dv):
    """One group of waves, two buffers, whole tiles in the ring and in the step's rows, the ring's seam inside a tile and at its edge."""
    portions([400, 129, 640, 300, 257, 128, 200, 512], [0, 511, 900, 448, 1024, 512, 64, 700], dk, dv, 5.0, 512)


def portions(n_new, pos0, dk, dv, cap, window):
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.batching import StepBatch
    gen = torch.Generator(device=DEV).manual_seed(window + dk)
    H, G = 4, 2
    T = sum(n_new)
    batch = StepBatch.build(list(range(len(n_new))), pos0, n_new, DEV)
    qkv = torch.randn((T, H * dk + G * (dk + dv)), device=DEV, generator=gen).to(torch.bfloat16)
    kc, vc = (torch.randn((len(n_new), window, G * d), device=DEV, generator=gen).to(torch.bfloat16) for d in (dk, dv))
    vec = lambda lo, hi: torch.rand(H, device=DEV, generator=gen) * (hi - lo) + lo
    m = SimpleNamespace(window=window, nk=G * dk, nv=G * dv, heads=H, kv_heads=G, dim=dk, vdim=dv, dist_mul=vec(0.05, 0.6), dist_rate=vec(0.05, 0.6),
                        gate_bias=vec(-3, 1), scale=dk ** -0.5, softcap=cap)
    got = M.window_attention(qkv, kc, vc, batch, m).double().view(T, H, dv)
    r0 = 0
    for b, (n, p) in enumerate(zip(n_new, pos0)):
        q, k, v = qkv[r0:r0 + n].double().split([H * dk, G * dk, G * dv], -1)
        old = torch.arange(max(0, p - window + 1), p, device=DEV)
        k, v = (torch.cat([c[b, old % window].double(), t]).view(-1, G, d) for c, t, d in ((kc, k, dk), (vc, v, dv)))
        j, i = torch.cat([old, torch.arange(p, p + n, device=DEV)]), torch.arange(p, p + n, device=DEV)
        dist = i[:, None] - j[None]
        for h in range(H):
            s = q[:, h * dk:(h + 1) * dk] @ k[:, h // 2].t() * m.scale
            s = cap * torch.tanh(s / cap) if cap else s
            z = s - m.dist_mul[h].double() * torch.log1p(m.dist_rate[h].double() * dist.clamp(min=0)) + m.gate_bias[h].double()
            g = torch.sigmoid(z).masked_fill((dist < 0) | (dist >= window), 0.0)
            want, spread, total = g @ v[:, h // 2], (g ** 2 @ v[:, h // 2] ** 2).sqrt(), g @ v[:, h // 2].abs()
            err = (got[r0:r0 + n, h] - want).abs()
            assert bool((err <= 3 * 2.0 ** -8 * (want.abs() + spread) + 2.0 ** -18 * total + 1e-6).all()), (n, p, h, float(err.max()))
        r0 += n


@pytest.mark.parametrize("dk,dv", [(64, 64), (128, 128), (192, 128)])
def test_a_soft_cap_below_zero_is_none(dk, dv):
    """In prompt portions as in steps of single tokens: the same bits as without one."""
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.batching import StepBatch
    gen = torch.Generator(device=DEV).manual_seed(dk)
    H, G, W, n_new, pos0 = 4, 2, 100, [1, 140, 1, 33], [30, 0, 7, 64]
    batch = StepBatch.build(list(range(4)), pos0, n_new, DEV)
    qkv = torch.randn((sum(n_new), H * dk + G * (dk + dv)), device=DEV, generator=gen).to(torch.bfloat16)
    kc, vc = (torch.randn((4, W, G * d), device=DEV, generator=gen).to(torch.bfloat16) for d in (dk, dv))
    vec = lambda: torch.rand(H, device=DEV, generator=gen)
    m = SimpleNamespace(window=W, nk=G * dk, nv=G * dv, heads=H, kv_heads=G, dim=dk, vdim=dv, dist_mul=vec(), dist_rate=vec(), gate_bias=vec() - 0.5,
                        scale=dk ** -0.5, softcap=0.0)
    want = M.window_attention(qkv, kc, vc, batch, m)
    m.softcap = -3.0
    assert torch.equal(M.window_attention(qkv, kc, vc, batch, m), want)
