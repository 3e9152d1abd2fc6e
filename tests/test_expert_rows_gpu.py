"""Row kernels of routed experts (csrc/mixers_moe.hip) at the edges of the vector form: contractions of one vector, around a step of 16 lanes and around the
steps in flight, channels that end inside a workgroup's 16, both types, every expert form, a factor per pair; beside sizes and addresses that take
the element form.  Reference: float64 of the same numbers.  Tolerance: fp32 sums of the terms' magnitudes, the hidden row and the result
rounded to the activation type once each, fast transcendentals (a few ulp of fp32) where that is bf16."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,f,off", [(8, 8, 0), (120, 16, 0), (128, 136, 0), (136, 24, 0), (512, 520, 0), (520, 504, 0), (2048, 768, 0), (12, 40, 0), (20, 7, 0), (128, 64, 1)])
@pytest.mark.parametrize("kind,scaled", [("silu", False), ("clamped_swish", True), ("relu2", True)])
def test_rows(dt, k, f, off, kind, scaled):
    rows(dt, k, f, off, kind, scaled, torch.tensor([[4, 0], [2, 4], [1, 2]], dtype=torch.int32, device=DEV), 5)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,f", [(8, 8), (136, 24), (264, 520)])
@pytest.mark.parametrize("t,e", [(8, 5), (9, 32), (15, 3), (1, 1)])
def test_runs_of_pairs(dt, k, f, t, e):
    """Pairs that share experts, blocks of channels in runs: both terms of the rule, units on and off the eighth."""
    top = min(2, e)
    idx = torch.stack([(torch.arange(top) * 7 + 5 * i + i // 3) % e for i in range(t)]).to(torch.int32).to(DEV)
    for kind in ("silu", "relu2"):
        rows(dt, k, f, 0, kind, False, idx, e)


def rows(dt, k, f, off, kind, scaled, idx, e):
    from gbx_lm_amd import mixer_ops as M
    t, top = idx.shape
    g = torch.Generator(device=DEV).manual_seed(k + f)
    rnd = lambda *s: torch.randn(s, device=DEV, generator=g).to(dt)
    h = torch.empty(t * k + off, dtype=dt, device=DEV)[off:].view(t, k).copy_(rnd(t, k))
    first, down = rnd(e, f * (1 if kind == "relu2" else 2), k) * k ** -0.5, rnd(e, k, f) * f ** -0.5
    scale = torch.rand((t, top), device=DEV, generator=g) + 0.5 if scaled else None
    got = M.expert_glu(h, first, down, idx, kind, 1.5, scale).double()
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -22
    for r in range(t):
        for s in range(top):
            w1, w2 = first[idx[r, s]].double(), down[idx[r, s]].double()
            z, mag = w1 @ h[r].double(), w1.abs() @ h[r].double().abs()
            m = 1.0 if scale is None else scale[r, s].double()
            z, slack = z * m, (k + 2) * 2.0 ** -24 * mag * m
            if kind == "relu2":
                a, room = z.clamp(min=0) ** 2, 2 * (z.abs() + slack) * slack
            else:
                u, v = z[:f], z[f:]
                room = 3 * (slack[:f] * (v.abs() + 2) + slack[f:] * (u.abs() + 1)) + 2.0 ** -20 * u.abs() * (v.abs() + 1)
                if kind == "clamped_swish":
                    u, v = u.clamp(max=1.5), v.clamp(-1.5, 1.5)
                    a = u * torch.sigmoid(1.702 * u) * (v + 1)
                else:
                    a = u * torch.sigmoid(u) * v
            want = w2 @ a
            bound = w2.abs() @ (room + eps * a.abs() + f * 2.0 ** -24 * a.abs()) + eps * want.abs() + 1e-9
            assert bool(((got[r, s] - want).abs() <= bound).all()), (r, s)
