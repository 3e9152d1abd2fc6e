"""Rows of recurrent mixers in groups of four channels (csrc/mixers_state.hip, mixers_headscan.hip): preparation with and without a convolution, one row a thread and
eight, sequences that start, go on or end inside a thread's rows, a slot used before, and both norms, against the forms for any layout (the same
tensors one element off the grid of their loads).  Tolerance: sums of up to 4096 squares in another order, 2^-20 in fp32, and one rounding to bf16."""
import pytest
import torch

from gbx_lm_amd import mixer_ops as M
from gbx_lm_amd.batching import StepBatch
from gbx_lm_amd.models import recurrent_mixers as RM
from gbx_lm_amd.models.cache import SequenceSlots

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def off(t):
    """The same values one element past an allocation's start."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    return flat.copy_(t)


def step(lens, first):
    slots = SequenceSlots(len(lens) + 1)
    return StepBatch.build([i + 1 for i in range(len(lens))], first, lens, DEV), slots


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens,first", [([5], [0]), ([1, 1, 1], [4, 0, 9]), ([700, 3, 1, 501], [0, 2, 0, 1]), ([1100, 1], [7, 3])])
@pytest.mark.parametrize("conv,unit,G,H,dk,dv", [(True, True, 2, 4, 64, 32), (False, False, 4, 4, 256, 64), (True, False, 3, 3, 4, 8), (False, True, 1, 2, 128, 260)])
def test_recurrent_prepare(dt, lens, first, conv, unit, G, H, dk, dv):
    prepare(dt, lens, first, conv, unit, G, H, dk, dv)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens,first", [([700, 3, 1, 2, 501], [0, 2, 1, 0, 5]), ([1] * 9 + [850], [i % 5 for i in range(10)]), ([901, 8, 1, 8, 5], [3, 0, 4, 1, 2])])
@pytest.mark.parametrize("conv,unit,G,H,dk,dv", [(True, True, 16, 32, 128, 128), (False, False, 16, 32, 128, 128), (True, False, 40, 40, 64, 64)])
def test_recurrent_prepare_eight_rows_a_thread(dt, lens, first, conv, unit, G, H, dk, dv):
    """Enough rows and channels for that form: sequences that start, go on and end inside a thread's eight, and a last thread of fewer."""
    cols = -(-(2 * G * dk + H * dv + H * dk) // 1024)
    assert sum(lens) * cols >= 8192 and sum(lens) % 8
    prepare(dt, lens, first, conv, unit, G, H, dk, dv)


def prepare(dt, lens, first, conv, unit, G, H, dk, dv):
    T, nq, nv = sum(lens), G * dk, H * dv
    batch, slots = step(lens, first)
    lay = RM.RecurrentLayout(H, G, dk, dv, 0, nq, 2 * nq, 2 * nq + nv)
    gen = torch.Generator(device=DEV).manual_seed(T + dk)
    pad = -(2 * nq + nv + H) % 4
    y = torch.randn((T, 2 * nq + nv + H + pad), device=DEV, generator=gen).to(dt)
    a = (torch.randn((T, H * dk), device=DEV, generator=gen) * 2).to(dt)
    bias, rate = torch.randn(H * dk, device=DEV, generator=gen), torch.rand(H, device=DEV, generator=gen) + 0.1
    taps = (torch.randn((2 * nq + nv, 4), device=DEV, generator=gen) * 0.7).to(dt) if conv else None
    cache = RM.SlotStateCache(H, dk, dv, 2 * nq + nv if conv else 0, 4 if conv else 0, slots)
    cache.reserve(dt, DEV)
    if conv:
        cache.tail.normal_(generator=gen)
    got = M.recurrent_prepare(y, a, lay, bias, rate, 1.0, taps, cache, batch, unit, 0.3, qkv_silu=not conv)
    want = M.recurrent_prepare(off(y), off(a), lay, bias, rate, 1.0, taps, cache, batch, unit, 0.3, qkv_silu=not conv)
    assert bool(((got - want).abs() <= 2.0 ** -20 * (1 + want.abs())).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lens,first", [([3000], [0]), ([1500, 2, 1, 1400], [3, 0, 1, 2])])
def test_ssm_prepare(dt, lens, first):
    H, dv, N, G = 8, 64, 64, 1
    C, T = H * dv + 2 * G * N + 2048, sum(lens)
    batch, slots = step(lens, first)
    gen = torch.Generator(device=DEV).manual_seed(T)
    y = torch.randn((T, C + H), device=DEV, generator=gen).to(dt)
    conv, bias = (torch.randn((4, C), device=DEV, generator=gen) * 0.7).to(dt), torch.randn(C, device=DEV, generator=gen)
    dt_bias, rate = torch.randn(H, device=DEV, generator=gen), torch.rand(H, device=DEV, generator=gen)
    from gbx_lm_amd import _lib
    import ctypes
    tail = torch.randn((len(lens) + 1, 3, C), device=DEV, generator=gen).to(dt)
    outs = []
    for rows in (y, off(y)):
        out, dts = torch.empty((T, C), dtype=dt, device=DEV), torch.empty((T, 2 * H), device=DEV)
        p = _lib.SsmPrepareArgs()
        p.y, p.y_stride, p.conv, p.bias, p.tail = rows.data_ptr(), rows.stride(0), conv.data_ptr(), bias.data_ptr(), tail.data_ptr()
        p.dt_bias, p.rate, p.seq, p.tok, p.out, p.dt_out = dt_bias.data_ptr(), rate.data_ptr(), batch.seq.data_ptr(), batch.tok.data_ptr(), out.data_ptr(), dts.data_ptr()
        p.T, p.C, p.H, p.taps, p.off_x, p.off_dt, p.move_tail, p.act = T, C, H, 4, 0, C, 0, M._act(rows, "rows")
        _lib.check_mixers(_lib.mixers().gbxm_ssm_prepare(ctypes.byref(p), torch.cuda.current_stream().cuda_stream))
        outs.append((out, dts))
    last = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -20            # (a bf16 value beside a tie may round either way)
    assert all(bool(((u.float() - v.float()).abs() <= last * (2.0 ** -12 + v.float().abs())).all()) for u, v in zip(*outs))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_norms(dt):
    gen = torch.Generator(device=DEV).manual_seed(3)
    last = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -20            # (a bf16 value beside a tie may round either way)

    def same(u, v):
        assert bool(((u.float() - v.float()).abs() <= last * v.float().abs() + 2.0 ** -30).all())

    for rows, heads, dv, kind, weighted in ((1, 1, 4, "silu", True), (37, 5, 64, "sigmoid", False), (3, 8, 256, "silu", True), (70, 33, 128, "silu", True)):
        o, gate = torch.randn((rows, heads * dv), device=DEV, generator=gen), torch.randn((rows, heads * dv), device=DEV, generator=gen).to(dt)
        w = torch.rand(dv, device=DEV, generator=gen) if weighted else None
        same(M.head_norm_gate(o, gate, w, heads, 1e-5, 1 if kind == "silu" else 2), M.head_norm_gate(o, off(gate), w, heads, 1e-5, 1 if kind == "silu" else 2))
    for rows, groups, size in ((1, 1, 4), (9, 3, 252), (5, 2, 260), (5, 8, 512), (3, 3, 516), (6, 1, 1024), (4, 2, 1028), (2, 1, 2048), (4, 2, 2056), (3, 1, 3072), (2, 2, 3076), (3, 1, 4096)):
        o, gate = torch.randn((rows, groups * size), device=DEV, generator=gen), torch.randn((rows, groups * size), device=DEV, generator=gen).to(dt)
        w = torch.rand(groups * size, device=DEV, generator=gen)
        same(M.gate_group_norm(o, gate, w, groups, 1e-5), M.gate_group_norm(o, off(gate), w, groups, 1e-5))
