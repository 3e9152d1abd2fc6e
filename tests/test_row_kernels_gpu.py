"""Row kernels that hold a row in one group of four channels per thread (csrc/mixers_common.h: row_threads): one group, a wave's end, ragged waves, the
widest row, the widths on either side that stay with the looping kernels, candidates beside the eight in flight, a base that is not aligned.
Reference: the torch path in float64 sums; tolerances: a few fp32 roundings of sums of positive terms, results rounded to the activation type."""
import pytest
import torch

from gbx_lm_amd.batching import StepBatch
from gbx_lm_amd.models import residual as R

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROW = {torch.float32: 2e-6, torch.bfloat16: 2.0 ** -8}
WIDTHS = (4, 6, 252, 256, 260, 2048, 4092, 4096, 4100)


def near(got, want, dt):
    tol = ROW[dt]
    return bool(((got.cpu().double() - want).abs() <= tol * want.abs() + 16 * 2.0 ** -24 * want.abs().amax(-1, keepdim=True)).all())


def shifted(x, n):
    """The same values at an address n elements past an allocation's start."""
    buf = torch.empty(x.numel() + n, dtype=x.dtype, device=DEV)
    buf[n:] = x.reshape(-1).to(DEV)
    return buf[n:].view(x.shape)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("s,top,off", [(4, 8, 0), (1, 1, 0), (8, 9, 0), (3, 2, 1)])
def test_streams(width, dt, s, top, off):
    g = torch.Generator().manual_seed(width + s)
    X, y = torch.randn((3, s, width), generator=g), torch.randn((3, top, width) if top > 1 else (3, width), generator=g).to(dt)
    y_mix = torch.rand((3, top), generator=g) if top > 1 else None
    mix, write, read = torch.randn((s, s), generator=g), torch.randn(s, generator=g), torch.rand(s, generator=g) + 0.1
    norm = R.StreamLayerNorm(width, 1e-2)
    norm.weight, norm.bias = torch.rand(width, generator=g) + 0.5, torch.randn(width, generator=g)
    z = y.double() if top == 1 else (y.double() * y_mix.double().unsqueeze(-1)).sum(1)
    Xn = torch.einsum("ij,tiw->tjw", mix.double(), X.double()) + write.double()[None, :, None] * z[:, None]
    bound = torch.einsum("ij,tiw->tjw", mix.double().abs(), X.double().abs()) + write.double().abs()[None, :, None] * (
        y.double().abs() if top == 1 else (y.double().abs() * y_mix.double().unsqueeze(-1)).sum(1))[:, None]
    u, room = (Xn * read.double()[None, :, None]).sum(1), (bound * read.double()[None, :, None]).sum(1)
    sd = (u - u.mean(-1, keepdim=True)).pow(2).mean(-1, keepdim=True).add(norm.eps).sqrt()
    want = (u - u.mean(-1, keepdim=True)) / sd * norm.weight.double() + norm.bias.double()
    dev = lambda t: None if t is None else t.to(DEV)
    nd = R.StreamLayerNorm(width, 1e-2)
    nd.weight, nd.bias = norm.weight.to(DEV), norm.bias.to(DEV)
    Xd = shifted(X, off)
    h = R.hyper_step_(Xd, shifted(y, off), dev(y_mix), dev(mix), dev(write), dev(read), nd, dt)
    terms = (s + top + 4) * 2.0 ** -24
    assert bool(((Xd.cpu().double() - Xn).abs() <= terms * bound).all())
    err = (2 * terms * room.amax(-1, keepdim=True) / sd * norm.weight.double() + ROW[dt] * want.abs() + 2.0 ** -20) * (1 + want.abs())
    assert bool(((h.cpu().double() - want).abs() <= err).all())
    total = R.hyper_step_(shifted(X, off), shifted(y, off), dev(y_mix), dev(mix), dev(write), None, None, dt)
    assert bool(((total.cpu().double() - Xn.sum(1)).abs() <= 2 * terms * bound.sum(1)).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("top,extra,off", [(1, False, 0), (8, True, 0), (9, False, 0), (2, True, 1)])
def test_branch_norm(width, dt, top, extra, off):
    g = torch.Generator().manual_seed(width + top)
    x, y = torch.randn((3, width), generator=g), torch.rand((3, top, width) if top > 1 else (3, width), generator=g).to(dt) + 0.5
    mix, ex = (torch.rand((3, top), generator=g) if top > 1 else None), (torch.rand((3, width), generator=g).to(dt) if extra else None)
    w, nw = torch.rand(width, generator=g) + 0.5, torch.rand(width, generator=g) + 0.5
    unit = lambda v: v / v.pow(2).mean(-1, keepdim=True).add(1e-5).sqrt()
    z = y.double() if top == 1 else (y.double() * mix.double().unsqueeze(-1)).sum(1)
    z = z + ex.double() if extra else z
    new = x.double() + unit(z) * w.double()
    xd = shifted(x, off)
    dev = lambda t: None if t is None else t.to(DEV)
    h = R.branch_norm_add_norm_(xd, shifted(y, off), dev(mix), dev(ex), w.to(DEV), 1e-5, nw.to(DEV), dt)
    assert near(xd, new, torch.float32) and near(h, unit(new) * nw.double(), dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", WIDTHS)
def test_shift(width, dt):
    """Two sequences over two steps: the slot's row is the norm that the next row would have computed, bit for bit."""
    from gbx_lm_amd.models.cache import SequenceSlots, SlotRowCache
    g = torch.Generator().manual_seed(width)
    x, w, shift = torch.randn((9, width), generator=g) + 0.5, torch.rand(width, generator=g) + 0.5, torch.rand(width, generator=g)
    n = x.double() / x.double().pow(2).mean(-1, keepdim=True).add(1e-5).sqrt() * w.double()
    prev = torch.cat([torch.zeros(1, width, dtype=torch.float64), n[:5], torch.zeros(1, width, dtype=torch.float64), n[6:8]])
    want = n + (prev - n) * shift.double()
    slots = SequenceSlots(2)
    slots.length[0] = slots.length[1] = 0
    cache = SlotRowCache(width, "f32", slots)
    cache.reserve(dt, DEV)
    cache.rows.fill_(7.0)
    run = lambda rows, batch: R.norm_token_shift(rows.to(DEV), w.to(DEV), 1e-5, shift.to(DEV), cache, batch, dt)
    whole = run(x, StepBatch.build([0, 1], [0, 0], [6, 3], DEV))
    kept = cache.rows.clone()
    assert near(whole, want, dt) and near(kept[:2], torch.stack([n[5], n[8]]), torch.float32)
    parts = [run(torch.cat([x[:2], x[6:7]]), StepBatch.build([0, 1], [0, 0], [2, 1], DEV)), run(torch.cat([x[2:6], x[7:]]), StepBatch.build([0, 1], [2, 1], [4, 2], DEV))]
    again = torch.cat([parts[0][:2], parts[1][:4], parts[0][2:], parts[1][4:]])
    assert torch.equal(again, whole) and torch.equal(cache.rows[:2], kept[:2])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("top,off", [(1, 0), (8, 0), (9, 0), (2, 1)])
def test_embedding_and_norms(width, dt, top, off):
    """Rows embedded (exact but for the scale's rounding), added behind a norm of one branch or of several candidates, normed."""
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator().manual_seed(width + top)
    table, tok, w = torch.randn((11, width), generator=g).to(dt), torch.tensor([3, 0, 10, 3]), torch.rand(width, generator=g) + 0.5
    x, h = M.embed_scaled(shifted(table, off), tok.to(DEV), 0.7)
    want = table[tok].float() * 0.7
    assert torch.equal(x.cpu(), want) and (h is x or torch.equal(h.cpu(), want.to(dt)))
    y = torch.rand((4, top, width) if top > 1 else (4, width), generator=g).to(dt) + 0.5
    mix = torch.rand((4, top), generator=g) if top > 1 else None
    z = y.double() if top == 1 else (y.double() * mix.double().unsqueeze(-1)).sum(1)
    new = want.double() + 0.3 * z / z.pow(2).mean(-1, keepdim=True).add(1e-5).sqrt() * w.double()
    xd = shifted(want, off)
    h = M.residual_norm_add(xd, shifted(y, off), None if mix is None else mix.to(DEV), w.to(DEV), 1e-5, 0.3, dt)
    assert near(xd, new, torch.float32) and near(h, new, dt)
    n = M.stream_rmsnorm(shifted(want, off), w.to(DEV), 1e-5, dt)
    assert near(n, want.double() / want.double().pow(2).mean(-1, keepdim=True).add(1e-5).sqrt() * w.double(), dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n0,n1,tail,off", [(4096, 512, 512, 0), (256, 256, 0, 0), (260, 4, 8, 0), (2048, 2048, 4, 0), (3840, 260, 0, 0), (6144, 2048, 0, 0), (8192, 512, 0, 0), (6, 4, 2, 0),
                                            (64, 64, 1, 0), (128, 64, 64, 1)])
def test_segments_and_window_rows(n0, n1, tail, off, dt):
    """Two segments of a row normed on their own: one and two groups a thread, the widest that fit, one more, rows off the grid of four; then the rows
    behind the first segment appended to the rings as they are."""
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator().manual_seed(n0 + n1)
    rows, w0, w1 = torch.randn((5, n0 + n1 + tail), generator=g).to(dt), torch.rand(n0, generator=g) + 0.5, torch.rand(n1, generator=g) + 0.5
    d = shifted(rows, off)
    M.segment_rmsnorm_(d, n0, n1, w0.to(DEV), w1.to(DEV), 1e-5)
    unit = lambda v: v.double() / v.double().pow(2).mean(-1, keepdim=True).add(1e-5).sqrt()
    assert near(d[:, :n0], unit(rows[:, :n0]) * w0.double(), dt) and near(d[:, n0:n0 + n1], unit(rows[:, n0:n0 + n1]) * w1.double(), dt)
    assert torch.equal(d[:, n0 + n1:].cpu(), rows[:, n0 + n1:])
    if tail:
        batch = StepBatch.build([1, 0], [0, 2], [3, 2], DEV)
        kc, vc = (torch.zeros((2, 4, n), dtype=dt, device=DEV) for n in (n1, tail))
        M.window_append(d, n0, n1, kc, vc, batch, 4)
        for slot, at, row in ((1, 0, 0), (1, 1, 1), (1, 2, 2), (0, 2, 3), (0, 3, 4)):
            assert torch.equal(kc[slot, at], d[row, n0:n0 + n1]) and torch.equal(vc[slot, at], d[row, n0 + n1:])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", WIDTHS)
@pytest.mark.parametrize("branch,top,mixed,extra,replace,normed,off", [(True, 0, False, False, False, True, 0), (False, 8, True, False, False, True, 0), (True, 9, True, True, True, False, 0),
                                                                         (False, 1, False, True, False, True, 0), (True, 2, True, False, False, True, 1)])
def test_layer_update(width, dt, branch, top, mixed, extra, replace, normed, off):
    """Every part of the sum alone and together, the stream replaced or added to, with and without the next norm; an image at a stride of its own."""
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator().manual_seed(width + top)
    x, w = torch.randn((3, width), generator=g), torch.rand(width, generator=g) + 0.5
    b = torch.randn((3, width), generator=g).to(dt) if branch else None
    cand = torch.randn((3, top, width), generator=g).to(dt) if top else None
    mix = torch.rand((3, top + 1), generator=g) if mixed else None
    ex = torch.randn((3, width), generator=g).to(dt) if extra else None
    parts = [p.double() for p in (None if replace else x, b, ex) if p is not None]
    if top:
        parts += [cand[:, k].double() * (mix[:, k:k + 1].double() if mixed else 1.0) for k in range(top)]
    want, room = sum(parts), sum(p.abs() for p in parts)
    dev = lambda t: None if t is None else shifted(t, off)
    xd, image = shifted(x, off), torch.zeros((3, width + 8), dtype=dt, device=DEV)
    h = M.layer_update_(xd, dev(b), dev(cand), None if mix is None else mix.to(DEV), w.to(DEV) if normed else None, 1e-5, image[:, :width], replace, dev(ex))
    assert bool(((xd.cpu().double() - want).abs() <= (top + 4) * 2.0 ** -24 * room).all())
    assert torch.equal(image[:, :width], xd.to(dt)) and float(image[:, width:].abs().max()) == 0.0
    if normed:
        unit = xd.cpu().double() / xd.cpu().double().pow(2).mean(-1, keepdim=True).add(1e-5).sqrt() * w.double()
        assert near(h, unit, dt)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,heads,n_in,n_out,tail", [(1, 1, 1, 8, 0), (2, 16, 128, 512, 64), (2, 16, 512, 128, 0), (3, 5, 100, 72, 8), (1, 8, 64, 1032, 0), (15, 17, 33, 40, 2), (16, 16, 128, 72, 8)])
def test_a_matrix_per_head(rows, heads, n_in, n_out, tail, dt):
    """Few rows times heads cut into runs of outputs -- a last run that is not full, inputs off the grid of a workgroup -- and one more, uncut; the tail as it is."""
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator().manual_seed(n_in + n_out)
    x, w = torch.randn((rows, heads, n_in + tail), generator=g).to(dt), torch.randn((heads, n_in, n_out), generator=g).to(dt)
    gate = torch.randn((rows, heads * n_out), generator=g).to(dt) if not tail else None
    got = M.head_project(x.to(DEV), w.to(DEV), tail, gate=None if gate is None else gate.to(DEV)).cpu().double()
    z, room = (torch.matmul(a.transpose(0, 1), b).transpose(0, 1) for a, b in ((x[..., :n_in].double(), w.double()), (x[..., :n_in].double().abs(), w.double().abs())))
    f = torch.sigmoid(gate.double()).view(rows, heads, n_out) if gate is not None else 1.0
    assert bool(((got[..., :n_out] - z * f).abs() <= (ROW[dt] if dt == torch.bfloat16 else 2.0 ** -20) * (z * f).abs() + (n_in + 8) * 2.0 ** -24 * room).all())
    assert torch.equal(got[..., n_out:], x[..., n_in:].double())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,n_in,n_out,tail", [(16, 128, 512, 64), (16, 512, 128, 0), (3, 33, 72, 8), (8, 1, 1032, 2), (5, 100, 40, 0), (4, 4100, 24, 0)])
def test_a_matrix_per_head_of_any_number_of_rows(heads, n_in, n_out, tail, dt):
    """A row's bits do not depend on how many others the step has: outputs cut into runs of every length, rows alone and in pairs."""
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator().manual_seed(n_in)
    x, w = torch.randn((260, heads, n_in + tail), generator=g).to(dt).to(DEV), torch.randn((heads, n_in, n_out), generator=g).to(dt).to(DEV)
    whole = M.head_project(x, w, tail)
    for rows in (1, 2, 5, 15, 16, 33, 64, 65, 86, 129):
        assert torch.equal(M.head_project(x[:rows], w, tail), whole[:rows])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("k,v,off", [(8, 4, 0), (576, 0, 0), (6, 4, 0), (8, 6, 0), (8, 8, 1), (1028, 512, 0)])
@pytest.mark.parametrize("window,keep", [(None, 0), (5, 3)])
def test_rows_appended_to_slots(k, v, off, dt, window, keep):
    from gbx_lm_amd import mixer_ops as M
    from gbx_lm_amd.models.cache import SequenceSlots, SlotKVCache
    g = torch.Generator().manual_seed(k + v)
    cache = SlotKVCache(k, v, window, keep, SequenceSlots(2), first_capacity=16)
    cache.reserve(16, dt, torch.device(DEV))
    batch = StepBatch.build([1, 0], [2, 9], [11, 1], DEV)
    kr, vr = torch.randn((12, k), generator=g).to(dt), torch.randn((12, v), generator=g).to(dt) if v else None
    M.slot_append(cache, shifted(kr, off), None if vr is None else shifted(vr, off), batch)
    rows = {}
    for r, (slot, pos) in enumerate([(1, 2 + i) for i in range(11)] + [(0, 9)]):
        rows[(slot, pos if pos < cache.keep else cache.keep + (pos - cache.keep) % cache.ring)] = r
    for (slot, at), r in rows.items():
        assert torch.equal(cache.keys[slot, at].cpu(), kr[r])
        if v:
            assert torch.equal(cache.values[slot, at].cpu(), vr[r])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dv,heads,off", [(256, 1, 0), (260, 3, 0), (1024, 1, 0), (1028, 2, 0), (2044, 1, 0), (2052, 1, 0), (4096, 1, 0), (4100, 1, 0), (2046, 1, 0), (2048, 1, 1)])
@pytest.mark.parametrize("kind,weighed", [(1, True), (2, False)])
def test_norm_of_heads_of_many_channels(dv, heads, off, dt, kind, weighed):
    """fp32 sums of dv squares: at most (dv / 1024 + 10) roundings each way, halved by the root; the product rounds four times more."""
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator().manual_seed(dv)
    o, gate, w = torch.randn((7, heads * dv), generator=g) * 3, torch.randn((7, heads * dv), generator=g).to(dt), torch.rand(dv, generator=g)
    got = M.head_norm_gate(o.to(DEV), shifted(gate, off), w.to(DEV) if weighed else None, heads, 1e-6, kind).cpu().double()
    x, z = o.double().view(7, heads, dv), gate.double().view(7, heads, dv)
    want = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * (w.double() if weighed else 1.0) * torch.sigmoid(z) * (z if kind == 1 else 1.0)
    assert bool(((got - want.view(got.shape)).abs() <= (ROW[dt] if dt == torch.bfloat16 else 2.0 ** -20) * want.view(got.shape).abs() + 1e-30).all())
