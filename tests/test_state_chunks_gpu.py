"""Prompt portions of the decayed states by chunks of 16 tokens (csrc/mixers_state_mfma.hip): sequences on either side of the fewest rows that go that way, whole chunks
and remainders, key channels in and off the 64s, value channels off the 16s, rows or value channels that are not in groups of four (token by token), fresh and carried states, decays down to zero, and numbers that the chunks leave to the
token-by-token form (infinities, NaN, decays above one, numbers whose products might not stay finite).  Reference: float64 token by token; tolerance: fp32 sums
over the key channels, the chunk's tokens and the tokens that a decay keeps, relative to the sums of absolute values."""
import pytest
import torch

from gbx_lm_amd.batching import StepBatch
from gbx_lm_amd.models import recurrent_mixers as RM
from gbx_lm_amd.models.cache import SequenceSlots, SlotStateCache

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def step(dk, dv, H, G, counts, delta, low, spoil=None):
    g = torch.Generator().manual_seed(dk + dv + counts[0])
    lay = RM.RecurrentLayout(H, G, dk, dv, 0, G * dk, 2 * G * dk, 2 * G * dk + H * dv if delta else -1)
    T, B = sum(counts), len(counts)
    q = torch.randn((T, G * dk), generator=g)
    k = torch.nn.functional.normalize(torch.randn((T, G, dk), generator=g), dim=-1).view(T, G * dk)
    v, d = torch.randn((T, H * dv), generator=g), torch.rand((T, H * dk), generator=g) * (1 - low) + low
    if low == 0:
        d[torch.rand(d.shape, generator=g) < 0.05] = 0.0
    beta = torch.rand((T, H), generator=g)
    if spoil:
        spoil(q, k, v, d, beta)
    r = torch.cat([q, k, v, d] + ([beta] if delta else []), 1)
    cache = SlotStateCache(H, dk, dv, 0, 0, SequenceSlots(B))
    cache.reserve(torch.float32, DEV)
    start = torch.randn(cache.state.shape, generator=g)
    cache.state.copy_(start)
    slots, pos = [B - 1 - i for i in range(B)], [0 if i % 2 else 5 for i in range(B)]
    out = RM.decayed_state_scan(r.to(DEV), lay, cache, StepBatch.build(slots, pos, list(counts), DEV), delta).cpu().double().view(T, H, dv)
    rep, r0 = H // G, 0
    for slot, pos0, n in zip(slots, pos, counts):
        S = start[slot].double().clone() if pos0 else torch.zeros_like(start[slot].double())          # [H, dv, dk]
        want, room = [], 1.0
        for t in range(r0, r0 + n):
            kt, qt = (x[t].double().view(G, 1, dk).repeat_interleave(rep, 0) for x in (k, q))
            S = S * d[t].double().view(H, 1, dk)
            u = v[t].double().view(H, dv)
            if delta:
                u = beta[t].double().view(H, 1) * (u - (S * kt).sum(-1))
            S = S + u.unsqueeze(-1) * kt
            want.append((S * qt).sum(-1))
            room = max(room, float((S.abs() * qt.abs()).sum(-1).nan_to_num(0, 0, 0).amax()))
        yield out[r0:r0 + n], torch.stack(want), room, cache.state[slot].cpu().double(), S
        r0 += n


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("dk,dv,H,G", [(64, 16, 4, 2), (128, 36, 4, 2), (100, 18, 4, 1), (192, 20, 4, 1), (256, 16, 4, 4), (128, 17, 4, 4), (128, 16, 3, 1)])
@pytest.mark.parametrize("counts,low", [((127, 128, 1, 129), 0.5), ((144, 40, 177), 0.9), ((200,), 0.0)])
def test_chunks(dk, dv, H, G, counts, low, delta):
    for out, want, room, state, S in step(dk, dv, H, G, counts, delta, low):
        bound = (dk + 60) * 2.0 ** -24 * 4
        assert float((out - want).abs().max()) < bound * room
        assert float((state - S).abs().max()) < bound * max(float(S.abs().max()), 1.0)


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("what", ["nan value", "inf value", "nan key", "growing decay", "large key"])
def test_left_to_the_tokens(what, delta):
    """Each token before the odd number stays exact, and what the token-by-token form gives is not finite in the same places."""
    def spoil(q, k, v, d, beta):
        if what == "nan value":
            v[37, 3] = float("nan")
        elif what == "inf value":
            v[37, 3] = float("inf")
        elif what == "nan key":
            k[37, 70] = float("nan")
        elif what == "growing decay":
            d[37, 5] = 1.5
        else:
            k[37, 5] = 1e13
    for out, want, room, state, S in step(128, 32, 4, 1, (144, 130), delta, 0.5, spoil):
        assert torch.equal(out.isfinite(), want.isfinite())
        if what in ("growing decay",):
            assert float((out - want).abs().max()) < 200 * 2.0 ** -24 * 4 * room
        assert float((out[:37] - want[:37]).abs().max()) < 200 * 2.0 ** -24 * 4 * 100


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("dk,dv,H,short,long", [(128, 36, 4, [127, 1, 64], [130]), (64, 16, 16, [3] * 299, [128]), (192, 16, 4, [40, 9], [128, 200]), (256, 32, 4, [33], [144])])
def test_the_others_of_the_step(dk, dv, H, short, long, delta):
    """Short sequences give the same bits beside long ones as without them: in the chunks' launch (few column blocks) and in one of their own."""
    g = torch.Generator().manual_seed(dk + dv)
    lay = RM.RecurrentLayout(H, H, dk, dv, 0, H * dk, 2 * H * dk, 2 * H * dk + H * dv if delta else -1)
    counts = short[:1] + long + short[1:]
    rows = [torch.rand((n, 3 * H * dk + H * dv + (H if delta else 0)), generator=g) * 0.9 / dk ** 0.25 for n in counts]
    start = torch.randn((len(counts), H, dv, dk), generator=g)

    def scan(which):
        cache = SlotStateCache(H, dk, dv, 0, 0, SequenceSlots(len(counts)))
        cache.reserve(torch.float32, DEV)
        cache.state.copy_(start)
        batch = StepBatch.build(which, [0 if i % 2 else 5 for i in which], [counts[i] for i in which], DEV)
        out = RM.decayed_state_scan(torch.cat([rows[i] for i in which]).to(DEV), lay, cache, batch, delta)
        return dict(zip(which, out.split([counts[i] for i in which]))), cache.state

    few = [i for i, n in enumerate(counts) if n < 128]
    (whole, state), (alone, kept) = scan(list(range(len(counts)))), scan(few)
    for i in few:
        assert torch.equal(whole[i], alone[i]) and torch.equal(state[i], kept[i])


@pytest.mark.parametrize("delta", [False, True])
@pytest.mark.parametrize("what", ["inf state", "nan state", "sums beyond the range"])
def test_carried_states_that_are_not_numbers(what, delta):
    """A state with an infinity behind a chunk's decays, and sums of finite numbers that leave the range inside one: as token by token, to the bit;
    other columns as ever."""
    H, dk, dv, n = 4, 128, 48, 150
    g = torch.Generator().manual_seed(3)
    lay = RM.RecurrentLayout(H, H, dk, dv, 0, H * dk, 2 * H * dk, 2 * H * dk + H * dv if delta else -1)
    r = torch.rand((n, 3 * H * dk + H * dv + (H if delta else 0)), generator=g) * 0.9
    r[:, :2 * H * dk] /= dk ** 0.5
    start = torch.randn((1, H, dv, dk), generator=g)
    if what == "sums beyond the range":
        r[:, 2 * H * dk + H * dv:3 * H * dk + H * dv] = 1.0
        start[0, 1, 20] = 2e38
        r[n // 2:, H * dk + dk:H * dk + 2 * dk] = 1e6
        r[n // 2:, 2 * H * dk + dv:2 * H * dk + 2 * dv] = 1e12
    else:
        start[0, 1, 20, 5] = float("inf" if what == "inf state" else "nan")
        r[:, 2 * H * dk + H * dv + dk:2 * H * dk + H * dv + 2 * dk] = 1e-6             # decays whose product over a chunk is zero in 32 bits

    from gbx_lm_amd import _lib
    L, got = _lib.mixers(), []
    seq = torch.tensor([[0, 7, n, 0]], dtype=torch.int32, device=DEV)
    rd = r.to(DEV)
    for nbytes in (L.gbxm_state_scan_workspace(1, n, n, H, dk, dv), 0):
        state, out, ws = start.to(DEV).clone(), torch.empty((n, H * dv), device=DEV), torch.empty((max(nbytes, 1),), dtype=torch.uint8, device=DEV)
        _lib.check_mixers(L.gbxm_state_scan_ws(rd.data_ptr(), rd.stride(0), state.data_ptr(), out.data_ptr(), seq.data_ptr(), 1, n, H, H, dk, dv, int(delta),
                                               ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream))
        got.append((out.cpu(), state.cpu()))
    (out, state), (out1, state1) = got
    assert not bool(state1[0, 1, 20].isfinite().all()) or not bool(out1.isfinite().all())
    wild, heads = torch.arange(dv) // 16 == 1, torch.arange(H) != 1                    # the column block that goes again; heads whose sums are ordinary
    assert torch.equal(out.view(n, H, dv)[:, 1, wild].nan_to_num(7.0), out1.view(n, H, dv)[:, 1, wild].nan_to_num(7.0))
    assert torch.equal(state[0, 1, wild].nan_to_num(7.0), state1[0, 1, wild].nan_to_num(7.0))
    assert torch.equal(out.isnan(), out1.isnan()) and torch.equal(state.isnan(), state1.isnan())
    assert float((out - out1).view(n, H, dv)[:, heads].abs().max()) < (dk + 60) * 2.0 ** -22 * 32
    assert float((state - state1)[0, heads].abs().max()) < (dk + 60) * 2.0 ** -22 * 32


@pytest.mark.parametrize("what,delta", [(what, delta) for what in ("nothing", "nan value", "inf value", "nan key", "growing decay", "large key") for delta in (False, True)] + [("nan beta", True)])
def test_which_form_ran(what, delta):
    """The flags that lead the workspace, [heads][places]: zero for a head of ordinary numbers, and its sums are the chunks'; raised only for the head and the
    sequence whose inputs are not, and what that one gives -- rows before the odd number, later ones and the state -- is the token-by-token form's to the bit.
    A workspace that is a byte short leaves every sequence to that form."""
    from gbx_lm_amd import _lib
    L, H, dk, dv, counts = _lib.mixers(), 4, 128, 32, [40, 150, 144, 9, 200]
    T, B, g = sum(counts), len(counts), torch.Generator().manual_seed(11)
    first = [sum(counts[:b]) for b in range(B)]
    odd, at = 2, first[2] + 37
    width = 3 * H * dk + H * dv
    r = torch.rand((T, width + (H if delta else 0)), generator=g) * 0.9
    r[:, :2 * H * dk] /= dk ** 0.5
    head = {"value": 2 * H * dk + dv + 3, "key": H * dk + dk + 70, "decay": 2 * H * dk + H * dv + dk + 5, "beta": width + 1}
    if what != "nothing":
        kind, name = what.split()
        r[at, head[name]] = {"nan": float("nan"), "inf": float("inf"), "growing": 1.5, "large": 1e13}[kind]
    start = torch.randn((B, H, dv, dk), generator=g)
    seq = torch.tensor([[b, b % 2 * 5, counts[b], first[b]] for b in range(B)], dtype=torch.int32, device=DEV)
    rd, need = r.to(DEV), L.gbxm_state_scan_workspace(B, T, max(counts), H, dk, dv)
    places = T // 16 + B
    assert need > 4 * H * places

    def scan(nbytes):
        state, out, ws = start.to(DEV), torch.empty((T, H * dv), device=DEV), torch.full((need,), 0x5a, dtype=torch.uint8, device=DEV)
        _lib.check_mixers(L.gbxm_state_scan_ws(rd.data_ptr(), rd.stride(0), state.data_ptr(), out.data_ptr(), seq.data_ptr(), B, T, H, H, dk, dv, int(delta),
                                               ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream))
        return out.cpu().view(T, H, dv), state.cpu(), ws.cpu()

    same = lambda a, b: torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(7.0), b.nan_to_num(7.0))
    out, state, ws = scan(need)
    token, kept, _ = scan(0)
    short, shorts, untouched = scan(need - 1)
    assert same(short, token) and same(shorts, kept) and bool((untouched == 0x5a).all())
    flags = ws[:4 * H * places].view(torch.int32).view(H, places)
    for b, n in enumerate(counts):
        rows = slice(first[b], first[b] + n)
        for h in range(H):
            if n >= 128:
                raised = flags[h, first[b] // 16 + b:][:(n + 15) // 16] != 0
                assert bool(raised.any()) == (what != "nothing" and (b, h) == (odd, 1))
            if n < 128 or (what != "nothing" and (b, h) == (odd, 1)):
                assert same(out[rows, h], token[rows, h]) and same(state[b, h], kept[b, h])
            else:
                assert not torch.equal(out[rows, h], token[rows, h])          # (other orders of sums)
                assert float((out - token)[rows, h].abs().max()) < (dk + 60) * 2.0 ** -22 * 32
                assert float((state - kept)[b, h].abs().max()) < (dk + 60) * 2.0 ** -22 * 32
