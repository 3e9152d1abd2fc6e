"""Generation whose next step is enqueued before the host has read the tokens (BatchScheduler._step_ahead), and log-probabilities straight from the output head's rows."""
import pytest
import torch

from gbx_lm_amd import _lib, ops, synthetic as S
from gbx_lm_amd.batching import BatchScheduler
from gbx_lm_amd.mixer_ops import log_probabilities

pytestmark = pytest.mark.gpu


def _model(name):
    if name == "tugolix":
        cfg = S.tugolix_config(width=256, delta=dict(heads=4, kv_heads=2, dim=64, vdim=64, conv=4), gla=dict(heads=2, dim=64, vdim=128, tau=16.0),
                               latent=dict(heads=4, dim=64, vdim=64, kv_rank=128), ff=512, moe=dict(experts=8, top=2, ff=128, groups=(4, 2)), pattern="dgls")
        return S.build_tugolix(cfg, device="cuda:0", seed=3), cfg["vocab"]
    cfg = S.gibalorn_config(width=256, latent=dict(heads=4, dim=64, rot_dim=32, vdim=64, kv_rank=128, q_rank=128),
                            mamba2=dict(heads=8, vdim=64, state=64, groups=1, conv=4, norm_groups=1), attention=dict(heads=4, kv_heads=2, dim=64, rot_dims=32),
                            moe=dict(experts=8, top=2, ff=128), pattern="mla")
    return S.build_gibalorn(cfg, device="cuda:0", seed=3), cfg["vocab"]


@pytest.mark.parametrize("name", ["tugolix", "gibalorn"])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
@pytest.mark.parametrize("stops", [{}, {1: 9}, {0: 8, 2: 8}, {0: 7, 1: 8, 2: 9}])
def test_the_same_tokens_and_log_probabilities(name, dtype, stops):
    """Odd numbers of sequences (tables off the grid of 16 bytes), sequences that a token ends at different steps and all at once; a continuation that the caller
    supplies, so that both orders of host and device compute the same rows."""
    model, vocab = _model(name)
    steps, stop = 14, vocab - 1
    gen = torch.Generator().manual_seed(5)
    prompts = [torch.randint(0, stop, (n,), generator=gen).tolist() for n in (5, 1, 12)]
    forced = torch.randint(0, stop, (steps, 3), generator=gen)
    for seq, at in stops.items():
        forced[at, seq] = stop
    runs = []
    for ahead in (True, False):
        engine = BatchScheduler(model)
        took = []
        inner = engine._step_ahead

        def counted(ids, toks):
            got = inner(ids, toks) if ahead else None
            took.append(got is not None)
            return got

        engine._step_ahead = counted
        rows = []
        for again in range(2):                                    # the second time replays what the first captured
            live, n = [0, 1, 2], [0]

            def sampler(lp):
                row = forced[n[0], live].clone()
                rows.append((list(live), lp))
                live[:] = [i for i in live if forced[n[0], i] != stop]
                n[0] += 1
                return row.to("cuda:0", dtype)

            out = engine.generate(prompts, max_tokens=steps, sampler=sampler, stop_tokens=[stop])
            for i in range(3):
                want = forced[:stops.get(i, steps - 1) + 1, i].tolist()
                assert out[i] == want
        assert any(took) == ahead
        assert not engine.slot_of and all(v < 0 for v in engine.slots.length)      # every slot was given back
        runs.append(rows)
    assert len(runs[0]) == len(runs[1])
    first, each = min(stops.values(), default=steps), len(runs[0]) // 2
    for i, ((a, x), (b, y)) in enumerate(zip(*runs)):
        assert a == b and x.shape == y.shape
        if i % each <= first:
            assert torch.equal(x, y)
        # bf16 activations: a step that still holds a sequence which has ended may take another kernel for its rows
        assert (x - y).abs().max() <= 0.05 * y.std()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,n", [(1, 8), (1, 32000), (2, 24584), (3, 24579), (15, 30001), (16, 1003), (33, 8192), (1, 151936)])
@pytest.mark.parametrize("scale", [1.0, 0.25, 3.0])
def test_rows_of_the_head(dtype, rows, n, scale):
    x = (torch.randn((rows, n), generator=torch.Generator(device="cuda").manual_seed(n + rows), device="cuda") * 4).to(dtype)
    got = log_probabilities(x, scale)
    assert got.dtype == torch.float32
    y = x.double() * scale
    want = y - torch.logsumexp(y, -1, keepdim=True)
    # fp32: a product, a difference and a logarithm, each within an ulp of values up to 2^6; n exponentials sum to a relative 2^-24 sqrt(n) at most 2^-15
    assert ((got.double() - want).abs() <= 2.0 ** -17 * want.abs().clamp(min=1.0) + 2.0 ** -15).all()


@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
@pytest.mark.parametrize("b", [1, 5, 256])
def test_tokens_ahead_of_the_host_stay_inside_the_embedding(dtype, b):
    """Ids just outside the table and far from it become token 0; positions go on by one."""
    rows, far = 1000, torch.iinfo(dtype)
    ids = torch.tensor([-1, rows, rows - 1, 0, far.max, far.min, rows + 1, 1, 2 ** 31 - 1, -rows], dtype=dtype).repeat(26)[:b]
    seq, tok = torch.arange(4 * b, dtype=torch.int32), torch.arange(2 * b, dtype=torch.int32)
    dev = [t.to("cuda:0") for t in (ids, torch.full((b,), 7, dtype=torch.int64), seq, tok)]
    L = _lib.mixers()
    call = lambda n: L.gbxm_step_advance(dev[0].data_ptr(), ids.element_size(), n, dev[1].data_ptr(), dev[2].data_ptr(), dev[3].data_ptr(), b, ops._stream_ptr(dev[0].device))
    assert call(0) == _lib.GBX_ERR_INVALID and call(-1) == _lib.GBX_ERR_INVALID
    assert call(rows) == _lib.GBX_OK
    assert torch.equal(dev[1].cpu(), torch.where((ids >= 0) & (ids < rows), ids, 0).long())
    seq[1::4] += 1
    tok[1::2] += 1
    assert torch.equal(dev[2].cpu(), seq) and torch.equal(dev[3].cpu(), tok)


@pytest.mark.parametrize("stop", [-1, "rows", 2 ** 40])
def test_stop_tokens_that_are_no_tokens(stop):
    """A sampler's end mark that the embedding has no row for ends its sequence, and the others get what they get from a loop that waits for the host."""
    model, vocab = _model("tugolix")
    assert model.token_rows == vocab
    stop = vocab if stop == "rows" else stop
    steps = 12
    gen = torch.Generator().manual_seed(6)
    forced = torch.randint(0, vocab, (steps, 2), generator=gen)
    forced[9, 1] = stop
    runs = []
    for ahead in (True, False):
        engine = BatchScheduler(model)
        took, inner = [], engine._step_ahead

        def counted(ids, toks):
            got = inner(ids, toks) if ahead else None
            took.append(got is not None)
            return got

        engine._step_ahead = counted
        rows, n = [], [0]

        def sampler(lp):
            rows.append(lp)
            n[0] += 1
            return forced[n[0] - 1, :lp.shape[0]].to("cuda:0")

        out = engine.generate([[5, 6], [7]], max_tokens=steps, sampler=sampler, stop_tokens=[stop])
        assert out == [forced[:, 0].tolist(), forced[:10, 1].tolist()]
        assert took[9] == ahead and not engine.slot_of
        runs.append(rows)
    for i, (x, y) in enumerate(zip(*runs)):
        assert x.shape == y.shape and (torch.equal(x, y) if i <= 9 else (x - y).abs().max() <= 0.05 * y.std())      # (the bounds of the comparison above)


def test_a_token_that_is_none_and_does_not_stop_raises():
    model, vocab = _model("tugolix")
    engine, n = BatchScheduler(model), [0]

    def sampler(lp):
        n[0] += 1
        return torch.tensor([vocab if n[0] == 8 else 3], device="cuda:0")

    with pytest.raises(ValueError, match="neither a stop token"):
        engine.generate([[1, 2, 3]], max_tokens=20, sampler=sampler)
    assert n[0] == 8


@pytest.mark.parametrize("at_capture", [False, True])
def test_a_captured_step_is_finished_as_it_was_captured(at_capture):
    """``logits`` set on a model whose step is captured already, or taken off again: what the replay's rows still lack does not change."""
    cfg = S.tugolix_config(width=256, delta=dict(heads=4, kv_heads=2, dim=64, vdim=64, conv=4), gla=dict(heads=2, dim=64, vdim=128, tau=16.0),
                           latent=dict(heads=4, dim=64, vdim=64, kv_rank=128), ff=512, moe=dict(experts=8, top=2, ff=128, groups=(4, 2)), pattern="dgls")
    cfg["logit_scale"] = 0.5
    model = S.build_tugolix(cfg, device="cuda:0", seed=3)
    assert model.logit_scale == 0.5
    plain = model.logits

    def toggle(on):
        if on:
            model.logits = lambda x: plain(x)
        else:
            model.__dict__.pop("logits", None)

    toggle(at_capture)
    engine, twin = BatchScheduler(model), BatchScheduler(model)
    twin.use_graphs = False
    for i in range(8):
        if i == 5:                                                # (a graph replays from the third single-token step on)
            assert engine._graphs and all(g.graph is not None for g in engine._graphs.values())
            toggle(not at_capture)
        entries = [("a", [3 + i]), ("b", [40 - i])]
        got, want = engine.step(entries), twin.step(entries)
        assert torch.equal(got, want)


def test_a_step_replaced_on_the_way():
    """A step that a sampler puts in place of the scheduler's takes over at once, and each token is consumed once."""
    model, vocab = _model("tugolix")
    forced = torch.randint(0, vocab, (12,), generator=torch.Generator().manual_seed(8)).tolist()
    seen = {}
    for replace in (False, True):
        engine, n = BatchScheduler(model), [0]
        rows, fed = seen.setdefault(replace, []), []

        def sampler(lp):
            rows.append(lp)
            n[0] += 1
            if replace and n[0] == 8:
                inner = engine.step
                engine.step = lambda entries: (fed.extend(t for _, ts in entries for t in ts), inner(entries))[1]
            return torch.tensor([forced[n[0] - 1]], device="cuda:0")

        assert engine.generate([[5, 6, 7]], max_tokens=12, sampler=sampler) == [forced]
        assert fed == ([] if not replace else forced[7:11])
    for x, y in zip(*seen.values()):
        assert torch.equal(x, y)


def _ring(engine):
    leaves = [leaf for c in engine.caches for leaf in (c._leaves() if hasattr(c, "_leaves") else [c])]
    rings = {leaf.ring for leaf in leaves if getattr(leaf, "window", 0) is None}
    assert len(rings) == 1
    return rings.pop()


@pytest.mark.parametrize("name", ["tugolix", "gibalorn"])
def test_tables_do_not_grow_for_a_token_that_ends_the_last_sequence(name):
    """A table of 256 rows holds a sequence whose last fed token takes row 255; the end mark behind it needs none."""
    model, vocab = _model(name)
    stop, engine, n = vocab - 1, BatchScheduler(model), [0]

    def sampler(lp):
        n[0] += 1
        return torch.tensor([stop if n[0] == 7 else n[0]], device="cuda:0")

    assert engine.generate([list(range(1, 251))], max_tokens=20, sampler=sampler, stop_tokens=[stop]) == [[1, 2, 3, 4, 5, 6, stop]]
    assert _ring(engine) == 256


@pytest.mark.parametrize("name", ["tugolix", "gibalorn"])
def test_sequences_outgrow_their_tables_while_steps_go_ahead(name):
    """The step that needs the 257th row waits for the host, which moves the tables; the steps behind it go ahead again."""
    model, vocab = _model(name)
    steps = 24
    gen = torch.Generator().manual_seed(11)
    prompts = [torch.randint(0, vocab, (n,), generator=gen).tolist() for n in (247, 31)]
    forced = torch.randint(0, vocab, (steps, 2), generator=gen)
    runs = []
    for ahead in (True, False):
        engine = BatchScheduler(model)
        took, inner = [], engine._step_ahead

        def counted(ids, toks):
            got = inner(ids, toks) if ahead else None
            took.append(got is not None)
            return got

        engine._step_ahead = counted
        rows, n = [], [0]

        def sampler(lp):
            rows.append(lp)
            n[0] += 1
            return forced[n[0] - 1].to("cuda:0")

        assert engine.generate(prompts, max_tokens=steps, sampler=sampler) == forced.t().tolist()
        assert _ring(engine) == 512
        # token i is fed at place 247 + i; a set of slots is captured at its third single-token step, before and after the tables have moved
        assert [i for i, t in enumerate(took) if t] == ([3, 4, 5, 6, 7, 8] + list(range(12, steps - 1)) if ahead else [])
        runs.append(rows)
    for x, y in zip(*runs):
        assert torch.equal(x, y)


@pytest.mark.parametrize("scale", [0.5, 3.0])
def test_log_probabilities_of_a_scaled_head(scale):
    """Those that a sampler gets while steps go ahead against the logarithm of the softmax, in 64 bits, of what ``step`` returns for the same tokens one by one."""
    cfg = S.tugolix_config(width=256, delta=dict(heads=4, kv_heads=2, dim=64, vdim=64, conv=4), gla=dict(heads=2, dim=64, vdim=128, tau=16.0),
                           latent=dict(heads=4, dim=64, vdim=64, kv_rank=128), ff=512, moe=dict(experts=8, top=2, ff=128, groups=(4, 2)), pattern="dgls")
    cfg["logit_scale"] = scale
    model = S.build_tugolix(cfg, device="cuda:0", seed=3)
    steps = 12
    forced = torch.randint(0, cfg["vocab"], (steps, 2), generator=torch.Generator().manual_seed(4))
    engine, rows, took = BatchScheduler(model), [], []
    inner = engine._step_ahead

    def counted(ids, toks):
        got = inner(ids, toks)
        took.append(got is not None)
        return got

    engine._step_ahead = counted

    def sampler(lp):
        rows.append(lp)
        return forced[len(rows) - 1].to("cuda:0")

    engine.generate([[5, 6], [7]], max_tokens=steps, sampler=sampler)
    assert sum(took) >= steps - 5
    twin = BatchScheduler(model)
    for i, got in enumerate(rows):
        logits = twin.step([("a", [5, 6]), ("b", [7])] if i == 0 else [("a", [int(forced[i - 1, 0])]), ("b", [int(forced[i - 1, 1])])])
        want = torch.log_softmax(logits.double(), -1)
        # fp32 sums and logarithms as in test_rows_of_the_head
        assert ((got.double() - want).abs() <= 2.0 ** -17 * want.abs().clamp(min=1.0) + 2.0 ** -15).all()
