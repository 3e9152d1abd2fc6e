"""Routed experts over packed weights for many (row, choice) pairs (csrc/mixers_moe_packed.hip) at the edges of their tiles: experts with no
pair, one, and one less / as many / one more than 16, 32 and 64; output rows off the 64 / 128 / 256 grid; contractions of one, two, three
chunks; every width, group size and activation type.  Reference: float64 from the oracle's unpacking.  Tolerance: fields and activations
enter exactly, sums are fp32 (K 2^-24 of the terms' absolute sum with the offset C = 128 or 1024 in every field), the result is rounded once:
2^-8 (bf16) / 2^-11 (fp16) of its size."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
COUNTS = [1, 0, 15, 16, 17, 31, 32, 33, 63, 64, 65, 130]


def make(oracle, E, N, K, bits, g, dt, seed):
    rng = np.random.default_rng(seed)
    qw = rng.integers(0, 2**32, (E, N, K * bits // 32), dtype=np.uint32)
    qmax = float((1 << bits) - 1)
    s = torch.from_numpy(((rng.random((E, N, K // g)) + 0.5) * (0.04 / qmax)).astype(np.float32)).to(dt)
    z = (-s.float() * qmax / 2.0 + torch.from_numpy(rng.standard_normal(s.shape).astype(np.float32)) * 0.1 * s.float()).to(dt)
    q = torch.from_numpy(np.stack([oracle.unpack(qw[e], bits) for e in range(E)]).astype(np.float64))
    w = q * s.double().repeat_interleave(g, -1) + z.double().repeat_interleave(g, -1)
    mag = (q + (128 if dt == torch.bfloat16 else 1024)) * s.double().repeat_interleave(g, -1) + z.double().abs().repeat_interleave(g, -1)
    return torch.from_numpy(qw.view(np.int32)).view(torch.uint32).to(DEV), s.to(DEV), z.to(DEV), w.to(DEV), mag.to(DEV)


def indices(seed):
    idx = torch.cat([torch.full((n,), e) for e, n in enumerate(COUNTS)])
    return idx[torch.randperm(idx.numel(), generator=torch.Generator().manual_seed(seed))]


def rows(x, w, idx):
    y = torch.empty((x.shape[0], w.shape[1]), dtype=torch.float64, device=DEV)
    for e in idx.unique().tolist():
        at = idx == e
        y[at] = x[at] @ w[e].t()
    return y


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("g", [32, 64, 128])
@pytest.mark.parametrize("bits", [2, 3, 4])
def test_tiles_of_every_height(oracle, bits, g, dt):
    from gbx_lm_amd import ops
    E, eps = len(COUNTS), 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    for N, K in ((200, 128), (72, 384), (257, 256)):
        qw, s, z, w, mag = make(oracle, E, N, K, bits, g, dt, seed=bits + g + N)
        idx = indices(N).to(DEV)
        P = idx.numel()
        gen = torch.Generator(device=DEV).manual_seed(N)
        x = torch.randn((P, 1, 1, K), device=DEV, generator=gen).to(dt)
        bias = (torch.randn((E, N), device=DEV, generator=gen) * 0.1).to(dt)
        want, room = rows(x.view(P, K).double(), w, idx), K * 2.0 ** -24 * rows(x.view(P, K).double().abs(), mag, idx)
        got = ops.gather_quantized_matmul(x, qw, s, z, idx[:, None], group_size=g, bits=bits).view(P, N).double()
        assert bool(((got - want).abs() <= eps * want.abs() + room + 1e-7).all()), (N, K)
        got = ops.gather_quantized_matmul(x, qw, s, z, idx[:, None], group_size=g, bits=bits, bias=bias).view(P, N).double()
        want = want + bias.double()[idx]                            # (the product is rounded in front of the bias, the sum once more)
        assert bool(((got - want).abs() <= 2 * eps * (want.abs() + bias.double()[idx].abs()) + room + 1e-7).all()), (N, K)


@pytest.mark.parametrize("bits,g", [(2, 64), (3, 128), (3, 32), (4, 128)])
def test_gated_pairs_round_like_the_three_operations(oracle, bits, g):
    """silu(gate) * up of shared rows (several choices per row) equals the separate products and ``ops.swiglu`` bit for bit."""
    from gbx_lm_amd import ops
    from gbx_lm_amd.models.switch_layers import QuantizedSwitchLinear
    E, N, K, T, k = 7, 200, 256, 90, 3
    mods = []
    for seed in (1, 2):
        qw, s, z, _, _ = make(oracle, E, N, K, bits, g, torch.bfloat16, seed)
        m = QuantizedSwitchLinear(K, N, E, bias=False, group_size=g, bits=bits)
        m._buffers["qweight"], m._buffers["scales"], m._buffers["zeros"] = qw, s, z
        mods.append(m)
    x = torch.randn((T, 1, 1, K), device=DEV).to(torch.bfloat16)
    idx = torch.rand((T, E), device=DEV).topk(k, -1).indices.to(torch.int32)
    got = ops.gather_swiglu(x, mods[0], mods[1], idx)
    want = ops.swiglu(mods[0](x, idx), mods[1](x, idx))
    assert got.shape == want.shape == (T, k, 1, N)
    assert torch.equal(got, want)


def test_index_without_an_expert_gives_no_number(oracle):
    from gbx_lm_amd import ops
    E, N, K = 5, 72, 128
    qw, s, z, w, _ = make(oracle, E, N, K, 4, 64, torch.bfloat16, 9)
    idx = torch.arange(100, device=DEV) % E
    x = torch.randn((100, 1, 1, K), device=DEV).to(torch.bfloat16)
    good = ops.gather_quantized_matmul(x, qw, s, z, idx[:, None], group_size=64, bits=4).view(100, N)
    bad = idx.clone()
    bad[3], bad[70] = E, -1
    got = ops.gather_quantized_matmul(x, qw, s, z, bad[:, None], group_size=64, bits=4).view(100, N)
    keep = bad == idx
    assert torch.isnan(got[~keep].float()).all() and torch.equal(got[keep], good[keep])


def test_replays_in_a_graph(oracle):
    """A step whose pairs were grouped on the host could not be captured; the launches can."""
    from gbx_lm_amd import graphs, ops
    E, N, K = 6, 256, 256
    qw, s, z, _, _ = make(oracle, E, N, K, 4, 128, torch.bfloat16, 4)
    x = torch.randn((96, 1, 1, K), device=DEV).to(torch.bfloat16)
    idx = torch.zeros((96, 1), dtype=torch.int32, device=DEV)
    run = lambda: ops.gather_quantized_matmul(x, qw, s, z, idx, group_size=128, bits=4)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with graphs.capture(graph):
        y = run()
    for seed in range(4):
        gen = torch.Generator(device=DEV).manual_seed(seed)
        x.copy_(torch.randn(x.shape, device=DEV, generator=gen))
        idx.copy_(torch.randint(0, E, idx.shape, device=DEV, generator=gen))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, run())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,g", [(2, 64), (3, 32), (3, 128), (4, 32), (4, 128)])
def test_infinite_and_undefined_activations(oracle, bits, g, dt):
    """An infinity times the weight, not infinity minus infinity; rows beside it keep their bits.  Tiles of every height, and the gated form."""
    from gbx_lm_amd import ops
    from gbx_lm_amd.models.switch_layers import QuantizedSwitchLinear
    E, N, K = len(COUNTS), 200, 384
    qw, s, z, w, _ = make(oracle, E, N, K, bits, g, dt, seed=bits)
    idx = indices(3).to(DEV)
    P = idx.numel()
    x = torch.randn((P, 1, 1, K), device=DEV).to(dt)
    plain = ops.gather_quantized_matmul(x, qw, s, z, idx[:, None], group_size=g, bits=bits).view(P, N)
    odd = torch.arange(0, P, 3, device=DEV)
    x.view(P, K)[odd, odd % K] = torch.tensor([float("inf"), float("-inf")], device=DEV, dtype=dt)[odd % 2]
    x.view(P, K)[odd[::7], 17] = float("nan")
    got = ops.gather_quantized_matmul(x, qw, s, z, idx[:, None], group_size=g, bits=bits).view(P, N)
    sign = torch.where(odd % 2 == 0, 1.0, -1.0).double()[:, None] * w[idx[odd], :, odd % K].sign()
    want = sign * float("inf")
    want[::7] = float("nan")
    assert bool((torch.isnan(got[odd]) == torch.isnan(want)).all()) and torch.equal(got[odd].double().nan_to_num(0, 1, -1), want.nan_to_num(0, 1, -1))
    rest = torch.ones(P, dtype=torch.bool, device=DEV)
    rest[odd] = False
    assert torch.equal(got[rest], plain[rest])
    if dt == torch.bfloat16:
        up = make(oracle, E, N, K, bits, g, dt, seed=bits + 9)[:3]
        mods = []
        for t in ((qw, s, z), up):
            m = QuantizedSwitchLinear(K, N, E, bias=False, group_size=g, bits=bits)
            m._buffers["qweight"], m._buffers["scales"], m._buffers["zeros"] = t
            mods.append(m)
        a, b = ops.gather_swiglu(x, mods[0], mods[1], idx[:, None]), ops.swiglu(mods[0](x, idx[:, None]), mods[1](x, idx[:, None]))
        assert torch.equal(a.float().nan_to_num(7e9, 8e9, -8e9), b.float().nan_to_num(7e9, 8e9, -8e9))


def test_a_bias_in_another_order_is_read_in_its_own(oracle):
    from gbx_lm_amd import ops
    E, N, K = 5, 72, 128
    qw, s, z, _, _ = make(oracle, E, N, K, 4, 64, torch.bfloat16, 9)
    idx = (torch.arange(100, device=DEV) % E)[:, None]
    x, bias = torch.randn((100, 1, 1, K), device=DEV).to(torch.bfloat16), torch.randn((E, N), device=DEV).to(torch.bfloat16)
    run = lambda b: ops.gather_quantized_matmul(x, qw, s, z, idx, group_size=64, bits=4, bias=b)
    assert torch.equal(run(bias.t().contiguous().t()), run(bias))


def test_rows_in_32_bits_are_refused(oracle):
    """The launch reads 16-bit rows: anything else raises, as one matrix at a time does."""
    from gbx_lm_amd import ops
    from gbx_lm_amd.models.switch_layers import QuantizedSwitchLinear
    E, N, K = 6, 64, 256
    mods = []
    for seed in (1, 2):
        qw, s, z, _, _ = make(oracle, E, N, K, 4, 64, torch.float32, seed)
        m = QuantizedSwitchLinear(K, N, E, bias=False, group_size=64, bits=4)
        m._buffers["qweight"], m._buffers["scales"], m._buffers["zeros"] = qw, s, z
        mods.append(m)
    idx = (torch.arange(100, device=DEV) % E)[:, None].to(torch.int32)
    x = torch.randn((100, 1, 1, K), device=DEV)
    assert ops.gather_swiglu(x, mods[0], mods[1], idx) is None
    with pytest.raises(ValueError):
        mods[0](x, idx)


@pytest.mark.parametrize("bits,g", [(3, 32), (2, 64), (4, 128)])
def test_thousands_of_pairs_per_expert_go_one_expert_at_a_time(oracle, monkeypatch, bits, g):
    """Both sides of the rule, and a capture beyond it.  Tolerance: every weight rounded (2^-8 of it) on the way of the general path, fp32 sums, one rounding."""
    from gbx_lm_amd import graphs, ops
    E, N, K = 2, 136, 256
    qw, s, z, w, mag = make(oracle, E, N, K, bits, g, torch.bfloat16, 5)
    P = 3000
    x, idx = torch.randn((P, 1, 1, K), device=DEV).to(torch.bfloat16), torch.randint(0, E, (P, 1), device=DEV)
    want, calls, real = rows(x.view(P, K).double(), w, idx.view(-1)), [], ops.quantized_matmul
    room = 2.0 ** -7 * want.abs() + 4 * 2.0 ** -8 * rows(x.view(P, K).double() ** 2, w ** 2, idx.view(-1)).sqrt() + K * 2.0 ** -24 * rows(x.view(P, K).double().abs(), mag, idx.view(-1))
    monkeypatch.setattr(ops, "quantized_matmul", lambda *a, **k: calls.append(1) or real(*a, **k))
    run = lambda: ops.gather_quantized_matmul(x, qw, s, z, idx, group_size=g, bits=bits).view(P, N)
    for line, n in ((P * N * K // E + 1, 0), (P * N * K // E, E)):
        monkeypatch.setitem(ops._EXPERT_WORK, g, line)
        del calls[:]
        assert bool(((run().double() - want).abs() <= room).all()) and len(calls) == n
    del calls[:]
    graph = torch.cuda.CUDAGraph()
    with graphs.capture(graph):
        y = run()
    graph.replay()
    torch.cuda.synchronize()
    assert not calls and bool(((y.double() - want).abs() <= room).all())
