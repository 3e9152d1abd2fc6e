"""Packed products of 33 to 4096 rows as groups of up to 32 (gbx_qlinear_groups): rows and outputs that end inside a group or a tile, every width, group and type, a bias, infinities in
one group's rows; against float64.  And the calls: what takes that way, what keeps the one it had."""
import numpy as np
import pytest
import torch

from gbx_lm_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(n, k, bits, group, dt, seed, bias=False):
    gen = torch.Generator().manual_seed(seed)
    top = float((1 << bits) - 1)
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 32 * bits), generator=gen, dtype=torch.int64).to(torch.int32)
    s = (torch.rand((n, k // group), generator=gen) + 0.5) * (0.04 / top)
    z = -s * top / 2 + torch.randn((n, k // group), generator=gen) * 0.1 * s
    return w.to(DEV), s.to(dt).to(DEV), z.to(dt).to(DEV), torch.randn((n,), generator=gen).to(dt).to(DEV) if bias else None


def _dense(w, s, z, bits, group):
    u = np.pad(w.cpu().numpy().view(np.uint32).astype(np.uint64), ((0, 0), (0, 1)))
    at = np.arange(w.shape[1] * 32 // bits) * bits
    q = ((u[:, at // 32] | (u[:, at // 32 + 1] << np.uint64(32))) >> (at % 32).astype(np.uint64)) & np.uint64((1 << bits) - 1)
    sw, zw = (t.double().repeat_interleave(group, 1) for t in (s, z))
    return torch.from_numpy(q.astype(np.float64)).to(DEV) * sw + zw


def _groups(x, w, s, z, bias, bits, group, always=1):
    y = torch.full((x.shape[0], w.shape[0]), float("nan"), dtype=x.dtype, device=DEV)
    rc = _lib.lib().gbx_qlinear_groups(x.data_ptr(), w.data_ptr(), s.data_ptr(), z.data_ptr(), None if bias is None else bias.data_ptr(), y.data_ptr(), x.shape[0], w.shape[0],
                                       x.shape[1], bits, group, ops._DT[x.dtype], always, ops._stream_ptr(x.device))
    return y if rc == 0 else rc


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,group", [(b, g) for b in (2, 3, 4) for g in (32, 64, 128)])
@pytest.mark.parametrize("rows,n,k", [(33, 16, 1024), (64, 17, 4096), (65, 700, 1152), (97, 1, 2048), (511, 4111, 1280), (1023, 31, 3072), (200, 9000, 1024), (4096, 40, 128), (70, 300, 640)])
def test_against_float64(dt, bits, group, rows, n, k):
    w, s, z, bias = _layer(n, k, bits, group, dt, rows + n, bias=n == 700)
    x = torch.randn((rows, k), generator=torch.Generator().manual_seed(k)).to(dt).to(DEV)
    y = _groups(x, w, s, z, bias, bits, group)
    exact = x.double() @ _dense(w, s, z, bits, group).t()
    # one rounding to 16 bits (two with a bias) of fp32 sums, in which the fields stand as numbers of up to 2^10 + q
    half = 2.0 ** (-9 if dt == torch.bfloat16 else -12)
    size = x.double().abs() @ (s.double().repeat_interleave(group, 1) * 1040 + z.double().abs().repeat_interleave(group, 1)).t()
    bound = 2 * half * exact.abs() + 2.0 ** -21 * size
    if bias is not None:
        exact = exact + bias.double()
        bound = bound + 2 * half * exact.abs()
    assert ((y.double() - exact).abs() <= bound).all()
    for m in (32, rows // 2):                                             # a row's result does not depend on the rows beside it
        if 32 < m:
            assert torch.equal(_groups(x[:m].contiguous(), w, s, z, bias, bits, group), y[:m])


def test_infinities_stay_in_their_rows():
    w, s, z, _ = _layer(300, 1024, 4, 64, torch.bfloat16, 1)
    x = torch.randn((70, 1024), generator=torch.Generator().manual_seed(2)).bfloat16().to(DEV)
    plain = _groups(x, w, s, z, None, 4, 64)
    x[50, 3], x[69, 1000] = float("inf"), float("nan")
    y = _groups(x, w, s, z, None, 4, 64)
    rest = [r for r in range(70) if r not in (50, 69)]
    assert torch.equal(y[rest], plain[rest]) and y[69].isnan().all()
    inf = _dense(w, s, z, 4, 64)[:, 3]
    assert torch.equal(y[50][inf > 0], torch.full_like(y[50][inf > 0], float("inf"))) and torch.equal(y[50][inf < 0], torch.full_like(y[50][inf < 0], float("-inf")))


def test_what_it_does_not_take():
    for rows, n, k, bits, group in ((32, 64, 1024, 4, 64), (4097, 64, 1024, 4, 64), (64, 64, 1088, 4, 64), (64, 64, 4224, 4, 64)):
        w, s, z, _ = _layer(n, k, bits, group, torch.bfloat16, 3)
        assert _groups(torch.zeros((rows, k), device=DEV).bfloat16(), w, s, z, None, bits, group) == 1
    w, s, z, _ = _layer(11008, 4096, 3, 32, torch.bfloat16, 3)
    x = torch.zeros((200, 4096), device=DEV).bfloat16()
    assert _groups(x, w, s, z, None, 3, 32, always=0) == 1 and torch.is_tensor(_groups(x, w, s, z, None, 3, 32)) and torch.is_tensor(_groups(x[:64], w, s, z, None, 3, 32, always=0))


@pytest.mark.parametrize("rows", [33, 100, 255, 256, 600, 2000])
@pytest.mark.parametrize("native", [True, False])
def test_calls(monkeypatch, rows, native):
    """Rows of one sequence go that way, by the native call and by the general one; those of several keep theirs, and 256 to 1023 rows whose weight has a resident image."""
    k, n = 2048, 512
    w, s, z, bias = _layer(n, k, 4, 128, torch.bfloat16, rows, bias=True)
    if not native:
        monkeypatch.setattr(ops, "_few_rows", lambda *a: None)
    ops.dense_cache_clear()
    x = torch.randn((rows, k), generator=torch.Generator().manual_seed(rows)).bfloat16().to(DEV)
    want = _groups(x, w, s, z, bias, 4, 128, always=0)
    call = lambda t: ops.quantized_matmul(t, w, s, z, group_size=128, bits=4, bias=bias)
    assert torch.equal(call(x), want) and torch.equal(call(x[None]), want[None]) and torch.equal(call(x[:, None].transpose(0, 1)), want[None])
    assert ops._dense_cache.get((w, s, z), (n, k, 4, 128, x.dtype, x.device.index)) is None       # (no image was built for it)
    if rows % 2 == 0:
        other = call(x.view(2, rows // 2, k)).view(rows, n)
        assert ((other.double() - want.double()).abs() <= 2.0 ** -6 * want.double().abs() + 0.05).all()
        assert not torch.equal(other, want)
        ops.dense_cache_clear()
    if rows == 600:
        image = ops.dequantize(w, s, z, 128, 4)
        ops._dense_cache.put((w, s, z), (n, k, 4, 128, x.dtype, x.device.index), image)
        dense, exact = call(x), x.double() @ image.double().t()
        assert not torch.equal(dense, want)
        # two roundings to 8 bits, of the product and of its sum with the bias
        assert ((dense.double() - exact - bias.double()).abs() <= 2.0 ** -8 * (exact.abs() + (exact + bias.double()).abs()) + 1e-4).all()
        ops.dense_cache_clear()


@pytest.mark.parametrize("bits,group,k", [(2, 128, 4096), (3, 64, 1152), (4, 32, 640)])
@pytest.mark.parametrize("rows", [33, 64])
def test_layers_of_one_input(bits, group, k, rows):
    """Two or three layers in one launch: the bits of a call each; rows of several sequences keep the launch that they had."""
    from gbx_lm_amd.models.quantized_linear_gba import QuantizedLinear
    mods = []
    for i, n in enumerate((544, 32, 96)):
        w, s, z, bias = _layer(n, k, bits, group, torch.bfloat16, 7 * i + rows, bias=i == 1)
        q = QuantizedLinear(k, n, i == 1, group, bits)
        q._buffers.update(qweight=w, scales=s, zeros=z, **({"bias": bias} if i == 1 else {}))
        mods.append(q)
    x = torch.randn((rows, k), generator=torch.Generator().manual_seed(rows)).bfloat16().to(DEV)
    for some in (mods, mods[:2]):
        for y, q in zip(ops.quantized_matmul_multi(x, some), some):
            assert torch.equal(y, q(x)) and torch.equal(y, _groups(x, q.qweight, q.scales, q.zeros, q.bias, bits, group, always=0))
    one = ops.quantized_matmul_multi(x[None], mods)
    assert all(torch.equal(y[0], q(x)) for y, q in zip(one, mods))
    for y, v in zip(ops.quantized_matmul_multi(x[:, None], mods), one):
        assert ((y[:, 0].double() - v[0].double()).abs() <= 2.0 ** -6 * v[0].double().abs() + 0.05).all()


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("rows,n,k,bits,group", [(1024, 1024, 1024, 4, 128), (2000, 200, 3072, 3, 64), (4096, 64, 4096, 2, 32), (1025, 500, 128, 4, 32)])
def test_many_rows_go_one_way_whatever_is_resident(monkeypatch, native, rows, n, k, bits, group):
    """From 1024 rows on the bits of a layer do not depend on an image that an earlier call has left, its own or another's."""
    w, s, z, _ = _layer(n, k, bits, group, torch.bfloat16, rows)
    if not native:
        monkeypatch.setattr(ops, "_few_rows", lambda *a: None)
    x = torch.randn((rows, k), generator=torch.Generator().manual_seed(rows)).bfloat16().to(DEV)
    call = lambda: ops.quantized_matmul(x, w, s, z, group_size=group, bits=bits)
    ops.dense_cache_clear()
    want = _groups(x, w, s, z, None, bits, group, always=0)
    assert torch.equal(call(), want) and ops.dense_cache_bytes() == 0
    other = _layer(n, k, bits, group, torch.bfloat16, rows + 1)[:3]
    for t in (other, (w, s, z)):
        ops._dense_cache.put(t, (n, k, bits, group, x.dtype, x.device.index), ops.dequantize(*t, group, bits))
        assert torch.equal(call(), want)
    ops.dense_cache_clear()
