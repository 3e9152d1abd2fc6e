"""Quantised products of 2 to 32 rows: every width of field and group, one row tile and two, their edges, contractions that give waves one chunk each or
unequal numbers, outputs that end inside a workgroup, a bias, and scales that are not aligned to a chunk's (the dequantising kernel).  Contractions of 1024 to
4096 run in the kernel that keeps the rows in registers (csrc/mfma_slab_impl.h), or, for few rows off the grid of 1024, in csrc/mfma_rows.hip; longer ones there
(both output tilings: up to and beyond 4096 outputs) or, in groups of 128 on that grid, in csrc/mfma_batch.hip.  Reference: float64; tolerance: the result's rounding (two with a bias; the
dequantising kernel rounds every weight too) and fp32 sums of K terms as large as C + q = 143 (bf16) or 1039 (fp16)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def run(m, n, k, bits, g, dt, bias, shift, seed):
    from gbx_lm_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(seed)
    qw = torch.randint(-2**31, 2**31, (n, k // 32 * bits), device=DEV, generator=gen, dtype=torch.int64).to(torch.int32).view(torch.uint32)
    top = (1 << bits) - 1
    s = (torch.rand((n, k // g), device=DEV, generator=gen) + 0.5) * (0.1 / top)
    z = (-s * top / 2 + torch.randn(s.shape, device=DEV, generator=gen) * 0.2 * s).to(dt)
    s = s.to(dt)
    if shift:                                                   # an address one element past the allocation's
        s, z = (torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape) for t in (s, z))
    x = torch.randn((m, k), device=DEV, generator=gen).to(dt)
    b = torch.randn(n, device=DEV, generator=gen).to(dt) if bias else None
    w = ops.unpack(qw, bits).double() * s.double().repeat_interleave(g, 1) + z.double().repeat_interleave(g, 1)
    want = x.double() @ w.t() + (b.double() if bias else 0.0)
    y = ops.quantized_matmul(x, qw, s, z, group_size=g, bits=bits, bias=b)
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    terms = x.double().abs() @ (s.double().repeat_interleave(g, 1) * (144 if dt == torch.bfloat16 else 1040)).t()
    room = 2 * eps * (want.abs() + (b.double().abs() if bias else 0.0)) + 2.0 ** -22 * terms
    if shift:
        room = room + 4 * eps * (x.double() ** 2 @ (w ** 2).t()).sqrt()
    assert bool(((y.double() - want).abs() <= room).all())
    return x, qw, s, z, b, y


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,g", [(2, 32), (2, 64), (2, 128), (3, 32), (3, 64), (3, 128), (4, 32), (4, 64), (4, 128)])
@pytest.mark.parametrize("m,n,k,bias", [(2, 16, 1024, False), (16, 33, 1280, True), (17, 17, 1152, False), (27, 4097, 1408, True), (32, 4112, 2176, False), (31, 100, 3200, False)])
def test_fields_groups_and_edges(dt, bits, g, m, n, k, bias):
    run(m, n, k, bits, g, dt, bias, False, m + n + k + bits + g)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,g", [(2, 32), (2, 64), (2, 128), (3, 32), (3, 64), (3, 128), (4, 32), (4, 64), (4, 128)])
@pytest.mark.parametrize("m,n,k,bias", [(2, 4097, 4224, True), (16, 33, 11008, False), (17, 4096, 4224, False), (32, 4112, 11008, True), (9, 100, 4352, True), (3, 70, 1152, True)])
def test_rows_that_stay_in_memory(dt, bits, g, m, n, k, bias):
    """Contractions beyond 4096 that are no multiple of 1024, and few rows of a short one."""
    run(m, n, k, bits, g, dt, bias, False, m + n + k + bits + g)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,g", [(2, 32), (2, 64), (2, 128), (3, 128), (4, 128)])
@pytest.mark.parametrize("m,n,bias", [(32, 24584, False), (7, 12300, True), (16, 5130, False), (2, 1000, True), (33, 24576, False)])
def test_unsplit_workgroups_of_the_batch_kernel(dt, bits, g, m, n, bias):
    """Its 128, 64, 32 and 16 output rows a workgroup (64 for 128 in groups of 32 and 64), outputs that end inside one, and 33 rows in two launches."""
    run(m, n, 5120, bits, g, dt, bias, False, m + n + bits + g)


@pytest.mark.parametrize("bits,g", [(3, 32), (3, 64), (4, 32), (4, 64)])
def test_whole_kilochannels_and_unaligned_scales(bits, g):
    for m in (2, 15, 32):
        run(m, 5000, 1024, bits, g, torch.bfloat16, m == 15, False, m)
        run(m, 72, 3072, bits, g, torch.float16, m == 15, False, m)
        run(m, 72, 1024, bits, g, torch.bfloat16, False, True, m)


def test_a_row_does_not_depend_on_the_others():
    from gbx_lm_amd import ops
    x, qw, s, z, b, y = run(32, 4100, 1152, 3, 64, torch.bfloat16, False, False, 5)
    for rows in (slice(0, 2), slice(3, 19), slice(1, 18)):
        assert torch.equal(ops.quantized_matmul(x[rows].contiguous(), qw, s, z, group_size=64, bits=3), y[rows])


def extremes(dt, m, k, seed):
    """Rows with infinities (of one sign, in one group, of both signs), one that is not a number, and one so large that its products with C + q leave
    fp32 where those with the weights do not (bf16), beside ordinary rows."""
    x = torch.randn((m, k), device=DEV, generator=torch.Generator(device=DEV).manual_seed(seed)).to(dt)
    x[0, 3], x[1, k - 1], x[2, 5], x[2, 6], x[3, 70], x[4, 9], x[4, k - 7] = [float("inf"), float("-inf"), float("inf"), float("inf"), float("nan"),
                                                                              float("inf"), float("-inf")]
    x[5, 100] = 3e36 if dt == torch.bfloat16 else 60000.0
    return x


def same_numbers(y, want, eps, room):
    """Infinities and NaN where the reference has them, the rest within the tolerance."""
    y, most = y.double(), 3.3e38 if eps > 2.0 ** -10 else 65504.0
    want = torch.where(want.abs() > most, want.sign() * float("inf"), want)
    finite = torch.isfinite(want)
    assert torch.equal(torch.isnan(y), torch.isnan(want)) and torch.equal(y[~finite & ~torch.isnan(want)], want[~finite & ~torch.isnan(want)])
    assert bool(((y - want).abs() <= eps * want.abs() + room)[finite].all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,g", [(2, 32), (2, 64), (3, 32), (3, 64), (3, 128), (4, 32), (4, 64), (4, 128)])
@pytest.mark.parametrize("k", [1152, 2176, 4224])                   # in registers and, of up to 12 and 6 rows, not; beyond them
def test_infinite_undefined_and_huge_activations(dt, bits, g, k):
    """An infinity times the weight, not infinity minus infinity.  Tolerance: the roundings of the result and, where a row is huge, of its weights; fp32 sums
    of K terms as large as C + q."""
    from gbx_lm_amd import ops
    n = 100
    gen = torch.Generator(device=DEV).manual_seed(bits * g)
    qw = torch.randint(-2**31, 2**31, (n, k // 32 * bits), device=DEV, generator=gen, dtype=torch.int64).to(torch.int32).view(torch.uint32)
    s = ((torch.rand((n, k // g), device=DEV, generator=gen) + 0.5) * 0.03).to(dt)
    z = (-s.float() * ((1 << bits) - 1) / 2 * 0.9).to(dt)
    w = ops.unpack(qw, bits).double() * s.double().repeat_interleave(g, 1) + z.double().repeat_interleave(g, 1)
    for m in (6, 8, 20):
        x = extremes(dt, m, k, m)
        y = ops.quantized_matmul(x, qw, s, z, group_size=g, bits=bits)
        eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
        room = 2.0 ** -22 * (x.double().nan_to_num(0, 0, 0).abs() @ (s.double().repeat_interleave(g, 1) * (144 if dt == torch.bfloat16 else 1040)).t())
        room[5] *= dt != torch.bfloat16                             # (there: every weight rounded, the terms as they are)
        same_numbers(y, torch.stack([row @ w.t() if torch.isfinite(row).all() else ieee(row, w) for row in x.double()]), 3 * eps, room + 2.0 ** -10)


def ieee(row, w):
    """sum_k row[k] w[n, k] with infinities and NaN as they are (a matrix product may order its sums, which decides nothing here)."""
    odd = ~torch.isfinite(row)
    return (row[odd][None] * w[:, odd]).sum(1)
