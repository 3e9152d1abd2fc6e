"""q, k and v of a prompt in one dense launch (gbx_dense_forward_multi, ops.quantized_matmul_prompt): matrices that end inside a tile or hold less than one, rows that do,
biases on some; against float64 from the same 16-bit weights, and the module path against each module alone."""
import ctypes

import pytest
import torch

from gbx_lm_amd import _lib, ops
from gbx_lm_amd.models.quantized_linear_gba import QuantizedLinear
from gbx_lm_amd.utils import load_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,outs,k", [(1, (256,), 64), (257, (264, 8, 1), 128), (192, (192, 193), 320), (700, (768, 256, 256), 512), (513, (7, 1000, 513), 64)])
def test_launch_against_float64(dtype, rows, outs, k):
    gen = torch.Generator(device="cuda").manual_seed(rows + k)
    x = torch.randn((rows, k), generator=gen, device="cuda").to(dtype)
    ws = [(torch.randn((n, k), generator=gen, device="cuda") / k ** 0.5).to(dtype) for n in outs]
    bias = [None if i == 1 else torch.randn((n,), generator=gen, device="cuda").to(dtype) for i, n in enumerate(outs)]
    ys = [torch.full((rows, n), float("nan"), device="cuda", dtype=dtype) for n in outs]
    c = len(outs)
    VP, I32 = ctypes.c_void_p * c, ctypes.c_int32 * c
    _lib.check(_lib.lib().gbx_dense_forward_multi(x.data_ptr(), c, VP(*[w.data_ptr() for w in ws]), VP(*[None if b is None else b.data_ptr() for b in bias]),
                                                  VP(*[y.data_ptr() for y in ys]), I32(*outs), rows, k, ops._DT[dtype], ops._stream_ptr(x.device)))
    half = 2.0 ** (-9 if dtype == torch.bfloat16 else -12)                # half a unit in the last place, relative to a value's leading power of two
    for y, w, b in zip(ys, ws, bias):
        exact = x.double() @ w.double().t()
        bound = 2 * half * exact.abs() + 1e-5                             # one rounding, at most 2^-p of the value; sums in fp32 far below it
        if b is not None:
            exact = exact + b.double()
            bound = bound + 2 * half * exact.abs()                        # the sum with the bias is rounded again
        assert ((y.double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("rows", [255, 256, 1025, 3100])
def test_modules_share_a_launch(rows):
    """The same values as each module alone, up to the order of a split contraction's sums and, where it alone needs no image, the image's rounding; fewer rows, and images that are not there, take the modules' own path."""
    k, outs = 1024, (1024, 256, 256)
    mods = []
    for i, n in enumerate(outs):
        gen = torch.Generator().manual_seed(i)
        m = QuantizedLinear(k, n, i == 0, 64, 4)
        t = {"qweight": torch.randint(-2 ** 31, 2 ** 31 - 1, (n, k // 8), generator=gen, dtype=torch.int64).to(torch.int32),
             "scales": (torch.rand((n, k // 64), generator=gen) * 0.01).bfloat16(), "zeros": (torch.randn((n, k // 64), generator=gen) * 0.01).bfloat16()}
        if i == 0:
            t["bias"] = torch.randn((n,), generator=gen).bfloat16()
        load_weights(m, t, device="cuda:0")
        mods.append(m)
    x = torch.randn((1, rows, k), generator=torch.Generator().manual_seed(9)).bfloat16().cuda()
    ops.dense_cache_clear()
    if rows < 1024:
        assert ops.quantized_matmul_prompt(x, mods) is None               # nothing is resident, and nothing is built for few rows
        for m in mods:
            assert ops._dense_image(m, 8192, x.dtype, x.device) is not None
    got = ops.quantized_matmul_prompt(x, mods)
    assert (got is None) == (rows < 256 or any(ops._dense_image(m, rows, x.dtype, x.device) is None for m in mods))
    if got is not None:
        for y, m in zip(got, mods):
            alone = m(x)
            assert y.shape == alone.shape
            bound = 2.0 ** -7 * alone.double().abs() + 2.0 ** -7                                  # a unit in the last place of values near 1
            if rows >= 1024 and _lib.lib().gbx_qlinear_groups_win(rows, m.output_dims, k, m.bits, m.group_size):
                # alone it goes as groups of 32 rows, which round no weight; the image's are off by up to half a unit in the last place each, 2^-9 of the value
                bound = bound + 2.0 ** -9 * (x.double().abs() @ ops._dense_image(m, rows, x.dtype, x.device).double().abs().t())
            assert ((y.double() - alone.double()).abs() <= bound).all()
        handle = mods[1].register_forward_hook(lambda *a: None)
        assert ops.quantized_matmul_prompt(x, mods) is None               # what watches a module sees its call
        handle.remove()
    ops.dense_cache_clear()


def test_a_batch_keeps_its_sums(monkeypatch):
    """Several sequences' rows take each product alone, one sequence's together."""
    from gbx_lm_amd import synthetic as S
    from gbx_lm_amd.models.cache import make_prompt_cache
    model = S.build_model(S.TINY, S.make_strategy("S40", 2), device="cuda:0", seed=0)
    calls = []
    monkeypatch.setattr(ops, "quantized_matmul_prompt", lambda x, mods: calls.append(x.shape[0]))
    with torch.no_grad():
        for rows, length in ((4, 300), (1, 300)):
            model(torch.ones((rows, length), dtype=torch.long, device="cuda:0"), cache=make_prompt_cache(model))
    assert calls and set(calls) == {1}
