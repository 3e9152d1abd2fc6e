"""A step over several streams in its two forms, up to 256 rows and more: the same bits, whatever the other rows."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("s,top,width", [(1, 1, 64), (4, 1, 1024), (4, 3, 252), (4, 8, 256), (4, 9, 2048), (3, 17, 512), (2, 2, 4096)])
@pytest.mark.parametrize("read,norm", [(True, True), (False, True), (True, False)])
def test_rows_do_not_depend_on_the_form(dt, s, top, width, read, norm):
    from gbx_lm_amd import mixer_ops as M
    g = torch.Generator(device=DEV).manual_seed(s + top + width)

    def rnd(*shape):
        return torch.randn(shape, device=DEV, generator=g)

    t = 257
    streams, y = rnd(t, s, width), rnd(t, *([top] if top > 1 else []), width).to(dt)
    y_mix = rnd(t, top) if top > 1 else None
    mix, write, rd = rnd(s, s), rnd(s), rnd(s) if read else None
    nm = types.SimpleNamespace(weight=rnd(width), bias=rnd(width), eps=1e-5) if norm else None

    def step(r0, r1):
        x = streams[r0:r1].clone()
        return M.hyper_step_(x, y[r0:r1], None if y_mix is None else y_mix[r0:r1], mix, write, rd, nm, dt), x

    many, x_many = step(0, t)
    few, x_few = step(0, 256)
    one, x_one = step(t - 1, t)
    assert torch.equal(many[:256], few) and torch.equal(many[256:], one)
    assert torch.equal(x_many[:256], x_few) and torch.equal(x_many[256:], x_one)
    z = y.double().view(t, -1, width)
    z = z[:, 0] if y_mix is None else (y_mix.double()[:, :, None] * z).sum(1)
    want = torch.einsum("tic,ij->tjc", streams.double(), mix.double()) + write.double()[None, :, None] * z[:, None]
    # s + top + 1 products and additions of numbers of order 1 in fp32
    scale = torch.einsum("tic,ij->tjc", streams.double().abs(), mix.double().abs()) + write.double().abs()[None, :, None] * (
        z.abs() if y_mix is None else (y_mix.double().abs()[:, :, None] * y.double().abs()).sum(1))[:, None]
    assert ((x_many.double() - want).abs() <= (s + top + 3) * 2.0 ** -24 * scale).all()
