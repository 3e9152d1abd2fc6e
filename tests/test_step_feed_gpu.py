"""The hand-over of a decode step in one launch each (gbx_step_feed, gbx_step_words) against the copies and fills it stands for, and what goes to those as before."""
import pytest
import torch

from gbx_lm_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("shape", [(1,), (3, 1), (64,), (65,), (1000, 1)])
@pytest.mark.parametrize("token", ["long", "int", "host", "strided", "column"])
def test_feed(shape, token):
    n = shape[0]
    ids = torch.randint(-5, 1 << 40 if token != "int" else 1 << 30, (n,))
    given = {"long": lambda: ids.to(DEV), "int": lambda: ids.to(torch.int32).to(DEV), "host": lambda: ids, "column": lambda: ids.to(DEV)[:, None],
             "strided": lambda: ids.to(DEV).repeat_interleave(2)[::2]}[token]()
    tok, pos = torch.full(shape, -1, device=DEV), torch.full((1,), -1, device=DEV)
    ops.step_feed(given, tok, pos, (1 << 33) + 7)
    assert torch.equal(tok.cpu().reshape(-1), ids) and pos.item() == (1 << 33) + 7
    ops.step_feed(tok, tok, pos, 3)
    assert torch.equal(tok.cpu().reshape(-1), ids) and pos.item() == 3
    if len(shape) == 1:
        ops.step_feed(torch.tensor([9], device=DEV), tok, pos, 0)         # one id for all, as a copy spreads it
        assert (tok == 9).all()
    else:
        with pytest.raises(RuntimeError):
            ops.step_feed(torch.zeros((n + 1,), dtype=torch.long, device=DEV), tok, pos, 0)


@pytest.mark.parametrize("count", [0, 1, 2, 3, 4])
def test_words(count):
    words = [torch.full((2,), -7 + i, dtype=torch.int32, device=DEV)[1:] for i in range(count)]
    out = torch.full((4,), 99, device=DEV)
    taken = ops.step_words(torch.tensor([1 << 35, 5], device=DEV), words, out)
    assert taken == (count <= 3)
    if taken:
        assert out.tolist() == [1 << 35] + [-7 + i for i in range(count)] + [0] * (3 - count)
    assert not ops.step_words(torch.tensor([1], dtype=torch.int32, device=DEV), words[:1], out)
