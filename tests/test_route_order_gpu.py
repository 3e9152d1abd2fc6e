"""The choice of a softmax / top-k router in one launch (gbx_moe_route): ties, every width of a wave's share, signs and extremes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _oracle(logits, k, mode, renorm):
    """fp32 by the definition: the k largest in the activation dtype, ties to the lowest index."""
    v = torch.softmax(logits.float(), -1).to(logits.dtype).float() if mode == 0 else logits.float()
    idx = torch.argsort(v, dim=-1, descending=True, stable=True)[:, :k]
    top = v.gather(1, idx)
    if mode == 0:
        w = top / top.sum(-1, keepdim=True).to(logits.dtype).float() if renorm else top
    else:
        w = torch.softmax(top, -1)
    return idx, w.to(logits.dtype)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("t,e,k,mode,renorm", [(1, 1, 1, 0, 1), (3, 63, 8, 1, 1), (2, 64, 1, 1, 1), (4, 65, 7, 1, 1), (5, 128, 8, 1, 1), (2, 129, 3, 1, 1), (3, 256, 8, 1, 1),
                                               (2, 1024, 8, 1, 1), (33, 8, 8, 1, 1), (6, 128, 8, 0, 1), (6, 60, 4, 0, 0)])
def test_choice(dt, t, e, k, mode, renorm):
    from gbx_lm_amd import ops
    g = torch.Generator().manual_seed(e + k)
    logits = (torch.randint(-6, 7, (t, e), generator=g).float() / 2).to(dt)           # few values: ties everywhere
    logits[0, ::3] = -0.0
    logits[-1, : max(e // 2, 1)] = torch.finfo(dt).min                                # the lowest value is still a value
    if mode == 0:
        logits = (torch.arange(t * e).reshape(t, e) * 7919 % 251).float().div(32).to(dt)   # (softmax rounds near a tie differently: values 1/32 apart or equal)
    inds, scores = ops.moe_route(logits.to(DEV), k, mode, bool(renorm))
    want_i, want_w = _oracle(logits, k, mode, renorm)
    assert torch.equal(inds.cpu().long(), want_i)
    eps = torch.finfo(dt).eps                                                        # one rounding of the weight, one of a neighbour's share of the sum
    assert ((scores.cpu().float() - want_w.float()).abs() <= 2 * eps * want_w.float() + 1e-7).all()
