"""What the entry points accept and refuse, and how they write their results, is the same whether the native call path
takes a call or leaves it to the Python path."""

import pytest
import torch

from _util import inputs_mod

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _layer(M, E=16, k=4, H=512, I=256):
    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("c", E=E, k=k, H=H, I=I), M, seed=M).to(DEV)
    return d, d.fused_experts_args(), d.fused_experts_kwargs()


@pytest.mark.parametrize("M", [1, 37])
@pytest.mark.parametrize("inplace", [True, 1, "yes", False, 0, None])
def test_inplace_goes_by_truth(pra, M, inplace):
    d, args, kw = _layer(M)
    want = pra.fused_experts(*args, **kw)
    logits = torch.randn(M, 16, device=DEV)
    routed = pra.fused_moe(d.hidden_states, d.w1, d.w2, logits, 4, True, **kw)
    for call, result in ((lambda x: pra.fused_experts(x, *args[1:], inplace=inplace, **kw), want),
                         (lambda x: pra.fused_moe(x, d.w1, d.w2, logits, 4, True, inplace=inplace, **kw), routed)):
        x = d.hidden_states.clone()
        got = call(x)
        assert torch.equal(got, result)
        assert (got.data_ptr() == x.data_ptr()) == bool(inplace)
        assert torch.equal(x, result if inplace else d.hidden_states)
