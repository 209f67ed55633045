"""The native call path of the entry points against the Python path of the same call: what it does not take
(other id types, a caller's stride, a first call without a workspace) must give the same result, and a default
workspace that is outgrown or only just large enough for the layer must not change one."""

import pytest
import torch

from _util import inputs_mod

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M", [1, 37])
def test_both_paths_agree(pra, M):
    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("h", E=16, k=4, H=512, I=256), M, seed=M).to(DEV)
    kw = d.fused_experts_kwargs()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        want = pra.fused_experts(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids.to(torch.int64), **kw)
        for _ in range(2):
            assert torch.equal(pra.fused_experts(*d.fused_experts_args(), **kw), want)
        # a workspace of exactly the layer's size, then a routed call that needs room for the routing behind it
        pra.api._workspaces.pop((0, stream.cuda_stream))
        pra._abi.host().forget(0, stream.cuda_stream)
        pra.api._workspace(d.w1.device, stream.cuda_stream, pra.workspace_bytes(M, 4, 16, 512, 256, 64))
        logits = torch.randn(M, 16, device=DEV)
        w, ids = pra.route_topk(logits, 4)
        routed = pra.fused_experts(d.hidden_states, d.w1, d.w2, w, ids, **kw)
        for _ in range(2):
            assert torch.equal(pra.fused_moe(d.hidden_states, d.w1, d.w2, logits, 4, True, **kw), routed)
        x = d.hidden_states
        y = pra.apply_int8_linear(x, d.w1[0], d.w1_scale[0])
        assert torch.equal(pra.apply_int8_linear(x, d.w1[0].t(), d.w1_scale[0]), y)
        big = pra.fused_experts(x.repeat(50, 1), d.w1, d.w2, d.topk_weights.repeat(50, 1), d.topk_ids.repeat(50, 1), **kw)
        assert torch.equal(big[:M], pra.fused_experts(*d.fused_experts_args(), **kw)) or torch.allclose(
            big[:M].float(), want.float(), rtol=1e-2, atol=1e-2 * float(want.float().abs().max()))
        assert torch.equal(pra.fused_experts(*d.fused_experts_args(), inplace=True, **kw), want)
    torch.cuda.synchronize()
