"""GPU parity of the kernels for a handful of tokens: the streaming family's split-reduction kernel (one block and many,
row counts up to its limit, ragged channels and reductions, self-quantising or not, both sides of the hand-over to the
streaming kernel), the two-launch layer, the narrow tiles and the top-k combine at every k that has its own variant."""

import pytest
import torch

from _util import inputs_mod

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("E,k,H,I,M,B", [
    (1, 1, 64, 64, 1, 16), (8, 2, 192, 128, 2, 64), (16, 8, 2048, 768, 1, 64), (16, 8, 2048, 768, 5, 64),
    (4, 4, 4096, 1408, 3, 32), (3, 3, 7168, 2048, 2, 64), (2, 1, 8192, 64, 16, 128), (1, 1, 1088, 960, 16, 64),
    (9, 9, 4096, 1408, 1, 64), (40, 6, 512, 2112, 9, 16),
])
def test_few_tokens_equal_the_tiled_families_stages(pra, oracle, E, k, H, I, M, B):
    im = inputs_mod()
    inp = im.make_inputs(im.LayerShape("f", E=E, k=k, H=H, I=I), M, seed=E + M + H)
    st = oracle.fused_experts_staged(inp.hidden_states, inp.w1, inp.w2, inp.topk_weights, inp.topk_ids, inp.w1_scale,
                                     inp.w2_scale, B)
    d = inp.to(DEV)
    s, e, npp = pra.moe_align_block_size(d.topk_ids, B, E)
    act = pra.gemm_gate_up_silu(st["x_q"].to(DEV), st["a1_scale"].to(DEV), d.w1, d.w1_scale, s, e, npp, k, B, M * k, "stream")
    # the epilogue's exponential is the one thing the oracle does not share bit for bit
    diff = (act.float().cpu() - st["cache2"].float()).abs() > 0.02 * st["cache2"].float().abs() + 1e-6
    assert not bool(diff.any())
    down = pra.gemm_down(st["h_q"].to(DEV), st["a2_scale"].to(DEV), d.w2, d.w2_scale, d.topk_weights, s, e, npp, B, "stream")
    assert torch.equal(down.cpu(), st["cache3"].reshape(M * k, H))
    # the layer, which may quantise inside the down GEMM, against its own stages
    hq, a2 = pra.per_token_quant_int8(act)
    want = torch.empty(M, H, dtype=torch.bfloat16, device=DEV)
    pra.moe_sum(pra.gemm_down(hq, a2, d.w2, d.w2_scale, d.topk_weights, s, e, npp, B, "stream").view(M, k, H), want)
    got = pra.fused_experts(*d.fused_experts_args(), **d.fused_experts_kwargs(), block_size_m=B, gemm_variant="stream")
    assert torch.equal(got, want)


@pytest.mark.parametrize("E,k,H,I", [(8, 2, 4096, 1408), (16, 2, 2048, 1024), (8, 2, 2048, 5632)])
@pytest.mark.parametrize("M", [5, 9, 10, 11, 12, 16])
def test_either_side_of_the_line_between_the_streaming_kernels(pra, E, k, H, I, M):
    """Token rows in LDS: whether all workgroups of the split-reduction kernel are resident at once decides which
    kernel runs (9 and 10 rows of 4096, 11 and 12 of 2048)."""
    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("s", E=E, k=k, H=H, I=I), M, seed=E + M).to(DEV)
    kw = d.fused_experts_kwargs()
    got = pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="stream")
    assert torch.equal(got, pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="narrow"))


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 16])
@pytest.mark.parametrize("M,H", [(1, 8), (3, 2048), (33, 7168)])
def test_combine_at_every_k(pra, oracle, k, M, H):
    x = torch.randn(M, k, H, generator=torch.Generator().manual_seed(k)).to(torch.bfloat16)
    out = torch.empty(M, H, dtype=torch.bfloat16, device=DEV)
    pra.moe_sum(x.to(DEV), out)
    assert torch.equal(out.cpu(), oracle.moe_sum(x))


@pytest.mark.parametrize("E,k,H,I,M,B", [
    (3, 1, 512, 512, 17, 64), (40, 8, 640, 768, 20, 64), (5, 5, 1408, 896, 32, 128), (128, 2, 512, 1024, 33, 64),
    (300, 4, 2048, 512, 90, 128), (2, 2, 4096, 1408, 65, 64), (700, 6, 512, 640, 31, 64),
])
def test_narrow_tiles_at_short_reductions_and_many_tasks(pra, oracle, E, k, H, I, M, B):
    """The narrow family at its shortest reductions (where its loads run fewer steps ahead), with 32- and 64-row
    tiles, one task per workgroup and more than 64 candidates per workgroup."""
    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("n", E=E, k=k, H=H, I=I, routing="zipf"), M, seed=E + M).to(DEV)
    s, e, npp = pra.moe_align_block_size(d.topk_ids, B, E)
    xq, a1 = pra.per_token_quant_int8(d.hidden_states)
    for w, row_div, a in ((d.w1, k, xq), (d.w2, 1, torch.randint(-127, 128, (M * k, I), dtype=torch.int8, device=DEV))):
        got = pra.gemm_acc_i32(a, w, s, e, npp, row_div, B, M * k, "narrow")
        assert torch.equal(got, pra.gemm_acc_i32(a, w, s, e, npp, row_div, B, M * k, "stream"))
    kw = d.fused_experts_kwargs()
    out = pra.fused_experts(*d.fused_experts_args(), **kw, block_size_m=B, gemm_variant="narrow")
    assert torch.equal(out, pra.fused_experts(*d.fused_experts_args(), **kw, block_size_m=B, gemm_variant="stream"))


@pytest.mark.parametrize("E,k,H,I,M", [
    (16, 8, 2048, 768, 1), (4, 4, 64, 64, 1), (40, 20, 1088, 192, 1), (1, 1, 8192, 4096, 1), (9, 9, 4096, 1408, 1),
    (16, 8, 2048, 768, 8), (5, 2, 1024, 1024, 2), (6, 3, 1088, 1088, 3), (4, 4, 7168, 2112, 4), (12, 1, 3072, 3072, 4),
    (64, 8, 5120, 64, 7), (70, 64, 192, 320, 1), (8, 8, 6144, 128, 8), (10, 8, 6144, 128, 8),
])
def test_layer_of_a_few_tokens_equals_the_chain_of_stages(pra, E, k, H, I, M):
    """The two-launch layer against the chain through moe_align, tokens sharing experts or not."""
    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("t", E=E, k=k, H=H, I=I), M, seed=E + M + H).to(DEV)
    for ids in (d.topk_ids.clone(), d.topk_ids[:1].expand(M, k).contiguous()):
        d.topk_ids.copy_(ids)
        want = pra.fused_experts(*d.fused_experts_args(), **d.fused_experts_kwargs(), gemm_variant="stream")
        assert torch.equal(pra.fused_experts(*d.fused_experts_args(), **d.fused_experts_kwargs()), want)
    x = d.hidden_states.clone()
    got = pra.fused_experts(x, *d.fused_experts_args()[1:], **d.fused_experts_kwargs(), inplace=True)
    assert got.data_ptr() == x.data_ptr() and torch.equal(x, want)


@pytest.mark.parametrize("E,k,H,I,groups,score,bias,M", [
    (128, 8, 2048, 768, None, "softmax", False, 1), (256, 8, 7168, 256, (8, 4), "sigmoid", True, 1),
    (100, 3, 512, 64, None, "sigmoid", True, 1), (192, 16, 1088, 192, None, "softmax", False, 1),
    (40, 2, 256, 128, None, "softmax", False, 1), (300, 4, 256, 64, None, "softmax", False, 1), (128, 8, 512, 128, None, "softmax", False, 4),
])
def test_routed_call_of_a_few_tokens_equals_router_and_layer(pra, E, k, H, I, groups, score, bias, M):
    """Routing inside the layer's first launch (one token), in front of the two launches, or of the chain."""
    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("r", E=E, k=k, H=H, I=I), M, seed=E + k).to(DEV)
    g = torch.Generator(device=DEV).manual_seed(E)
    logits = torch.randn(M, E, device=DEV, generator=g)
    how = dict(scoring_func=score, routed_scaling_factor=2.5 if bias else 1.0,
               e_score_correction_bias=torch.randn(E, device=DEV, generator=g) * 0.1 if bias else None)
    if groups:
        how.update(use_grouped_topk=True, num_expert_group=groups[0], topk_group=groups[1])
    kw = {n: v for n, v in d.fused_experts_kwargs().items() if n not in ("topk_weights", "topk_ids")}
    record = torch.zeros(M, 3, k, dtype=torch.uint16, device=DEV)
    x, w1, w2 = d.fused_experts_args()[:3]
    got = pra.fused_moe(x, w1, w2, logits, k, True, routed_experts_out=(record, 1), **how, **kw)
    if groups:
        w, ids = pra.grouped_topk(x, logits, k, True, *groups, score, 2.5, how["e_score_correction_bias"])
    else:
        w, ids = pra.route_topk(logits, k, score_func=score, renormalize=True, route_scale=how["routed_scaling_factor"],
                                selection_bias=how["e_score_correction_bias"])
    assert torch.equal(record[:, 1].to(torch.int32), ids) and int(record[:, ::2].to(torch.int32).sum()) == 0
    assert torch.equal(got, pra.fused_experts(x, w1, w2, w, ids, **kw, gemm_variant="stream"))


@pytest.mark.parametrize("H", [4096, 4160, 7168, 8192, 8256])
@pytest.mark.parametrize("M", [9, 1101, 4101])  # alignment in one, two and three launches
def test_layer_quantises_long_rows_as_the_row_quantiser_does(pra, H, M):
    """Rows held by one wavefront, by four, and read twice, in each launch that quantises the layer's input."""
    E, k, I, B = 8, 8, 64, 64
    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("q", E=E, k=k, H=H, I=I), M, seed=H + M).to(DEV)
    s, e, npp = pra.moe_align_block_size(d.topk_ids, B, E)
    x_q, a1 = pra.per_token_quant_int8(d.hidden_states)
    act = pra.gemm_gate_up_silu(x_q, a1, d.w1, d.w1_scale, s, e, npp, k, B, M * k, "stream")
    h_q, a2 = pra.per_token_quant_int8(act)
    want = torch.empty(M, H, dtype=torch.bfloat16, device=DEV)
    pra.moe_sum(pra.gemm_down(h_q, a2, d.w2, d.w2_scale, d.topk_weights, s, e, npp, B, "stream").view(M, k, H), want)
    got = pra.fused_experts(*d.fused_experts_args(), **d.fused_experts_kwargs(), block_size_m=B, gemm_variant="stream")
    assert torch.equal(got, want)


@pytest.mark.parametrize("E,k,H,I,M,B", [
    (66, 8, 4160, 576, 9, 64),    # 17 windows, the last of 64 bytes; down whole
    (40, 4, 4096, 1088, 16, 16),  # starting windows; down whole, the longest of its kind
    (33, 2, 7168, 320, 40, 64),   # up to 40 rows of an expert: several passes; down whole
    (17, 4, 1600, 320, 40, 64),   # down of so few workgroups that its 2 windows are halved, several passes
    (32, 4, 2048, 576, 9, 32),    # the most workgroups of that kind: 3 windows, the last of 64 bytes
    (70, 4, 1088, 2064, 5, 32),   # a reduction too short to be halved: whole
    (70, 4, 1600, 2064, 5, 32),   # an odd number of tile pairs (gate_up alone takes it), 7 windows, the last of 64 bytes
    (40, 4, 1536, 1408, 9, 64),   # the shortest that gate_up halves: 6 windows
    (40, 4, 4096, 1152, 16, 16),  # the shortest that down halves: 5 windows, the last of 128 bytes
    (33, 2, 2048, 1216, 40, 64),  # down in several passes: 5 windows, the last of 192 bytes
    (17, 2, 1024, 4096, 9, 32),   # starting windows in down
])
def test_reductions_halved_between_wavefronts(pra, oracle, E, k, H, I, M, B):
    """The streaming kernel with a tile pair's reduction in two wavefronts: windows that do not halve evenly, a last
    window that is partial, a workgroup with one tile pair of two, starting windows, blocks of one and of several passes."""
    im = inputs_mod()
    inp = im.make_inputs(im.LayerShape("h", E=E, k=k, H=H, I=I), M, seed=E + M + H)
    inp.topk_ids[:, 0] = 0  # an expert that every token visits
    inp.topk_ids[:, 1:] = inp.topk_ids[:, 1:].clamp(min=1)
    st = oracle.fused_experts_staged(inp.hidden_states, inp.w1, inp.w2, inp.topk_weights, inp.topk_ids, inp.w1_scale,
                                     inp.w2_scale, B)
    d = inp.to(DEV)
    s, e, npp = pra.moe_align_block_size(d.topk_ids, B, E)
    act = pra.gemm_gate_up_silu(st["x_q"].to(DEV), st["a1_scale"].to(DEV), d.w1, d.w1_scale, s, e, npp, k, B, M * k, "stream")
    diff = (act.float().cpu() - st["cache2"].float()).abs() > 0.02 * st["cache2"].float().abs() + 1e-6  # (the exponential)
    assert not bool(diff.any())
    if I % 64:
        return
    down = pra.gemm_down(st["h_q"].to(DEV), st["a2_scale"].to(DEV), d.w2, d.w2_scale, d.topk_weights, s, e, npp, B, "stream")
    assert torch.equal(down.cpu(), st["cache3"].reshape(M * k, H))
