"""Rows that hold a NaN or an infinity: every quantiser skips a NaN in the row's maximum and makes it 0, so such a row
gives what it gives with 0 in the NaN's place, whatever the number of rows and the kernel that quantises them."""

import pytest
import torch

from _util import inputs_mod

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SAME = dict(rtol=0, atol=0, equal_nan=True)


def _spoil(x, value):
    """The largest element of row 0, and `value` beside it, at both ends of its eight elements and alone in others."""
    x = x.clone()
    x[0, 16], x[-1, -2] = 30.0, -30.0
    for row, col in ((0, 17), (0, 23), (0, 40), (-1, x.shape[1] - 1), (-1, 0)):
        x[row, col] = value
    return x


@pytest.mark.parametrize("M,N,K", [(1, 64, 128), (4, 512, 2048), (5, 512, 1088), (16, 1024, 1024), (40, 512, 2048)])
def test_linear_and_quantisers_skip_a_nan(pra, oracle, M, N, K):
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    s = torch.rand(N, generator=g) * 0.008 + 0.002
    nan, zero = _spoil(x, float("nan")), _spoil(x, 0.0)
    for sign in (1, -1):
        got = pra.apply_int8_linear((nan * sign).to(DEV), w.to(DEV), s.to(DEV))
        assert torch.equal(got.cpu(), oracle.w8a8_linear(zero * sign, w, s))
    q, a = pra.per_token_quant_int8(nan.to(DEV))
    qo, ao = oracle.per_token_quant_int8(zero)
    assert torch.equal(q.cpu(), qo) and torch.equal(a.cpu(), ao)
    # an infinity: no finite scale, so the row's products are 0 * inf; the other rows are not touched
    inf = _spoil(x, float("inf")).to(DEV)
    got = pra.apply_int8_linear(inf, w.to(DEV), s.to(DEV))
    torch.testing.assert_close(got, pra.apply_int8_linear(inf, w.to(DEV), s.to(DEV), gemm_variant="stream"), **SAME)
    assert bool(got[0].isnan().all()) and (M <= 2 or torch.equal(got[1:-1].cpu(), oracle.w8a8_linear(x, w, s)[1:-1]))


@pytest.mark.parametrize("E,k,H,I,M", [(16, 8, 2048, 768, 1), (8, 2, 512, 1088, 3), (6, 3, 4096, 1408, 4), (16, 4, 1024, 512, 8),
                                       (16, 4, 1024, 512, 60)])
def test_layer_and_mlp_skip_a_nan(pra, E, k, H, I, M):
    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("n", E=E, k=k, H=H, I=I), M, seed=E + M).to(DEV)
    args, kw = d.fused_experts_args(), d.fused_experts_kwargs()
    x = d.hidden_states
    nan, zero, inf = (_spoil(x.cpu(), v).to(DEV) for v in (float("nan"), 0.0, float("inf")))
    got = pra.fused_experts(nan, *args[1:], **kw)
    assert torch.equal(got, pra.fused_experts(zero, *args[1:], **kw, gemm_variant="stream"))
    torch.testing.assert_close(pra.fused_experts(inf, *args[1:], **kw),
                               pra.fused_experts(inf, *args[1:], **kw, gemm_variant="stream"), **SAME)
    mlp = (d.w1[0], d.w1_scale[0].reshape(-1), d.w2[0], d.w2_scale[0].reshape(-1))
    assert torch.equal(pra.w8a8_mlp(nan, *mlp), pra.w8a8_mlp(zero, *mlp, gemm_variant="stream"))
    # NaNs between the two projections: channels without a usable scale, next to every row's largest activations
    s1 = kw["w1_scale"].clone()
    s1.view(E, 2 * I)[:, 1:I:8] = float("nan")
    kw_nan = {**kw, "w1_scale": s1}
    torch.testing.assert_close(pra.fused_experts(x, *args[1:], **kw_nan),
                               pra.fused_experts(x, *args[1:], **kw_nan, gemm_variant="stream"), **SAME)
    mlp = (d.w1[0], s1[0].reshape(-1), *mlp[2:])
    torch.testing.assert_close(pra.w8a8_mlp(x, *mlp), pra.w8a8_mlp(x, *mlp, gemm_variant="stream"), **SAME)
