"""GPU parity of the dense GEMM kernel at the sizes where its tiles and its split reduction can go wrong:
one row, tile edges and remainders of every tile the library picks by itself, channels that fill no tile,
reductions shorter than a workgroup's split and odd multiples of 64."""

import pytest
import torch

DEV = "cuda:0"
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [
    (1, 16, 64), (1, 2144, 1536), (3, 528, 6080), (16, 4096, 704), (17, 2528, 5056), (31, 48, 192), (33, 4096, 1088),
    (64, 8192, 1984), (65, 1904, 3968), (129, 4112, 2112), (333, 4096, 2048), (500, 10240, 1472), (1000, 6144, 832),
    (2049, 4096, 576), (5000, 528, 1024),
])
def test_linear_and_mlp(pra, oracle, M, N, K):
    g = torch.Generator().manual_seed(M * 7 + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    s = torch.rand(N, generator=g) * 0.008 + 0.002
    out = pra.apply_int8_linear(x.to(DEV), w.to(DEV), s.to(DEV))
    assert torch.equal(out.cpu(), oracle.w8a8_linear(x, w, s))
    # the gated MLP: gate_up over N rows of weights, down back to K channels, against the streaming family
    inter = N // 2 // 64 * 64
    if inter:
        w13, s13 = w[: 2 * inter].to(DEV), (s[: 2 * inter] * 0.1).to(DEV)
        w2 = torch.randint(-127, 128, (K, inter), generator=g, dtype=torch.int8).to(DEV)
        s2 = (torch.rand(K, generator=g) * 1e-3 + 1e-3).to(DEV)
        got = pra.w8a8_mlp(x.to(DEV), w13, s13, w2, s2)
        assert torch.equal(got, pra.w8a8_mlp(x.to(DEV), w13, s13, w2, s2, gemm_variant="stream"))


@pytest.mark.parametrize("M,N,K", [
    (1, 16, 64), (1, 8192, 8192), (2, 304, 1088), (3, 9344, 2048), (4, 4096, 8128), (5, 2816, 4096), (6, 8192, 4096),
    (7, 1648, 3008), (8, 2064, 5120), (8, 12288, 960), (9, 400, 1024), (16, 1024, 1024), (13, 176, 5952),
])
def test_few_rows_in_one_launch(pra, oracle, M, N, K):
    """Rows quantised by the workgroups that multiply them: every row count per wavefront, remainders of
    channels and of the 1 KB pieces of a reduction, more channel groups than workgroups."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    x[0, : K // 2] = torch.arange(K // 2) % 255 - 127  # exact ties and the largest values
    w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    s = torch.rand(N, generator=g) * 0.008 + 0.002
    assert torch.equal(pra.apply_int8_linear(x.to(DEV), w.to(DEV), s.to(DEV)).cpu(), oracle.w8a8_linear(x, w, s))
    inter = N // 2 // 64 * 64
    if inter:
        w2 = torch.randint(-127, 128, (K, inter), generator=g, dtype=torch.int8).to(DEV)
        args = (x.to(DEV), w[: 2 * inter].to(DEV), (s[: 2 * inter] * 0.1).to(DEV), w2, (torch.rand(K, generator=g) * 1e-3).to(DEV))
        assert torch.equal(pra.w8a8_mlp(*args), pra.w8a8_mlp(*args, gemm_variant="stream"))


@pytest.mark.parametrize("M,N,K", [
    (16, 16, 64), (17, 560, 576), (33, 1040, 1024), (64, 864, 384), (5, 10880, 384), (100, 2064, 960), (500, 272, 1024),
    (13, 11568, 256), (31, 8208, 512), (43, 11616, 640), (65, 8464, 192), (245, 2752, 1024), (600, 1552, 448), (54, 1248, 1152),
    (16, 4112, 2048), (28, 8208, 1088), (30, 8176, 2048), (47, 5008, 1984), (9, 16912, 1344), (45, 624, 2880), (17, 1040, 4096),
    (15, 528, 2112), (16, 2544, 3968), (16, 64, 4096), (69, 1280, 3904), (31, 8496, 576),
])
def test_rows_quantised_by_their_tiles(pra, oracle, M, N, K):
    """Rows quantised by the workgroups whose tiles they are in: every tile and length of its registers, rows and channels
    that fill no tile, reductions of odd multiples of 64 and shorter than a workgroup's split, one round and several."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    x[0, : K // 2] = torch.arange(K // 2) % 255 - 127  # exact ties and the largest values
    x[M // 2] = 0
    x[M - 1, K - 1] = float("nan")  # skipped in the maximum, 0 as a value
    clean = x.nan_to_num(0.0)
    w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    s = torch.rand(N, generator=g) * 0.008 + 0.002
    assert torch.equal(pra.apply_int8_linear(x.to(DEV), w.to(DEV), s.to(DEV)).cpu(), oracle.w8a8_linear(clean, w, s))
    inter = N // 2 // 64 * 64
    if inter:
        w2 = torch.randint(-127, 128, (K, inter), generator=g, dtype=torch.int8).to(DEV)
        args = (w[: 2 * inter].to(DEV), (s[: 2 * inter] * 0.1).to(DEV), w2, (torch.rand(K, generator=g) * 1e-3).to(DEV))
        assert torch.equal(pra.w8a8_mlp(x.to(DEV), *args), pra.w8a8_mlp(clean.to(DEV), *args, gemm_variant="stream"))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [
    (673, 5552, 576), (643, 5392, 192), (1421, 5584, 576), (1300, 5904, 64), (2051, 5616, 576), (1800, 6176, 192),
    (2315, 6176, 576), (4804, 2912, 64), (2309, 6192, 1088),
    (9935, 1168, 448), (779, 14608, 448), (1054, 14592, 64),                            # 192 x 320 and 192 x 384
    (11398, 4416, 576), (18529, 2720, 64), (21775, 2592, 576), (21327, 2368, 576),      # more than 96 MB of results
])
def test_large_tiles(pra, oracle, M, N, K):
    """The tiles whose results are finished in registers, one round of them and several: rows and channels that fill no tile,
    reductions of odd multiples of 64 and of one step, plain results and gate_up's."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8)
    s = torch.rand(N, generator=g) * 0.008 + 0.002
    dx, dw, ds = x.to(DEV), w.to(DEV), s.to(DEV)
    out = pra.apply_int8_linear(dx, dw, ds)
    assert torch.equal(out, pra.apply_int8_linear(dx, dw, ds, gemm_variant="stream"))
    rows = torch.cat([torch.arange(0, M, 97), torch.arange(M - 40, M)])
    assert torch.equal(out[rows.to(DEV)].cpu(), oracle.w8a8_linear(x[rows], w, s))
    inter = N // 2 // 64 * 64
    w2 = torch.randint(-127, 128, (K, inter), generator=g, dtype=torch.int8).to(DEV)
    args = (dw[: 2 * inter], ds[: 2 * inter] * 0.1, w2, (torch.rand(K, generator=g) * 1e-3).to(DEV))
    assert torch.equal(pra.w8a8_mlp(dx, *args), pra.w8a8_mlp(dx, *args, gemm_variant="stream"))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(570, 3824, 1600), (1400, 1600, 576), (1921, 1040, 4160), (1913, 1072, 4096), (560, 3776, 2560)])
def test_tiles_of_96(pra, oracle, M, N, K):
    """96 x 96 tiles, their reduction halved: rows and channels that fill no tile, an odd number of pieces and one of 64 bytes."""
    test_large_tiles(pra, oracle, M, N, K)


@pytest.mark.parametrize("M,N,K", [
    (250, 3632, 960), (14, 50000, 448), (45, 11600, 1024), (33, 21760, 64),              # 16 x 256
    (97, 10512, 64), (700, 1968, 576), (209, 4624, 1024), (481, 4080, 512), (1690, 768, 960),  # 32 x 256
    (250, 8208, 448), (449, 8176, 512), (1000, 4096, 192),                               # 32 x 512
])
def test_rows_quantised_by_wide_tiles(pra, oracle, M, N, K):
    """Tiles whose wavefronts do not split the reduction: rows and channels that fill no tile, reductions of one step and up to the longest."""
    test_rows_quantised_by_their_tiles(pra, oracle, M, N, K)


@pytest.mark.parametrize("M,N,K", [(16, 128, 8192), (16, 240, 4224), (15, 128, 6016), (14, 144, 7168), (6, 8192, 4160), (6, 4096, 8192)])
def test_most_rows_in_one_launch(pra, oracle, M, N, K):
    """As many rows as one launch of the kernel of a few rows takes, where no other kernel that quantises its rows can run."""
    assert pra.linear_plan(M, N, K)["kernel"] == "dense_few"
    assert pra.mlp_plan(M, K, N // 2 // 64 * 64)["gate_up"]["kernel"] == "dense_few"
    test_few_rows_in_one_launch(pra, oracle, M, N, K)


@pytest.mark.parametrize("M,N,K", [(3, 160, 8384), (21, 208, 5056), (23, 9008, 2496), (4717, 688, 64), (1182, 3680, 64)])  # 16 x 16, 32 x 64, 128 x 128
def test_tiles_of_few_and_of_short_problems(pra, oracle, M, N, K):
    test_linear_and_mlp(pra, oracle, M, N, K)


@pytest.mark.parametrize("M,N,K", [
    (1371, 75024, 192), (967, 106960, 448), (37219, 2832, 192), (25597, 3984, 64),  # 128 x 128, two workgroups to a compute unit
    (1926, 55008, 1216),  # 256 x 192
    (85854, 1280, 448),   # 192 x 320
    (960, 114992, 448),   # 192 x 384
])
def test_results_of_more_than_96_mb(pra, oracle, M, N, K):
    """Results that are left in the L2s, gate_up's as well (M x N / 2), in every tile that is picked for so many."""
    assert not pra.linear_plan(M, N, K)["through"] and not pra.mlp_plan(M, K, N // 2 // 64 * 64)["gate_up"]["through"]
    test_large_tiles(pra, oracle, M, N, K)
