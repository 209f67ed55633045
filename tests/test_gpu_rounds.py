"""GPU parity of the kernels with LDS-staged tiles where an XCD's last round of tasks is cut into pieces (channels of the narrow
and deep tiles, blocks of the wide ones), and where tasks start their reductions at different steps (a stride of 4096
bytes): int32 accumulators against the oracle's, exactly."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(pra, oracle, variant, counts, N, K, B=64):
    gen = torch.Generator().manual_seed(N + K + len(counts))
    E, P = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(E, dtype=torch.int32), torch.tensor(counts))
    ids = ids[torch.randperm(P, generator=gen)].view(P, 1)
    a = torch.randint(-127, 128, (P, K), dtype=torch.int8, generator=gen)
    w = torch.randint(-127, 128, (E, N, K), dtype=torch.int8, generator=gen)
    s, e, npp = pra.moe_align_block_size(ids.to(DEV), B, E)
    got = pra.gemm_acc_i32(a.to(DEV), w.to(DEV), s, e, npp, 1, B, P, variant).cpu()
    want = oracle.grouped_int_gemm(a, w, ids, 1)
    assert torch.equal(got, want.view_as(got)), int((got != want.view_as(got)).sum())


# (an XCD has 32 workgroups and up to ceil(tiles / 8) tasks, the last one a few less; 70 rows are one deep or wide tile and two narrow
# ones, 64 are one of each: in one tile these are 1, 8 and 9, 16 and 17 tasks, which is where a round of 32 is no longer cut into
# four and into two pieces, then 33, 40 and 41, 49, 67; in two about twice as many)
@pytest.mark.parametrize("variant,rows", [("narrow", 70), ("tile_deep", 70), ("tile_wide", 70), ("narrow", 64)])
@pytest.mark.parametrize("tiles", [1, 63, 65, 127, 129, 135, 257, 256 + 64, 256 + 72, 256 + 130, 512 + 17])
def test_rest_of_the_last_round(pra, oracle, variant, rows, tiles):
    channels = 128 if variant == "narrow" else 256
    _check(pra, oracle, variant, [rows], tiles * channels - 16 * (tiles % 3), 512)


# The layer's task list is built from ids that are known to ascend.  Eight tiles: an XCD gets as many tasks as there are channel
# tiles; the other routings put several tiles of an expert into a group (deep tiles 9 and 8, wide ones 5 and 4).
@pytest.mark.parametrize("variant", ["tile_deep", "tile_wide"])
@pytest.mark.parametrize("counts", [[100, 0, 1, 64, 65, 128, 33, 7, 90], [700, 0, 130, 40], [1000]])
@pytest.mark.parametrize("ntiles", [3, 8, 9, 16, 17, 31, 32, 33, 40, 41, 48, 49, 65])
def test_layer_tasks_around_a_round(pra, variant, counts, ntiles):
    from _util import inputs_mod

    im, M = inputs_mod(), sum(counts)
    for H, I in ((512, 128 * ntiles), (256 * ntiles, 512)):  # the first GEMM's channel tiles, the second one's
        d = im.make_inputs(im.LayerShape("r", E=len(counts), k=1, H=H, I=I), M, seed=ntiles, device=DEV, weights_on_device=True)
        ids = torch.repeat_interleave(torch.arange(len(counts), dtype=torch.int32), torch.tensor(counts))
        d.topk_ids.copy_(ids[torch.randperm(M, generator=torch.Generator().manual_seed(ntiles))].view(M, 1))
        kw = d.fused_experts_kwargs()
        got = pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant=variant)
        assert torch.equal(got, pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="stream")), (H, I)


@pytest.mark.parametrize("variant,K", [("tile_deep", 384), ("tile_wide", 256)])
def test_more_channel_tiles_than_fifteen_bits_count(pra, variant, K):
    N, P = 32768 * 256 + 5 * 256 + 16, 40
    gen = torch.Generator(device=DEV).manual_seed(K)
    a = torch.randint(-127, 128, (P, K), dtype=torch.int8, device=DEV, generator=gen)
    w = torch.randint(-127, 128, (1, N, K), dtype=torch.int8, device=DEV, generator=gen)
    s, e, npp = pra.moe_align_block_size(torch.zeros((P, 1), dtype=torch.int32, device=DEV), 64, 1)
    got = pra.gemm_acc_i32(a, w, s, e, npp, 1, 64, P, variant).view(P, N)
    # (the magnitude of every partial sum is below 384 * 127 * 127 < 2^24: exact in float32)
    for at in range(0, N, 1 << 20):
        want = a.float() @ w[0, at:at + (1 << 20)].float().T
        assert torch.equal(got[:, at:at + (1 << 20)].float(), want), at


@pytest.mark.parametrize("variant", ["narrow", "tile_deep", "tile_wide"])
@pytest.mark.parametrize("counts", [[260, 5, 0, 64, 129], [1] * 37])
def test_pieces_of_tiles_of_several_sizes(pra, oracle, variant, counts):
    _check(pra, oracle, variant, counts, 2 * 256 + 48, 768)
    _check(pra, oracle, variant, counts, 256, 768, B=128)


@pytest.mark.parametrize("variant", ["narrow", "tile_deep", "tile_wide", "stream"])
@pytest.mark.parametrize("K", [4096, 8192])
@pytest.mark.parametrize("experts", [1, 5, 8, 31, 33, 70])
def test_tasks_that_start_at_different_steps(pra, oracle, variant, K, experts):
    # 70 experts: the starting step wraps around twice; below 32 the starts are several steps apart
    _check(pra, oracle, variant, [(7 * i + 3) % 40 for i in range(experts)], 272, K)


@pytest.mark.parametrize("variant", ["narrow", "tile_deep"])
@pytest.mark.parametrize("inter", [768, 1024])
@pytest.mark.parametrize("skewed", [False, True])
def test_starting_steps_of_long_launches(pra, variant, inter, skewed):
    # 0.75 GiB and 1 GiB of weights in the first GEMM: on either side of the line
    from _util import inputs_mod

    im = inputs_mod()
    E, rows = 64, 24
    d = im.make_inputs(im.LayerShape("s", E=E, k=1, H=8192, I=inter), E * rows, seed=inter, device=DEV, weights_on_device=True)
    ids = torch.arange(E * rows) % E if not skewed else torch.cat([torch.arange(E), torch.full((400,), 5), torch.arange(E * (rows - 1) - 400) % 50])
    d.topk_ids.copy_(ids.to(torch.int32).view(-1, 1))
    kw = d.fused_experts_kwargs()
    got = pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant=variant)
    assert torch.equal(got, pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="stream"))


@pytest.mark.parametrize("steps", [4, 5, 6, 7, 8])
@pytest.mark.parametrize("most", [20, 60])
def test_narrow_reductions_around_the_depth_of_the_ring(pra, oracle, steps, most):
    # tiles of 64 token rows have six stages; those of 32 (no expert with more rows) seven, in the layer only
    _check(pra, oracle, "narrow", [most - i % 13 for i in range(24)], 1024 + 16, steps * 128)


@pytest.mark.parametrize("H,I", [(512, 1024), (768, 512), (896, 896), (4096, 1024)])
def test_narrow_layer_of_32_tokens(pra, H, I):
    from _util import inputs_mod

    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("n", E=24, k=4, H=H, I=I), 32, seed=H).to(DEV)
    kw = d.fused_experts_kwargs()
    got = pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="narrow")
    assert torch.equal(got, pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="stream"))


@pytest.mark.parametrize("H", [384, 512, 640])
@pytest.mark.parametrize("tokens", [120, 300, 1500])
def test_deep_layer_around_the_depth_of_the_ring(pra, H, tokens):
    # 3 to 5 steps in the first GEMM; several tasks per workgroup, so that a task's first steps run behind stores
    from _util import inputs_mod

    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("d", E=40, k=4, H=H, I=2560), tokens, seed=H + tokens).to(DEV)
    kw = d.fused_experts_kwargs()
    got = pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="tile_deep")
    assert torch.equal(got, pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="stream"))


@pytest.mark.parametrize("tokens", [255, 256, 300])
def test_narrow_results_around_the_size_that_is_written_through(pra, tokens):
    # 4 * tokens rows of 4096 bf16 from the second GEMM: 8 MB at 256 tokens
    from _util import inputs_mod

    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("t", E=24, k=4, H=4096, I=512), tokens, seed=tokens).to(DEV)
    kw = d.fused_experts_kwargs()
    got = pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="narrow")
    assert torch.equal(got, pra.fused_experts(*d.fused_experts_args(), **kw, gemm_variant="stream"))
