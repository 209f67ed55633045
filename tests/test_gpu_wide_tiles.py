"""GPU parity of the wide tiles at the edges of their row tiles (32 rows of 256), at the shortest reductions (two and
three steps) and with more tasks per workgroup than its table holds, against the streaming family."""

import pytest
import torch

from _util import inputs_mod

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B", [64, 128])
@pytest.mark.parametrize("H,I", [(256, 384), (384, 256), (1408, 640), (4096, 256), (1920, 256), (2048, 256)])  # (even tiles from a reduction of 2048 on)
def test_rows_around_the_edges_of_row_tiles(pra, H, I, B):
    counts = [1, 31, 32, 33, 63, 65, 127, 128, 129, 160, 161, 0, 224, 255, 256, 257, 300, 511, 513]
    M = sum(counts)
    im = inputs_mod()
    d = im.make_inputs(im.LayerShape("w", E=len(counts), k=1, H=H, I=I), M, seed=H + B).to(DEV)
    ids = torch.repeat_interleave(torch.arange(len(counts), dtype=torch.int32), torch.tensor(counts))
    d.topk_ids.copy_(ids[torch.randperm(M, generator=torch.Generator().manual_seed(1))].view(M, 1))
    kw = d.fused_experts_kwargs()
    got = pra.fused_experts(*d.fused_experts_args(), **kw, block_size_m=B, gemm_variant="tile_wide")
    assert torch.equal(got, pra.fused_experts(*d.fused_experts_args(), **kw, block_size_m=B, gemm_variant="stream"))


@pytest.mark.parametrize("E,N,P,k", [(520, 8320, 600, 3), (1, 8320, 5000, 1), (3, 304, 2000, 7)])
def test_many_tasks_and_row_divisors(pra, E, N, P, k):
    K, M = 256, (P + k - 1) // k
    gen = torch.Generator(device=DEV).manual_seed(E)
    w = torch.randint(-127, 128, (E, N, K), dtype=torch.int8, device=DEV, generator=gen)
    a = torch.randint(-127, 128, (M, K), dtype=torch.int8, device=DEV, generator=gen)
    ids = torch.randint(0, E, (M, k), dtype=torch.int32, device=DEV, generator=gen)
    s, e, npp = pra.moe_align_block_size(ids, 64, E)
    got = pra.gemm_acc_i32(a, w, s, e, npp, k, 64, M * k, "tile_wide")
    assert torch.equal(got, pra.gemm_acc_i32(a, w, s, e, npp, k, 64, M * k, "stream"))
