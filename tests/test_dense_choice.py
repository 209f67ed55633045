"""Which kernel and tile a dense call is given, and that the GPU tests of the dense kernels run every one of them."""

import pytest

import test_gpu_dense_kernel as gpu


def _cases(*tests):
    return [c for t in tests for mark in t.pytestmark if mark.name == "parametrize" for c in mark.args[1]]


def _reached(pra, cases):
    """The kernels and table entries of the linear layer and of the gated MLP's gate_up that the GPU tests run for these sizes."""
    linear, gate_up = set(), set()
    for m, n, k in cases:
        p = pra.linear_plan(m, n, k)
        linear.add((p["kernel"], p["entry"], p["through"]))
        inter = n // 2 // 64 * 64
        if inter:
            p = pra.mlp_plan(m, k, inter)["gate_up"]
            gate_up.add((p["kernel"], p["entry"], p["through"]))
    return linear, gate_up


def test_every_tile_of_rows_that_their_workgroups_quantise_is_run(pra):
    linear, gate_up = _reached(pra, _cases(gpu.test_rows_quantised_by_their_tiles, gpu.test_rows_quantised_by_wide_tiles))
    every = {("dense_rows", i, True) for i in range(10)}
    assert linear == every and gate_up >= every


def test_every_tile_of_the_dense_kernel_is_run(pra):
    linear, gate_up = _reached(pra, _cases(gpu.test_linear_and_mlp, gpu.test_large_tiles, gpu.test_tiles_of_96,
                                           gpu.test_tiles_of_few_and_of_short_problems, gpu.test_results_of_more_than_96_mb))
    every = {("dense", i, True) for i in range(13)} | {("dense", i, False) for i in (8, 10, 11, 12)}
    assert linear >= every and gate_up >= every
    assert {p for p in linear | gate_up if p[0] == "dense"} == every


def test_the_kernel_of_a_few_rows_is_run_with_every_number_of_rows_a_wavefront_can_have(pra):
    few = [(m, n, k) for m, n, k in _cases(gpu.test_few_rows_in_one_launch, gpu.test_most_rows_in_one_launch)
           if pra.linear_plan(m, n, k)["kernel"] == "dense_few"]
    assert {1, 2, 8, 13, 16} <= {m for m, _, _ in few}  # one row a wavefront, the second one of some and of all of them
    assert {(k + 1023) // 1024 for _, _, k in few} == set(range(1, 9))


def test_plans_follow_a_demanded_family_and_reject_what_a_call_rejects(pra):
    assert pra.linear_plan(333, 4096, 2048, gemm_variant="stream") == {"kernel": "stream", "tile": None, "entry": None, "through": False}
    assert pra.mlp_plan(333, 4096, 2048, gemm_variant="tile_wide")["down"]["kernel"] == "tile_wide"
    assert pra.linear_plan(333, 4096, 2048)["tile"] == (64, 128)
    assert pra.linear_plan(17, 2672, 896)["kernel"] == "dense_rows"
    assert pra.mlp_plan(5, 4096, 1408) == {w: {"kernel": "dense_few", "tile": None, "entry": None, "through": False} for w in ("gate_up", "down")}
    for sizes in ((0, 4096, 2048), (8, 4090, 2048), (8, 4096, 2016)):
        with pytest.raises(pra._abi.MoeI8Error):
            pra.linear_plan(*sizes)
    with pytest.raises(pra._abi.MoeI8Error):
        pra.mlp_plan(8, 4096, 1400)
    with pytest.raises(pra._abi.MoeI8Error):
        pra.linear_plan(8, 4096, 2048 + 64, gemm_variant="tile_wide")  # a reduction of no whole 128 bytes
    assert pra._abi.load().moe_i8_mlp_plan(8, 4096, 1408, pra._abi.GEMM_AUTO, None, None) == pra._abi.OK


def test_a_grouped_down_gemm_finds_the_routing_that_the_first_quantisation_writes(pra):
    """Weights of 4 GiB, which the dense kernels do not take: the kernel of a few rows writes no routing, so it does not run the
    gate_up in front of them, though it could."""
    plan = pra.mlp_plan(2, 8192, 1 << 19)
    assert plan["down"]["kernel"] == plan["gate_up"]["kernel"] == "stream"
    assert pra.linear_plan(2, 1 << 20, 8192)["kernel"] == "dense_few"


@pytest.mark.parametrize("m,hidden,inter,kernel,tile", [
    # gate_up with wide tiles, us: 2048 rows of 1024 x 3968 26.6 (192 x 384 tiles 30.4), 6510 of 640 x 5632 72.0 (81.4)
    (2048, 1024, 3968, "tile_wide", None),
    (6510, 640, 5632, "tile_wide", None),
    (4096, 4096, 1408, "tile_wide", None),  # 58.6 (256 x 192 tiles 58.5: even)
    (5047, 2304, 960, "dense", (256, 192)),  # 40.2 (37.7)
    (7411, 3840, 1088, "dense", (192, 384)),  # 95.7 (80.1)
])
def test_gate_up_is_charged_for_the_results_it_stores(pra, m, hidden, inter, kernel, tile):
    plan = pra.mlp_plan(m, hidden, inter)["gate_up"]
    assert (plan["kernel"], plan["tile"]) == (kernel, tile)


@pytest.mark.parametrize("m,n,k,kernel", [
    # us in the kernel of a few rows / in the one that quantises its tiles' rows: 5.2 / 3.6, 4.8 / 3.3, 4.5 / 3.2, 6.7 / 4.3
    (6, 6272, 192, "dense_rows"), (7, 4496, 256, "dense_rows"), (11, 864, 256, "dense_rows"), (16, 640, 1280, "dense_rows"),
    (4, 6272, 192, "dense_few"),  # up to 4 rows whatever the reduction
    # 3.5 / 4.2, 4.6 / 5.7, 5.0 / 7.2
    (5, 1792, 832, "dense_few"), (5, 3760, 2368, "dense_few"), (5, 640, 3904, "dense_few"),
    (5, 4096, 1408, "dense_few"),  # the gated MLP of it 10.0 / 10.75
    # 3.8 / 4.4, 4.0 / 4.5, 3.7 / 4.4, 6.3 / 8.2, 6.9 / 9.0
    (5, 3680, 576, "dense_few"), (6, 3264, 704, "dense_few"), (5, 2864, 576, "dense_few"), (6, 4080, 3072, "dense_few"),
    (8, 3504, 3392, "dense_few"),
])
def test_line_between_the_kernels_that_quantise_their_rows(pra, m, n, k, kernel):
    assert pra.linear_plan(m, n, k)["kernel"] == kernel


@pytest.mark.parametrize("m,n,k,kernel", [
    # us in the dense tile that the estimates come to next / with wide tiles: 43.9 / 35.2, 77.8 / 63.0, 82.4 / 69.5, 67.4 / 53.2
    (14508, 3328, 256, "tile_wide"), (9405, 11520, 256, "tile_wide"), (8747, 8448, 640, "tile_wide"), (5836, 14784, 256, "tile_wide"),
    (5780, 2672, 512, "dense"),  # 19.4 / 24.8
])
def test_linear_layers_of_short_reductions_are_charged_for_their_results(pra, m, n, k, kernel):
    assert pra.linear_plan(m, n, k)["kernel"] == kernel
