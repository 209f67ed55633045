"""What the entry points accept and refuse, and how they write their results, is the same whether the native call path
takes a call or leaves it to the Python path."""

import ctypes
import sys
import threading

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


def _calls(pra, M):
    """One call of every entry point the native path takes: (call, its result)."""
    d, args, kw = _layer(M)
    logits = torch.randn(M, 16, device=DEV)
    mlp = (d.w1[0], d.w1_scale[0].reshape(-1), d.w2[0], d.w2_scale[0].reshape(-1))
    gate, up, down = (torch.randn(s, device=DEV).to(torch.bfloat16) for s in ((2, 64, 128), (2, 64, 128), (2, 128, 64)))
    out = pra.quantize_expert_weights(gate, up, down)
    calls = (lambda: pra.fused_experts(*args, **kw), lambda: pra.fused_moe(d.hidden_states, d.w1, d.w2, logits, 4, True, **kw),
             lambda: pra.w8a8_mlp(d.hidden_states, *mlp), lambda: pra.apply_int8_linear(d.hidden_states, *mlp[:2]),
             lambda: pra.route_topk(logits, 4)[0], lambda: pra.quantize_expert_weights(gate, up, down, out=out)[0])
    return [(call, call().clone()) for call in calls]


def test_other_python_threads_run_during_the_launches(pra):
    """The interpreter lock is given up inside every call.  With a switch interval longer than the test nothing else
    makes this thread give it up, so another one gets it only there."""
    interval = sys.getswitchinterval()
    for call, _ in _calls(pra, 3):
        go, ran = threading.Event(), []

        def other():
            go.wait()
            ran.append(True)

        thread = threading.Thread(target=other)
        thread.start()
        sys.setswitchinterval(60.0)
        try:
            go.set()
            for _ in range(3000):
                if ran:
                    break
                call()
            seen = bool(ran)
        finally:
            sys.setswitchinterval(interval)
        thread.join()
        torch.cuda.synchronize()
        assert seen, call


@pytest.mark.parametrize("M", [2, 37, 200])
def test_threads_share_a_stream_and_its_workspace(pra, M):
    """Calls of several threads on one stream use one default workspace: their launches must not interleave."""
    calls, wrong = _calls(pra, M)[:4], []
    torch.cuda.synchronize()

    def work(call, want):
        for _ in range(60):
            if not torch.equal(call(), want):
                wrong.append(call)

    threads = [threading.Thread(target=work, args=c) for c in calls + calls]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_a_result_that_cannot_be_allocated_is_an_out_of_memory_error(pra):
    n, k = 16384, 64
    w, s = torch.zeros(n, k, dtype=torch.int8, device=DEV), torch.ones(n, device=DEV)
    x = torch.zeros(4096, k, dtype=torch.bfloat16, device=DEV)  # a result of 128 MB
    pra.apply_int8_linear(x, w[:16].contiguous(), s[:16])  # (the default workspace)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (16 << 20)) / total)
    try:
        with pytest.raises(torch.cuda.OutOfMemoryError):
            pra.apply_int8_linear(x, w, s)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert pra.apply_int8_linear(x, w, s).shape == (4096, n)


def test_what_the_python_path_refuses_is_refused(pra):
    d, args, kw = _layer(3)
    x, w1, w2 = args[:3]
    logits = torch.randn(3, 16, device=DEV)
    for block in (48, 2**32 + 64, 2**70):
        with pytest.raises(ValueError, match="block_size"):
            pra.fused_experts(*args, **kw, block_size_m=block)
        with pytest.raises(ValueError, match="block_size"):
            pra.fused_moe(x, w1, w2, logits, 4, True, **kw, block_size_m=block)
    for record in ((), [], False):
        with pytest.raises((ValueError, TypeError)):
            pra.route_topk(logits, 4, routed_experts_out=record)
        with pytest.raises((ValueError, TypeError)):
            pra.fused_moe(x, w1, w2, logits, 4, True, **kw, routed_experts_out=record)


def test_what_the_python_path_accepts_is_accepted(pra):
    d, args, kw = _layer(3)
    x, w1, w2 = args[:3]
    logits = torch.randn(3, 16, device=DEV)
    # group counts below one mean one group, as in grouped_topk
    w, ids = pra.grouped_topk(x, logits, 4, True, -1, -1)
    got = pra.fused_moe(x, w1, w2, logits, 4, True, **kw, use_grouped_topk=True, num_expert_group=-1, topk_group=-1)
    assert torch.equal(got, pra.fused_experts(x, w1, w2, w, ids, **kw))
    # the parameters to overwrite come as any iterable
    gate, up, down = (torch.randn(s, device=DEV).to(torch.bfloat16) for s in ((2, 64, 128), (2, 64, 128), (2, 128, 64)))
    want = pra.quantize_expert_weights(gate, up, down)
    for kind in (tuple, list, iter, lambda ts: (t for t in ts)):
        out = [torch.zeros_like(t) for t in want]
        got = pra.quantize_expert_weights(gate, up, down, out=kind(out))
        assert all(g is o and torch.equal(o, w) for g, o, w in zip(got, out, want))
    with pytest.raises(ValueError):
        pra.quantize_expert_weights(gate, up, down, out=want[:3])


@pytest.mark.parametrize("M", [1, 4, 16, 50])
@pytest.mark.parametrize("shift", [0, 16, -64])
def test_dense_output_may_overlap_its_input(pra, M, shift):
    """Through the C-ABI: the output on the input's memory, exactly or shifted by some elements."""
    K = 1024
    lib, abi = pra._abi.load(), pra._abi
    g = torch.Generator(device=DEV).manual_seed(M)
    x = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
    w = torch.randint(-127, 128, (K, K), dtype=torch.int8, device=DEV, generator=g)
    w13 = torch.randint(-127, 128, (2 * K, K), dtype=torch.int8, device=DEV, generator=g)
    s = torch.rand(2 * K, device=DEV, generator=g) * 1e-3
    ws = torch.empty(lib.moe_i8_dense_workspace_bytes(M, K, K), dtype=torch.uint8, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    for want, call in (
        (pra.apply_int8_linear(x, w, s[:K]), lambda i, o: lib.moe_i8_w8a8_linear(
            i, w.data_ptr(), s.data_ptr(), o, M, K, K, ws.data_ptr(), ws.numel(), abi.GEMM_AUTO, stream)),
        (pra.w8a8_mlp(x, w13, s, w, s[:K]), lambda i, o: lib.moe_i8_w8a8_mlp(
            i, w13.data_ptr(), s.data_ptr(), w.data_ptr(), s.data_ptr(), o, M, K, K, ws.data_ptr(), ws.numel(), abi.GEMM_AUTO, stream)),
    ):
        memory = torch.zeros(M * K + 128, dtype=torch.bfloat16, device=DEV)
        memory[64:64 + M * K] = x.view(-1)
        at = memory.data_ptr() + 2 * 64
        abi.check(call(at, at + 2 * shift))
        assert torch.equal(memory[64 + shift:64 + shift + M * K].view(M, K), want)


@pytest.mark.parametrize("M", [1, 5, 200])
def test_the_python_path_alone_gives_the_same_results(pra, monkeypatch, M):
    calls = _calls(pra, M)
    monkeypatch.setattr(pra._abi, "_host", pra._abi.PythonPathOnly())
    for call, want in calls:
        assert torch.equal(call(), want)


@pytest.mark.parametrize("M", [1, 2, 8, 9, 37, 200, 1500, 9000])
@pytest.mark.parametrize("E", [16, 128])
def test_layer_launches_are_what_a_captured_call_records(pra, M, E):
    k, H, I = 4, 512, 256
    d, args, kw = _layer(M, E=E, k=k, H=H, I=I)
    lib = pra._abi.load()  # (its handle finds the HIP runtime it is linked with)
    logits = torch.randn(M, E, device=DEV)
    w, ids = torch.empty(M, k, device=DEV), torch.empty(M, k, dtype=torch.int32, device=DEV)
    out = torch.empty_like(d.hidden_states)
    ws = torch.empty(pra.workspace_bytes(M, k, E, H, I, 64), dtype=torch.uint8, device=DEV)

    def routed():
        pra._abi.check(lib.moe_i8_fused_moe(
            d.hidden_states.data_ptr(), logits.data_ptr(), d.w1.data_ptr(), d.w2.data_ptr(), d.w1_scale.data_ptr(),
            d.w2_scale.data_ptr(), out.data_ptr(), M, k, E, H, I, 64, 0, None, 1, 1, 0, 1, 1.0, w.data_ptr(), ids.data_ptr(),
            None, 0, 0, 0, ws.data_ptr(), ws.numel(), 0, torch.cuda.current_stream().cuda_stream))

    for call, is_routed in ((lambda: pra.fused_experts(*args, **kw, workspace=ws, out=out), False), (routed, True)):
        call()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            call()
        nodes = ctypes.c_size_t()
        assert lib.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(nodes)) == 0
        assert nodes.value == pra.layer_launches(M, k, E, H, I, routed=is_routed)
