"""Graph capture of the boundary's entry points.

* The reference-signature op gptq_dequant_matmul_fused (inference/kernels/
  __init__.py:284-346) runs inside the reference's CUDA-graph capture
  (GLoRCQLinear.forward, inference/quantized_linear.py:307-311, under
  graph_wrapper.py:69-131).  After one warm-up call on the same codes it does
  no host sync and no repack, so it captures; every replay must equal the
  eager result bit for bit (same kernels, same inputs).
* A workspace replaced by a larger one stays allocated: a graph captured with
  the old buffer still writes into it, and memory allocated after the
  replacement must not be overwritten by its replays.

Each replay is separated by eager work and a synchronization, and checked.
"""

import pytest
import torch

from glorcq_amd import kernels as K_
from test_gptq_gpu import gptq_data, lora

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N,K,usv", [(1, 1408, 2048, False), (4, 2048, 1408, True),
                                       (32, 1408, 2048, True)])
def test_gptq_signature_captures_after_warmup(gpu, B, N, K, usv):
    x, q, s, z = gptq_data(B, N, K, seed=B)
    x, q, s, z = x.to(gpu), q.to(gpu), s.to(gpu), z.to(gpu)
    lu = tuple(t.to(gpu) for t in lora(K, N)) if usv else None
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        eager = K_.gptq_dequant_matmul_fused(x, q, s, z, 128, False, lora_USV=lu)  # warm-up
        eager = eager.clone()
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = K_.gptq_dequant_matmul_fused(x, q, s, z, 128, False, lora_USV=lu)
    torch.cuda.synchronize()
    for i in range(3):
        y.fill_(float("nan"))
        _ = (x * 2).sum()  # eager work between replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager), f"replay {i}"
    # the prepared codes are reused only while the tensor is unchanged
    q.add_(0)
    y2 = K_.gptq_dequant_matmul_fused(x, q, s, z, 128, False, lora_USV=lu)
    assert torch.equal(y2, eager)


def test_replaced_workspace_survives_for_captured_graph(gpu):
    """Capture a multi-row GEMV (x U partials in the per-stream workspace),
    then grow that stream's workspace with a larger eager call; replays still
    give the eager result and leave later allocations alone."""
    from glorcq_amd import format as fmt

    small = fmt.make_linear(512, 256, bits=4, group=128, rank=64, M=4, seed=3)
    # K = 8192 at 16 rows and rank 128: 32 K-slices x 16 x 128 x 4 B = 256 KiB of
    # partials, past the first buffer's 64 KiB
    big = fmt.make_linear(8192, 512, bits=4, group=128, rank=128, M=16, seed=4)
    d = lambda t: t.to(gpu)  # noqa: E731
    args = (d(small.x), d(small.codes), d(small.scales), d(small.zeros), 4, 128)
    kw = dict(U=d(small.U), SV=d(small.SV))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        eager = K_.packed_dequant_matmul_fused(*args, **kw).clone()
        ws0 = K_.gemv_workspace(gpu, 1)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        y = K_.packed_dequant_matmul_fused(*args, **kw)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        K_.packed_dequant_matmul_fused(d(big.x), d(big.codes), d(big.scales), d(big.zeros), 4,
                                       128, U=d(big.U), SV=d(big.SV))
        ws1 = K_.gemv_workspace(gpu, 1)
    torch.cuda.synchronize()
    assert ws1.data_ptr() != ws0.data_ptr(), "the large call should have grown the workspace"
    del ws0
    sentinels = [torch.full((1 << 16,), 7, dtype=torch.uint8, device=gpu) for _ in range(16)]
    for i in range(3):
        y.fill_(0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, eager), f"replay {i}"
        assert all(bool((t == 7).all()) for t in sentinels), f"replay {i} wrote into new memory"


def _recorded(monkeypatch, name, ws_arg):
    """Wraps a library entry point; the list collects its calls' workspaces as
    (first byte, bytes)."""
    from glorcq_amd import _lib

    lib, seen = _lib.load(), []
    real = getattr(lib, name)

    def call(*a):
        seen.append((a[ws_arg], a[ws_arg + 1]))
        return real(*a)

    monkeypatch.setattr(lib, name, call)
    return seen


def _two_graphs(gpu, seen, calls):
    """Captures the calls on one stream, a graph each, checks that their
    scratch does not overlap, and replays them on two streams at once."""
    stream = torch.cuda.Stream()
    graphs, outs, eager, spans = [], [], [], []
    for call in calls:
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            eager.append(call().clone())
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        n = len(seen)
        with torch.cuda.graph(g, stream=stream):
            outs.append(call())
        assert len(seen) > n, "the call under test was not reached"
        spans.append(seen[n:])
        graphs.append(g)
    assert all(a + n <= b or b + m <= a for a, n in spans[0] for b, m in spans[1]), spans
    sides = [torch.cuda.Stream(), torch.cuda.Stream()]
    for i in range(3):
        for o in outs:
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        for s, g in zip(sides, graphs):
            with torch.cuda.stream(s):
                for _ in range(4):
                    g.replay()
        torch.cuda.synchronize()
        for o, e in zip(outs, eager):
            assert torch.equal(o, e), f"replay {i}"


def test_moe_batch_graphs_of_one_stream_replay_on_two(gpu, monkeypatch):
    """MoE batches that run as a prompt, of two sizes, captured on one stream:
    each graph has its own scratch, so they may run side by side."""
    from glorcq_amd import format as fmt
    from glorcq_amd.moe_block import GraphCompatibleMoeBlock

    p = fmt.make_moe(H=512, E=8, inter=640, top_k=2, n_clusters=3, rank=40, shared_inter=512,
                     B=64, seed=3)
    blk = GraphCompatibleMoeBlock.from_problem(p, gpu)
    hs = [p.h[:T].reshape(1, T, p.H).to(gpu) for T in (64, 20)]
    assert all(blk._as_prompt(h.shape[1]) for h in hs)
    blk._prompt_pays = lambda T: True
    seen = _recorded(monkeypatch, "glq_moe_prefill", 1)
    _two_graphs(gpu, seen, [lambda h=h: blk(h)[0] for h in hs])


def test_turbo_prompt_graphs_of_one_stream_replay_on_two(gpu, monkeypatch):
    """The same for TurboQuant prompts."""
    from glorcq_amd import format as fmt
    from glorcq_amd.moe_block import GraphCompatibleMoeBlock

    p = fmt.make_turbo_moe(H=512, E=6, inter=384, top_k=2, n_clusters=3, rank=64, B=100, seed=3,
                           rot_gate_up="rht", rot_down="qr")
    blk = GraphCompatibleMoeBlock.from_problem(p, gpu)
    hs = [p.h[:T].reshape(1, T, p.H).to(gpu) for T in (100, 17)]
    seen = _recorded(monkeypatch, "glq_turbo_moe_prefill", 1)
    _two_graphs(gpu, seen, [lambda h=h: blk(h)[0] for h in hs])


@pytest.mark.parametrize("given", [False, True])
def test_prompt_linear_graphs_of_one_stream_replay_on_two(gpu, monkeypatch, given):
    """Projections over many rows that form no x U (no low-rank term, or a
    precomputed one), in the tile form: x in decode order and its group sums
    are the call's own."""
    from glorcq_amd import format as fmt

    monkeypatch.setenv("GLQ_PF_TILE", "64")
    p = fmt.make_linear(1024, 512, bits=4, group=128, rank=16, M=500, seed=5)
    d = {k: getattr(p, k).to(gpu) for k in ("x", "codes", "scales", "zeros", "U", "SV")}
    xu = (p.x.float() @ p.U.float()).half().to(gpu)

    def call(M):
        kw = dict(SV=d["SV"], precomputed_xU=xu[:M]) if given else {}
        return lambda: K_.packed_dequant_matmul_fused(d["x"][:M], d["codes"], d["scales"],
                                                      d["zeros"], 4, 128, **kw)

    seen = _recorded(monkeypatch, "glq_gemm_lora", 16)
    _two_graphs(gpu, seen, [call(500), call(333)])
