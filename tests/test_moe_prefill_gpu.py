"""MoE block over many tokens (glq_moe_prefill via GraphCompatibleMoeBlock with
more than 64 tokens): grouped dequant GEMMs over each active expert's gathered
tokens, the reference's _forward_sparse (inference/moe_block.py:704-740),
against the MoE oracle (oracle.moe_forward, pinned by
tests/test_moe_oracle_library.py against transformers' sparse MoE blocks).

Bars as tests/test_moe_gpu.py: routing ids identical (seeds with no near-tie
at the top-k boundary, asserted), router logits within one fp16 ulp, block
output within the MoE bar (atol 1e-3 + rtol 1e-2 |ref| + 2e-3 * row max)."""

import pytest
import torch

from glorcq_amd import format as fmt
from glorcq_amd.moe_block import GraphCompatibleMoeBlock
from oracle import glorcq_oracle as O
from test_moe_gpu import check_routing, margin
from test_moe_oracle import bar, lora_heavy

pytestmark = pytest.mark.gpu


def run(p, gpu, residual=None):
    blk = GraphCompatibleMoeBlock.from_problem(p, gpu)
    res = None if residual is None else residual.reshape(1, p.B, p.H).to(gpu)
    out, logits = blk(p.h.reshape(1, p.B, p.H).to(gpu), residual=res)
    torch.cuda.synchronize()
    return blk, out.reshape(p.B, p.H).cpu(), logits.cpu()


def check(p, out, logits, what):
    check_routing(p, logits)
    ref = O.moe_forward(p)
    assert bar(out, ref), (what, float((out.double() - ref).abs().max()))


def test_config3_prefill_512(gpu):
    """BASELINE config 3's prefill: a Mixtral-8x7B-shaped layer over 512 tokens
    (about 128 tokens per expert: 64-token tiles), LoRA factors x3."""
    p = lora_heavy(fmt.make_mixtral_layer(B=512, seed=42), f=3.0)
    assert margin(p) >= 2
    print("config 3 prefill T=512", flush=True)
    _, out, logits = run(p, gpu)
    check(p, out, logits, "config 3 T=512")


def test_config2_prefill(gpu):
    """A Qwen1.5-MoE-A2.7B block (60 experts, top-4, 16 clusters, 4-bit shared
    expert behind its sigmoid gate) over 80 tokens (32-token tiles)."""
    p = fmt.make_moe(B=80, seed=82)
    assert margin(p) >= 2
    _, out, logits = run(p, gpu)
    check(p, out, logits, "config 2 T=80")


@pytest.mark.parametrize("kw", [
    dict(),
    dict(norm_topk_prob=True),
    dict(rank=0),
    dict(bits=4),
    dict(shared_bits=2),
    dict(shared_inter=0),
    dict(n_clusters=1),
], ids=lambda kw: ",".join(f"{k}={v}" for k, v in kw.items()) or "base")
def test_prefill_variants(gpu, kw):
    """A small block (H 256, 8 experts, inter 384, top-2, 3 clusters, rank 16)
    over 200 tokens (64-token tiles), LoRA x30 where it has a rank."""
    args = dict(H=256, E=8, inter=384, top_k=2, n_clusters=3, rank=16, shared_inter=512)
    args.update(kw)
    # the first seed from 10 whose routing has no near-tie (routing only: cheap)
    seed = next(s for s in range(10, 60) if margin(fmt.make_moe(B=200, seed=s, **args)) >= 2)
    p = fmt.make_moe(B=200, seed=seed, **args)
    if p.rank:
        p = lora_heavy(p)
    _, out, logits = run(p, gpu)
    check(p, out, logits, str(kw))


def test_prefill_residual_and_tiles(gpu, monkeypatch):
    """The residual add is fused into the combine; every token tile size gives
    the same bits (rows are independent)."""
    p = lora_heavy(fmt.make_moe(H=256, E=8, inter=384, top_k=2, n_clusters=3, rank=16,
                                shared_inter=512, B=200, seed=10))
    res = (torch.randn(200, 256, generator=torch.Generator().manual_seed(3)) * 0.5).half()
    outs = []
    for tm in ("32", "64", "128"):
        monkeypatch.setenv("GLQ_PF_MOE_TM", tm)
        _, out, _ = run(p, gpu, residual=res)
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    ref = (O.moe_forward(p).half().double() + res.double())
    assert bar(outs[0], ref)


def test_prefill_matches_decode_steps(gpu):
    """The same 72 tokens as one prefill and as decode steps of 36: both within
    the bar of the oracle and of each other (different kernels, same math)."""
    p = lora_heavy(fmt.make_moe(H=256, E=8, inter=384, top_k=2, n_clusters=3, rank=16,
                                shared_inter=512, B=72, seed=10))
    blk, out, logits = run(p, gpu)
    h = p.h.to(gpu)
    d0, l0 = blk(h[:36].reshape(1, 36, p.H))
    d1, l1 = blk(h[36:].reshape(1, 36, p.H))
    torch.cuda.synchronize()
    dec = torch.cat([d0.reshape(36, p.H), d1.reshape(36, p.H)]).cpu()
    assert bar(out, dec.double())
    assert torch.equal(torch.cat([l0, l1]).cpu(), logits) or \
        float((torch.cat([l0, l1]).cpu().float() - logits.float()).abs().max()) < 1e-2


def test_non_integer_zeros_use_decode_steps(gpu):
    """Zero-points that are not integers (the prefill GEMMs take integer ones)
    run as 64-token decode steps: still within the bar."""
    p = fmt.make_moe(H=256, E=8, inter=384, top_k=2, n_clusters=3, rank=16, shared_inter=512,
                     B=100, seed=10)
    g = torch.Generator().manual_seed(9)
    for proj in fmt.PROJS:
        z = p.experts[proj].zeros.float()
        p.experts[proj].zeros = (z + torch.rand(z.shape, generator=g) * 0.5).half()
    assert margin(p) >= 2
    blk = GraphCompatibleMoeBlock.from_problem(p, gpu)
    assert not blk.zeros_integral
    out, logits = blk(p.h.reshape(1, 100, p.H).to(gpu))
    torch.cuda.synchronize()
    check(p, out.reshape(100, p.H).cpu(), logits.cpu(), "non-integer zeros")


def test_non_integer_shared_zeros_use_decode_steps(gpu):
    """Non-integer zero-points on the shared expert only (the routed ones stay
    integers): the block still takes decode steps, since the prefill GEMMs
    use round(z) for the shared expert too, and stays within the bar."""
    p = fmt.make_moe(H=256, E=8, inter=384, top_k=2, n_clusters=3, rank=16, shared_inter=512,
                     B=100, seed=10)
    g = torch.Generator().manual_seed(11)
    for proj in fmt.PROJS:
        z = p.shared[proj].zeros.float()
        p.shared[proj].zeros = (z + 0.25 + torch.rand(z.shape, generator=g) * 0.5).half()
    assert margin(p) >= 2
    blk = GraphCompatibleMoeBlock.from_problem(p, gpu)
    assert not blk.zeros_integral
    out, logits = blk(p.h.reshape(1, 100, p.H).to(gpu))
    torch.cuda.synchronize()
    check(p, out.reshape(100, p.H).cpu(), logits.cpu(), "non-integer shared zeros")


@pytest.mark.parametrize("T,E,top_k,H,inter,bits", [
    (65, 8, 2, 512, 1024, 2),    # 16 tokens an expert: 32-token tiles, scale pairs
    (65, 1, 1, 128, 128, 2),     # one expert, one group, one row block
    (129, 4, 2, 512, 640, 4),    # 64 an expert (64-token tiles), 8 and 5 groups, 4-bit
    (160, 4, 2, 1280, 512, 2),   # 80 an expert (128-token tiles), 10 and 4 groups
    (257, 2, 2, 640, 1024, 2),   # 257 rows on every expert: five 64-token tiles, one row over
], ids=str)
def test_prefill_tile_edges(gpu, T, E, top_k, H, inter, bits):
    """The tile form's token tiles (by the mean tokens an expert gets) at their
    edges: ragged last tiles, groups loaded one and two at a time, row blocks
    past the projection's rows."""
    args = dict(H=H, E=E, inter=inter, top_k=top_k, n_clusters=2, rank=24, shared_inter=256,
                bits=bits)
    seed = 10
    if E > top_k:  # the first seed whose routing has no near-tie
        seed = next(s for s in range(10, 60) if margin(fmt.make_moe(B=T, seed=s, **args)) >= 2)
    p = lora_heavy(fmt.make_moe(B=T, seed=seed, **args))
    _, out, logits = run(p, gpu)
    check(p, out, logits, str((T, E, top_k, H, inter, bits)))


@pytest.mark.parametrize("T,E,top_k,kw", [
    (17, 8, 2, {}),                        # from 16 tokens: two picks an expert
    (32, 40, 4, dict(shared_inter=1152)),  # the shared expert in the routed launches, 9 groups
    (33, 16, 1, dict(shared_bits=2)),      # past 32 tokens; 2-bit shared weights: own launches
    (64, 4, 2, dict(inter=2304, shared_inter=0)),  # routed down in K splits (18 groups)
], ids=str)
def test_large_decode_batches(gpu, T, E, top_k, kw):
    """17 to 64 tokens where they run as a prompt: against the oracle, the same
    bits on graph replays with eager work between them (the low-rank counters
    are cleared by every call)."""
    args = dict(H=512, E=E, inter=640, top_k=top_k, n_clusters=3, rank=40, shared_inter=512)
    args.update(kw)
    seed = next(s for s in range(10, 80) if margin(fmt.make_moe(B=T, seed=s, **args)) >= 2)
    p = lora_heavy(fmt.make_moe(B=T, seed=seed, **args))
    blk = GraphCompatibleMoeBlock.from_problem(p, gpu)
    assert blk._as_prompt(T)
    blk._prompt_pays = lambda T: True  # (small blocks: the step is the faster)
    h = p.h.reshape(1, T, p.H).to(gpu)
    out, logits = blk(h)
    torch.cuda.synchronize()
    check(p, out.reshape(T, p.H).cpu(), logits.cpu(), str((T, E, kw)))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        blk(h)
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        gout, glog = blk(h)
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(gout, out) and torch.equal(glog, logits)
        assert torch.equal(blk(h)[0], out)


@pytest.mark.parametrize("T", [8, 20, 65])
@pytest.mark.parametrize("pool", [False, True])
def test_cluster_ids_are_clamped(gpu, T, pool):
    """Cluster ids past the U pool read its last row (negative ones its first),
    in a decode step, in a batch that runs as a prompt and in a prompt; also
    through the rows of a cross-layer pool."""
    p = lora_heavy(fmt.make_moe(H=512, E=6, inter=256, top_k=2, n_clusters=3, rank=16,
                                shared_inter=0, B=T, seed=4))
    ids = torch.tensor([0, 7, -2, 2, 1, 3])
    outs = []
    for cl in (ids, ids.clamp(0, 2)):
        p.cluster_of = {proj: cl for proj in fmt.PROJS}
        blk = GraphCompatibleMoeBlock.from_problem(p, gpu)
        if pool:  # rows 4, 1, 2 of five hold the clusters; down's ids are rows
            slot = torch.tensor([4, 1, 2], dtype=torch.int32, device=gpu)
            for proj in fmt.PROJS:
                U = blk.t[f"U_{proj}"]
                big = torch.full((5, *U.shape[1:]), float("nan"), dtype=U.dtype, device=gpu)
                big[slot.long()] = U
                blk.t[f"U_{proj}"], blk.t[f"urows_{proj}"] = big, 5
            blk.t["uslot_gate"] = blk.t["uslot_up"] = slot
            blk.t["cluster_down"] = slot[ids.clamp(0, 2).to(gpu)].contiguous()
        blk._prompt_pays = lambda T: True
        outs.append(blk(p.h.reshape(1, T, p.H).to(gpu))[0])
    torch.cuda.synchronize()
    assert not bool(outs[0].isnan().any()) and torch.equal(*outs)
    check(p, outs[1].reshape(T, p.H).cpu(), blk(p.h.reshape(1, T, p.H).to(gpu))[1].cpu(), str(T))
