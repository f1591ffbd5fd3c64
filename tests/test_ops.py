"""The torch.library operator layer (glorcq_amd.ops, namespace glorcq_hip): the
counterpart of the reference's custom ops with fake kernels
(inference/kernels/__init__.py:63-107).

CPU: every operator is registered, its fake kernel gives the real kernel's
output shape and dtype on meta tensors, torch.library.opcheck passes its schema,
fake-tensor and AOT-dispatch checks there, and Dynamo traces a GLoRCQLinear
and a MoE block into one graph (fullgraph) under fake tensors.
GPU (tests marked gpu): opcheck on device tensors (fake vs real outputs), and
torch.compile(fullgraph=True) of GLoRCQLinear.forward and of the MoE block
equals eager, bit for bit."""

import pytest
import torch
from torch.library import opcheck

import glorcq_amd  # noqa: F401  (registers the operators)
from glorcq_amd import format as fmt
from glorcq_amd.moe_block import GraphCompatibleMoeBlock
from glorcq_amd.quantized_linear import GLoRCQLinear

OPS = ["packed_dequant_matmul", "turbo_dequant_matmul", "lowrank_xu", "rht", "moe_decode",
       "moe_prefill"]


def meta(*shape, dtype=torch.float16):
    return torch.empty(*shape, dtype=dtype, device="meta")


def gptq_args(M=4, K=2048, N=1408, r=64, dev="meta"):
    mk = (lambda *s, dtype=torch.float16: torch.empty(*s, dtype=dtype, device=dev))
    return (mk(M, K), mk(N, K // 16, dtype=torch.int32), mk(N, K // 128), mk(N, K // 128), 2,
            128, False, mk(K, r), mk(N, r), None, None)


def test_operators_registered():
    for name in OPS:
        assert hasattr(torch.ops.glorcq_hip, name), name


def test_fake_kernels_on_meta():
    y = torch.ops.glorcq_hip.packed_dequant_matmul(*gptq_args())
    assert y.shape == (4, 1408) and y.dtype == torch.float16
    t = torch.ops.glorcq_hip.turbo_dequant_matmul(meta(3, 1024), meta(512, 256, dtype=torch.uint8),
                                                  meta(512, dtype=torch.float32),
                                                  meta(4, dtype=torch.float32), None, None, None)
    assert t.shape == (3, 512)
    a = torch.ops.glorcq_hip.lowrank_xu(meta(5, 2048), meta(3, 2048, 64))
    assert a.shape == (3, 5, 64)
    r = torch.ops.glorcq_hip.rht(meta(2, 256), meta(256, dtype=torch.float32), False, True)
    assert r.shape == (2, 256) and r.dtype == torch.float32
    with pytest.raises(RuntimeError, match="does not match K"):
        torch.ops.glorcq_hip.packed_dequant_matmul(meta(4, 1024), *gptq_args()[1:])


def test_opcheck_on_meta():
    r = opcheck(torch.ops.glorcq_hip.packed_dequant_matmul.default, gptq_args())
    assert all(v == "SUCCESS" for v in r.values()), r
    r = opcheck(torch.ops.glorcq_hip.lowrank_xu.default, (meta(5, 2048), meta(2048, 64)))
    assert all(v == "SUCCESS" for v in r.values()), r


def linear(dev, M=3, seed=11):
    p = fmt.make_linear(2048, 1408, bits=2, rank=64, M=M, seed=seed)
    from oracle import glorcq_oracle as O
    lin = GLoRCQLinear(2048, 1408)
    lin.load_gptq({"qweight_int": torch.from_numpy(O.unpack_codes(p.codes.numpy(), 2, 2048)),
                   "scales": p.scales, "zeros": p.zeros, "bits": 2, "groupsize": 128},
                  device=dev)
    lin.load_sv(p.U, p.SV, device=dev)
    return lin, p.x.to(dev)


def test_dynamo_traces_linear_fullgraph_on_fake_tensors():
    """Dynamo + AOT (aot_eager) trace GLoRCQLinear.forward into one graph with
    the fake kernel standing in (no device code runs: the weights are CPU
    tensors faked as their GPU shapes by the traced op)."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    lin, x = linear("cpu")
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        fx = mode.from_tensor(x)
        lin.codes, lin.scales, lin.zeros, lin.U, lin.SV = (
            mode.from_tensor(t) for t in (lin.codes, lin.scales, lin.zeros, lin.U, lin.SV))
        gm, guards = torch._dynamo.export(lin.forward)(fx)
    names = [n.target for n in gm.graph.nodes if n.op == "call_function"]
    assert torch.ops.glorcq_hip.packed_dequant_matmul.default in names or \
        torch.ops.glorcq_hip.packed_dequant_matmul in names, names


# ------------------------------------------------------------------ GPU ----
@pytest.mark.gpu
def test_opcheck_real_vs_fake(gpu):
    lin, x = linear(gpu)
    args = (x, lin.codes, lin.scales, lin.zeros, 2, 128, False, lin.U, lin.SV, None, None)
    r = opcheck(torch.ops.glorcq_hip.packed_dequant_matmul.default, args)
    assert all(v == "SUCCESS" for v in r.values()), r


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 5, 40])
def test_compile_linear_fullgraph_equals_eager(gpu, M):
    lin, x = linear(gpu, M=M, seed=12 + M)
    eager = lin(x)
    torch._dynamo.reset()
    compiled = torch.compile(lin.forward, fullgraph=True, backend="aot_eager")
    got = compiled(x)
    torch.cuda.synchronize()
    assert torch.equal(got, eager)


@pytest.mark.gpu
def test_compile_moe_block_fullgraph_equals_eager(gpu):
    p = fmt.make_moe(H=256, E=8, inter=384, top_k=2, n_clusters=3, rank=16, shared_inter=512,
                     B=4, seed=5)
    blk = GraphCompatibleMoeBlock.from_problem(p, gpu)
    h = p.h.reshape(1, 4, p.H).to(gpu)
    eager, el = blk(h)
    torch._dynamo.reset()
    compiled = torch.compile(blk.forward, fullgraph=True, backend="aot_eager")
    got, gl = compiled(h)
    torch.cuda.synchronize()
    assert torch.equal(got, eager) and torch.equal(gl, el)


@pytest.mark.gpu
def test_direct_call_where_the_dispatch_adds_nothing(gpu):
    """packed_dequant_matmul_fused calls the library directly for plain tensors
    and goes through the operator wherever something watches or transforms the
    call: a dispatch mode sees it, vmap and forward-mode levels and recorded
    gradients get the operator's own answer."""
    from torch.utils._python_dispatch import TorchDispatchMode

    from glorcq_amd import kernels as K_

    p = fmt.make_linear(2048, 256, bits=2, rank=16, M=3, seed=8)
    t = {k: getattr(p, k).to(gpu) for k in ("x", "codes", "scales", "zeros", "U", "SV")}

    def call(x):
        return K_.packed_dequant_matmul_fused(x, t["codes"], t["scales"], t["zeros"], 2, 128,
                                              U=t["U"], SV=t["SV"])

    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    y = call(t["x"])
    assert K_._plain(*t.values())
    with Watch():
        assert torch.equal(call(t["x"]), y)
    assert any("packed_dequant_matmul" in s for s in seen)
    xg = t["x"].clone().requires_grad_()
    assert not K_._plain(xg)
    yg = call(xg)
    assert yg.requires_grad and torch.equal(yg.detach(), y)
    with pytest.raises(Exception):
        yg.sum().backward()  # no gradient formula, as through the operator
    with torch.no_grad():
        assert K_._plain(xg) and torch.equal(call(xg), y)
    assert torch.equal(torch.vmap(call)(torch.stack([t["x"], t["x"]])), torch.stack([y, y]))
    with torch.autograd.forward_ad.dual_level():
        assert not K_._plain(t["x"])
    assert not K_._plain(p.x)  # a CPU tensor


@pytest.mark.parametrize("T,top_k,E,hidden,prompt", [
    (16, 8, 8, 2048, False), (17, 2, 8, 2048, True), (17, 4, 60, 2048, False),
    (33, 4, 60, 2048, True), (64, 8, 128, 2048, True),
    (33, 16, 128, 2048, False), (64, 4, 60, 384, False),  # the step refuses these
    (65, 16, 128, 384, True),
])
def test_moe_batches_that_run_as_a_prompt(T, top_k, E, hidden, prompt):
    """The rule that sends a batch to glq_moe_prefill leaves what the decode
    step refuses (more than 512 picks, a hidden width not of 256s) to it."""
    from types import SimpleNamespace

    from glorcq_amd.moe_block import GraphCompatibleMoeBlock as B
    blk = SimpleNamespace(MAX_TOKENS=B.MAX_TOKENS, top_k=top_k, num_experts=E, hidden=hidden,
                          zeros_integral=True, rank=64)
    assert B._as_prompt(blk, T) is prompt


@pytest.mark.gpu
def test_profiler_sees_the_operator(gpu):
    """With a profiler active the call goes through the operator, so that it is
    recorded under its name."""
    from glorcq_amd import kernels as K_

    p = fmt.make_linear(2048, 256, bits=2, rank=16, M=3, seed=8)
    t = {k: getattr(p, k).to(gpu) for k in ("x", "codes", "scales", "zeros", "U", "SV")}
    assert K_._plain(*t.values())
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        assert not K_._plain(*t.values())
        K_.packed_dequant_matmul_fused(t["x"], t["codes"], t["scales"], t["zeros"], 2, 128,
                                       U=t["U"], SV=t["SV"])
    assert K_._plain(*t.values())
    assert "glorcq_hip::packed_dequant_matmul" in {e.key for e in prof.key_averages()}


@pytest.mark.gpu
def test_what_the_dispatch_resolves_or_refuses_first(gpu):
    """A lazily negated activation gives its own values' result, and names and
    sizes that are not integers are refused, as by the operator."""
    from glorcq_amd import kernels as K_

    p = fmt.make_linear(2048, 256, bits=2, rank=16, M=3, seed=8)
    t = {k: getattr(p, k).to(gpu) for k in ("x", "codes", "scales", "zeros", "U", "SV")}

    def call(x, bits=2, group=128, **kw):
        return K_.packed_dequant_matmul_fused(x, t["codes"], t["scales"], t["zeros"], bits, group,
                                              U=t["U"], SV=kw.get("SV", t["SV"]))

    neg = torch._neg_view(t["x"])  # as conj().imag is
    assert neg.is_neg() and torch.equal(call(neg), call((-t["x"]).contiguous()))
    assert torch.equal(call(t["x"], SV=torch._neg_view(t["SV"])), call(t["x"], SV=-t["SV"]))
    for bad in (lambda: call(t["x"].rename("a", "b")), lambda: call(t["x"], bits=2.0),
                lambda: call(t["x"], group=128.0)):
        with pytest.raises(RuntimeError):
            bad()


@pytest.mark.parametrize("block,T,pays", [
    # hidden, inter, experts, top_k, shared inter, bits, shared bits: step / prompt us
    ((2048, 1408, 60, 4, 5632, 2, 4), 32, True),    # 139 / 116
    ((2048, 768, 128, 8, 0, 2, 4), 32, True),       # 138 / 134
    ((4096, 14336, 8, 2, 0, 2, 4), 17, True),       # 437 / 240
    ((2048, 512, 256, 1, 0, 2, 4), 33, True),       # 195 / 96
    ((2048, 768, 4, 1, 0, 2, 4), 17, False),        # 44 / 58
    ((2048, 768, 2, 1, 1536, 4, 4), 17, False),     # 45 / 82
    ((2048, 768, 2, 1, 1536, 4, 4), 48, False),     # 72 / 94
    ((1024, 1024, 16, 2, 2048, 4, 4), 17, False),   # 58 / 73
    ((512, 512, 8, 2, 512, 2, 4), 20, False),       # 36 / 44
    ((5376, 128, 4, 2, 0, 2, 4), 17, True),         # the step refuses it (LDS)
])
def test_moe_batches_that_a_prompt_serves_faster(block, T, pays):
    from types import SimpleNamespace

    from glorcq_amd.moe_block import GraphCompatibleMoeBlock as B
    H, inter, E, k, S, bits, sbits = block
    blk = SimpleNamespace(hidden=H, inter=inter, num_experts=E, top_k=k, shared_inter=S,
                          bits=bits, shared_bits=sbits)
    assert B._prompt_pays(blk, T) is pays


@pytest.mark.gpu
@pytest.mark.parametrize("H,inter,S", [(5376, 128, 0), (4096, 256, 256), (2048, 128, 128)])
def test_moe_batches_of_wide_blocks_run(gpu, H, inter, S):
    """Batches of 17 to 64 tokens run whether or not the step takes the block's
    width."""
    p = fmt.make_moe(H=H, E=4, inter=inter, top_k=2, n_clusters=2, rank=16, shared_inter=S, B=65)
    blk = GraphCompatibleMoeBlock.from_problem(p, gpu)
    h = p.h.reshape(1, 65, p.H).to(gpu)
    ref = blk(h)[0]
    for T in (17, 33, 64):
        # (fp16 roundings of x U, the SwiGLU product and the output, sums in another order)
        err = (blk(h[:, :T])[0].float() - ref[:, :T].float()).abs()
        assert bool((err <= 2e-3 + 1e-2 * ref[:, :T].float().abs()).all()), float(err.max())
