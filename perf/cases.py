"""The work that stands for this framework's use, as cases that can be timed.

Shapes are the repository's own: the expert and attention projections of
Qwen1.5-MoE-A2.7B (hidden 2048, expert inter 1408, shared expert 5632, 60
experts, top-4), of a Qwen3-30B-A3B-shaped model (hidden 2048, expert inter
768, 128 experts, top-8, 32 query and 4 KV heads of 128) and of a
Mixtral-8x7B-shaped layer (hidden 4096, ffn 14336, 8 experts, top-2); 2- and
4-bit codes in groups of 128 and rank-64 low-rank factors; N(0, 1) fp16
activations.

kinds
  linear      GLoRCQLinear.forward, called as a module (one projection)
  moe_step    a decode step of GraphCompatibleMoeBlock (up to 64 tokens),
              captured once and replayed, as a decode loop runs it
  moe_prompt  GraphCompatibleMoeBlock.forward on a prompt, called as a module
  attention   kernels.decode_attention: one token a sequence over a KV cache
  model       GLoRCQGraphWrapper: prompt, then replayed decode steps

Every case is made from its seed on the GPU.  `exact` restates each kind but
`model` in 64 bits with plain torch.
"""

from __future__ import annotations

import math

import torch

from glorcq_amd import kernels
from glorcq_amd.format import LLOYD_MAX_2BIT, MoEProblem, QMat, TurboMat
from glorcq_amd.graph_wrapper import GLoRCQGraphWrapper
from glorcq_amd.hadamard_rotation import generate_rht_signs
from glorcq_amd.moe_block import GraphCompatibleMoeBlock
from glorcq_amd.quantized_linear import GLoRCQLinear

DEV = "cuda:0"
GROUP = 128
PROJS = ("gate", "up", "down")

# hidden, experts, inter, top_k, shared inter, renormalised weights
BLOCKS = {
    "qwen_moe": (2048, 60, 1408, 4, 5632, False),
    "qwen3_moe": (2048, 128, 768, 8, 0, True),
    "mixtral": (4096, 8, 14336, 2, 0, True),
}
# clusters of experts that share a U: usual, fewest and most drawn
CLUSTERS = {"qwen_moe": (16, 8, 48), "qwen3_moe": (64, 24, 100), "mixtral": (2, 1, 8)}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _linear(name, bits, K, N, M, rank=64, sym=False, bias=False):
    return {"name": name, "kind": "linear", "bits": bits, "K": K, "N": N, "M": M, "rank": rank,
            "sym": sym, "bias": bias}


def _moe(name, kind, block, tokens, quant="gptq", clusters=None):
    return {"name": name, "kind": kind, "block": block, "tokens": tokens, "quant": quant,
            "clusters": clusters or CLUSTERS[block][0]}


def _attention(name, seqs, length, max_len, heads=32, kv_heads=4):
    return {"name": name, "kind": "attention", "seqs": seqs, "length": length,
            "max_len": max_len, "heads": heads, "kv_heads": kv_heads}


def listed():
    return [
        # one expert projection for one token: the smallest call there is
        _linear("linear_one_token", 2, 2048, 1408, 1),
        # an attention projection for a small decode batch
        _linear("linear_batch", 4, 2048, 4096, 12),
        # an attention projection over a prompt of ragged length
        _linear("linear_prompt", 4, 2048, 4096, 777),
        # the block of a single user's decode step
        _moe("moe_one_token", "moe_step", "qwen_moe", 1),
        # the same block serving 32 users
        _moe("moe_batch", "moe_step", "qwen_moe", 32),
        # large experts, several tokens an expert
        _moe("mixtral_batch", "moe_step", "mixtral", 16),
        # a prompt through large experts (128 tokens an expert)
        _moe("mixtral_prompt", "moe_prompt", "mixtral", 512),
        # a long prompt of ragged length through many small experts
        _moe("qwen3_prompt", "moe_prompt", "qwen3_moe", 1500),
        # TurboQuant routed experts (the 2-bit expert format): a decode step
        _moe("turbo_batch", "moe_step", "qwen_moe", 4, "turbo"),
        # and a prompt
        _moe("turbo_prompt", "moe_prompt", "qwen_moe", 256, "turbo"),
        # attention of a decode step at 16 users with long contexts
        _attention("attention_long", 16, 4000, 4096),
        # the whole loop: a prompt, then decode steps under the graph
        {"name": "model", "kind": "model", "layers": 2, "vocab": 1024, "batch": 2, "prompt": 100,
         "steps": 24},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "moe_step", "moe_step", "moe_prompt",
                       "moe_prompt", "turbo", "attention", "model"])
    if kind == "linear":
        bits, K, N = rng.choice([
            (2, 2048, 1408), (2, 1408, 2048), (2, 2048, 768), (2, 768, 2048), (2, 4096, 14336),
            (2, 14336, 4096), (4, 2048, 2048), (4, 2048, 4096), (4, 4096, 2048), (4, 2048, 512),
            (4, 2048, 5632), (4, 5632, 2048)])
        c = _linear("", bits, K, N, _log_int(rng, 1, 2048), rng.choice([0, 32, 64, 64, 64, 128]),
                    rng.random() < 0.15, rng.random() < 0.25)
    elif kind == "moe_step":
        block = rng.choice(sorted(BLOCKS))
        c = _moe("", kind, block, _log_int(rng, 1, 64),
                 clusters=rng.randint(*CLUSTERS[block][1:]))
    elif kind == "moe_prompt":
        block = rng.choice(sorted(BLOCKS))
        c = _moe("", kind, block, _log_int(rng, 65, 1024 if block == "mixtral" else 2048),
                 clusters=rng.randint(*CLUSTERS[block][1:]))
    elif kind == "turbo":
        n = _log_int(rng, 1, 256)
        c = _moe("", "moe_step" if n <= 16 else "moe_prompt", "qwen_moe", n, "turbo",
                 rng.randint(*CLUSTERS["qwen_moe"][1:]))
    elif kind == "attention":
        n = _log_int(rng, 64, 8192)
        kv = rng.choice([2, 4, 8])
        c = _attention("", rng.randint(1, 16), n, (n + rng.randint(0, 600) + 7) // 8 * 8,
                       kv * rng.choice([4, 8]), kv)
    else:
        c = {"kind": "model", "layers": 2, "vocab": 1024, "batch": rng.randint(1, 4),
             "prompt": _log_int(rng, 16, 160), "steps": rng.randint(8, 24)}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).half()


def _scales(g, *shape):
    return (torch.randn(*shape, generator=g, device=DEV) * 0.02).abs().half()


def _linear_data(case, seed):
    g = _gen(seed)
    K, N, bits, r = case["K"], case["N"], case["bits"], case["rank"]
    half = 1 << (bits - 1)
    lo, hi = (-half, half) if case["sym"] else (0, 2 * half)
    d = {"q": torch.randint(lo, hi, (N, K), generator=g, device=DEV, dtype=torch.int32),
         "scales": _scales(g, N, K // GROUP), "zeros": None}
    if not case["sym"]:  # zero-points at the middle of the code range
        d["zeros"] = torch.randint(half - 1, half + 1, (N, K // GROUP), generator=g,
                                   device=DEV).half()
    d["U"] = _normal(g, K, r, std=0.01) if r else None
    d["SV"] = _normal(g, N, r, std=0.01) if r else None
    d["bias"] = _normal(g, N, std=0.1) if case["bias"] else None
    d["x"] = _normal(g, case["M"], K)
    return d


def _words(g, *shape):
    return torch.randint(-(2**31), 2**31, shape, generator=g, device=DEV,
                         dtype=torch.int64).to(torch.int32)


def _qmat(g, E, N, K, bits):
    half = 1 << (bits - 1)
    lo = 1 if bits == 2 else half - 1  # {1, 2} at 2 bits, {7, 8} at 4
    return QMat(codes=_words(g, E, N, K * bits // 32), scales=_scales(g, E, N, K // GROUP),
                zeros=torch.randint(lo, lo + 2, (E, N, K // GROUP), generator=g,
                                    device=DEV).half(), bits=bits, group=GROUP)


def _turbo_mats(g, E, H, I):
    """gate and up rotated by one Hadamard transform, down (its width is no
    power of two) by an orthogonal matrix."""
    signs = generate_rht_signs(H, 42).to(DEV)
    Q = torch.linalg.qr(torch.randn(I, I, generator=g, device=DEV))[0]
    mats = {}
    for proj, (K, N) in {"gate": (H, I), "up": (H, I), "down": (I, H)}.items():
        packed = torch.randint(0, 256, (E, N, K // 4), generator=g, device=DEV,
                               dtype=torch.int32).to(torch.uint8)
        mats[proj] = TurboMat(
            packed=packed, norms=torch.randn(E, N, generator=g, device=DEV).abs() * 0.5 + 0.5,
            centroids=torch.tensor(LLOYD_MAX_2BIT, device=DEV) / K ** 0.5,
            signs=None if proj == "down" else signs, Pi=Q.half() if proj == "down" else None)
    return mats


def _problem(case, seed):
    g = _gen(seed)
    H, E, I, k, S, norm = BLOCKS[case["block"]]
    C, r = case["clusters"], 64
    dims = {"gate": (H, I), "up": (H, I), "down": (I, H)}
    if case["quant"] == "turbo":
        experts = _turbo_mats(g, E, H, I)
    else:
        experts = {p: _qmat(g, E, dims[p][1], dims[p][0], 2) for p in PROJS}
    shared = None
    if S:
        shared = {p: _qmat(g, 1, n, m, 4)
                  for p, (m, n) in {"gate": (H, S), "up": (H, S), "down": (S, H)}.items()}
    return MoEProblem(
        H=H, E=E, inter=I, top_k=k, norm_topk_prob=norm, rank=r, n_clusters=C,
        router_w=_normal(g, E, H, std=0.02), shared_gate_w=_normal(g, 1, H, std=0.02),
        experts=experts, SV={p: _normal(g, E, dims[p][1], r, std=0.01) for p in PROJS},
        cluster_of={p: torch.randint(0, C, (E,), generator=g, device=DEV) for p in PROJS},
        U={p: _normal(g, C, dims[p][0], r, std=0.01) for p in PROJS}, shared=shared,
        h=_normal(g, case["tokens"], H))


def _attention_data(case, seed):
    g = _gen(seed)
    T, L, Hk = case["seqs"], case["max_len"], case["kv_heads"]
    return {"q": _normal(g, T, case["heads"], 128), "k": _normal(g, T, Hk, L, 128),
            "v": _normal(g, T, Hk, L, 128),
            "length": torch.full((1,), case["length"], dtype=torch.int32, device=DEV)}


_capture_stream = None


def _capture(step):
    """step() as a graph: warmed up and captured on one side stream."""
    global _capture_stream
    if _capture_stream is None:
        _capture_stream = torch.cuda.Stream()
    s = _capture_stream
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        outputs = step()
    return graph, outputs


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        d = _linear_data(case, seed)
        lin = GLoRCQLinear(case["K"], case["N"])
        lin.load_gptq({"qweight_int": d["q"], "scales": d["scales"], "zeros": d["zeros"],
                       "bits": case["bits"], "groupsize": GROUP, "sym": case["sym"]}, device=DEV)
        if case["rank"]:
            lin.load_sv(d["U"], d["SV"], device=DEV)
        if case["bias"]:
            lin.set_bias(d["bias"], device=DEV)
        return {"kind": kind, "layer": lin, "x": d["x"]}
    if kind == "attention":
        d = _attention_data(case, seed)
        return {"kind": kind, "args": d, "scale": 128 ** -0.5,
                "workspace": kernels.decode_attention_workspace(d["q"], d["k"])}
    if kind == "model":
        from glorcq_amd.synthetic_model import build_qwen3_moe, qwen3_moe_config

        model, _ = build_qwen3_moe(qwen3_moe_config(case["layers"], case["vocab"]), DEV,
                                   seed=seed)
        w = GLoRCQGraphWrapper(model, max_batch_size=case["batch"], max_seq_len=256)
        w.capture_graph()
        ids = torch.randint(0, case["vocab"], (case["batch"], case["prompt"] + case["steps"]),
                            generator=_gen(seed), device=DEV)
        return {"kind": kind, "wrapper": w, "ids": ids, "prompt": case["prompt"],
                "positions": torch.arange(case["prompt"], device=DEV)}
    p = _problem(case, seed)
    block = GraphCompatibleMoeBlock.from_problem(p, DEV)
    state = {"kind": kind, "block": block, "h": p.h}
    if kind == "moe_step":
        state["graph"], state["outputs"] = _capture(lambda: block(state["h"]))
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "moe_step":
        state["graph"].replay()
        return state["outputs"]
    if kind == "moe_prompt":
        return state["block"](state["h"])
    if kind == "attention":
        a = state["args"]
        return kernels.decode_attention(a["q"], a["k"], a["v"], a["length"], state["scale"],
                                        workspace=state["workspace"])
    # the prompt and the given tokens after it (a scored continuation)
    w, ids, n = state["wrapper"], state["ids"], state["prompt"]
    w.static_cache.reset()
    logits = [w.model(input_ids=ids[:, :n], cache_position=state["positions"],
                      past_key_values=w.static_cache, use_cache=True, return_dict=False)[0]]
    for pos in range(n, ids.shape[1]):
        logits.append(w.replay(ids[:, pos:pos + 1], pos).clone())
    return logits[0], torch.cat(logits[1:], dim=1)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _weight_bytes(N, K, bits):
    return N * K * bits / 8 + (4 * N * (K // GROUP) if bits else 0)


def _block_work(block, T, C, quant):
    H, E, I, k, S, _ = BLOCKS[block]
    r = 64
    active = E * (1 - (1 - k / E) ** T)
    clusters = C * (1 - (1 - 1 / C) ** active)
    bytes_ = 2 * E * H + 4 * T * H + 2 * T * E
    flops = 2 * T * E * H
    for N, K in ((I, H), (I, H), (H, I)):
        per = N * K / 4 + 4 * N if quant == "turbo" else _weight_bytes(N, K, 2)
        bytes_ += active * (per + 2 * r * N) + clusters * 2 * r * K
        flops += 2 * T * k * (N * K + r * (N + K))
        if S:
            n, m = (S if N == I else H), (H if K == H else S)
            bytes_ += _weight_bytes(n, m, 4)
            flops += 2 * T * n * m
    if quant == "turbo":
        bytes_ += 2 * I * I  # the down's rotation
        flops += 2 * T * k * I * I
    return bytes_, flops


def work(case):
    kind = case["kind"]
    if kind == "linear":
        K, N, M, r = case["K"], case["N"], case["M"], case["rank"]
        b = _weight_bytes(N, K, case["bits"]) + 2 * r * (K + N) + 2 * M * (K + N)
        if case["sym"]:
            b -= 2 * N * (K // GROUP)
        f = 2 * M * (N * K + r * (K + N))
    elif kind == "attention":
        T, L, Hq, Hk = case["seqs"], case["length"], case["heads"], case["kv_heads"]
        b = 2 * 2 * T * Hk * L * 128 + 2 * 2 * T * Hq * 128
        f = 2 * 2 * T * Hq * L * 128
    elif kind == "model":
        B, L, V, H, q, kv = case["batch"], case["layers"], case["vocab"], 2048, 4096, 512
        attn = sum(_weight_bytes(n, m, 4) + 128 * (n + m)
                   for n, m in ((q, H), (kv, H), (kv, H), (H, q)))
        b = f = 0
        for T, passes in ((B * case["prompt"], 1), (B, case["steps"])):
            mb, mf = _block_work("qwen3_moe", T, 64, "gptq")
            b += passes * (L * (mb + attn) + 2 * V * H + 2 * T * V)
            f += passes * (L * (mf + 2 * T * 2 * H * (q + kv)) + 2 * T * V * H)
    else:
        b, f = _block_work(case["block"], case["tokens"], case["clusters"], case["quant"])
    return {"bytes": b, "flops": f}


def tolerance(case):
    """fp16 results of fp32 sums: an output rounded the other way is off by
    2^-11 of its value, and so are the factors and activations that the path
    itself rounds to fp16 (x U, a SwiGLU product, a rotated input) before the
    next product.  About four times what sums in another order show: 1e-4
    for a projection; for a block 5e-4, its distance from the 64-bit result,
    most of which is its own fp16 roundings; 1e-3 for the model."""
    return {"linear": {"rel": 5e-4}, "attention": {"rel": 1e-3}, "moe_step": {"rel": 2e-3},
            "moe_prompt": {"rel": 2e-3}, "model": {"rel": 5e-3}}[case["kind"]]


# ---------------------------------------------------------------------------
# the results in 64 bits
# ---------------------------------------------------------------------------
def _unpack(words, bits):
    """(N, K bits / 32) int32 words -> (N, K) codes, low bits first."""
    shifts = torch.arange(0, 32, bits, device=words.device)
    w = words.to(torch.int64) & 0xFFFFFFFF
    return ((w.unsqueeze(-1) >> shifts) & ((1 << bits) - 1)).reshape(words.shape[0], -1)


def _dense(q, scales, zeros):
    n, K = q.shape
    w = q.double().reshape(n, K // GROUP, GROUP)
    if zeros is not None:
        w = w - zeros.double().unsqueeze(-1)
    return (w * scales.double().unsqueeze(-1)).reshape(n, K)


def _hadamard(d):
    m = torch.ones(1, 1, dtype=torch.float64, device=DEV)
    while m.shape[0] < d:
        m = torch.cat([torch.cat([m, m], 1), torch.cat([m, -m], 1)], 0)
    return m / d ** 0.5


def _silu(x):
    return x * torch.sigmoid(x)


def _exact_block(case, seed):
    p = _problem(case, seed)
    h = p.h.double()
    logits = h @ p.router_w.double().T
    # the router picks on logits rounded to fp16, ties to the lower index
    order = torch.sort(logits.half(), dim=1, descending=True, stable=True)[1][:, :p.top_k]
    weights = torch.softmax(logits.half().double(), dim=1).gather(1, order)
    if p.norm_topk_prob:
        weights = weights / weights.sum(1, keepdim=True)

    def rotation(m):  # x -> x R
        if m.Pi is not None:
            return m.Pi.double().T
        return m.signs.double().unsqueeze(1) * _hadamard(m.K)

    turbo = case["quant"] == "turbo"
    rots = {q: rotation(p.experts[q]) for q in ("gate", "down")} if turbo else {}
    if turbo:
        rots["up"] = rots["gate"]

    def project(proj, e, x):
        m = p.experts[proj]
        if turbo:
            codes = _unpack(m.words()[e], 2)
            W = m.centroids.double()[codes] * m.norms[e].double().unsqueeze(1)
            y = (x @ rots[proj]) @ W.T
        else:
            y = x @ _dense(_unpack(m.codes[e], m.bits), m.scales[e], m.zeros[e]).T
        return y + (x @ p.U[proj][p.cluster_of[proj][e]].double()) @ p.SV[proj][e].double().T

    out = torch.zeros_like(h)
    for e in range(p.E):
        tok, slot = torch.where(order == e)
        if tok.numel():
            x = h[tok]
            y = project("down", e, _silu(project("gate", e, x)) * project("up", e, x))
            out.index_add_(0, tok, y * weights[tok, slot].unsqueeze(1))
    if p.shared is not None:
        W = {q: _dense(_unpack(s.codes[0], s.bits), s.scales[0], s.zeros[0])
             for q, s in p.shared.items()}
        y = (_silu(h @ W["gate"].T) * (h @ W["up"].T)) @ W["down"].T
        out += torch.sigmoid(h @ p.shared_gate_w.double().T) * y
    return out, logits


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "model":  # its tokens' experts follow from rounded activations
        return None
    if kind == "linear":
        d = _linear_data(case, seed)
        x = d["x"].double()
        y = x @ _dense(d["q"], d["scales"], d["zeros"]).T
        if case["rank"]:
            y = y + (x @ d["U"].double()) @ d["SV"].double().T
        return y if d["bias"] is None else y + d["bias"].double()
    if kind == "attention":
        d = _attention_data(case, seed)
        T, L, Hk = case["seqs"], case["length"], case["kv_heads"]
        q = d["q"].double().reshape(T, Hk, -1, 128)
        rows = []
        for t in range(T):
            s = q[t] @ d["k"][t, :, :L].double().transpose(1, 2).contiguous() * 128 ** -0.5
            rows.append((torch.softmax(s, dim=-1) @ d["v"][t, :, :L].double()).reshape(-1))
        return torch.stack(rows)
    return _exact_block(case, seed)
