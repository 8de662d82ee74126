"""The work that is timed when this framework is measured: its paths through the public entry points, over the
sizes that a speculative-decoding server runs them at.

``kind`` of a case:
  block    one whole MoE block, router -> dispatch -> experts -> combine (``ops.MoeForwardPlan``)
  stack    the layers of a model as one call (``MoEOnlyStack.forward``)
  engine   layers through the calls an engine loop makes: RMSNorm, ``route_experts``, placement, ``forward_moe``
  attend   one layer's attention step: KV-cache store, then the paged (decode / verify) or packed (prefill) attention
  load     quantise-on-load of experts from a checkpoint's bf16 weights (``W4ExpertBank.load_expert``)
Model shapes are those of ``on_device_sd_amd.workloads.CONFIGS``; the attention cases use the heads of Qwen3-30B-A3B
(32 query / 4 KV heads of 128) and, when drawn, the other head layouts that the tests cover.
"""
from __future__ import annotations

import dataclasses
import math
import random

import torch

import on_device_sd_amd as odsd
from on_device_sd_amd import ops
from on_device_sd_amd.workloads import CONFIGS, LayerInputs

DEV = "cuda"
# Size of the residual stream that runs through several layers.  In a trained model it is much larger than what one
# layer adds; at 1 a stack of random layers is chaotic (a changed expert choice at a near-tie moves the token by 5 %,
# which changes further choices: two summation orders differ by 9 % after 48 layers, at 8 by about 0.5 %).
RESIDUAL_SCALE = 8.0
# model -> the configuration whose shape, dtype and top-k rule it has
MODELS = {"tiny": "tiny", "mixtral": "mixtral_t5", "qwen3_30b": "qwen3_30b_stack48_t256", "qwen3_235b": "qwen3_235b_t4096"}


def _workload(case, seed=0):
    wl = CONFIGS[MODELS[case["model"]]]
    return dataclasses.replace(wl, T=case["T"], layers=case.get("layers", 1), seed=1000 * seed,
                               zipf_s=1.1 if case.get("skew") else None)


def listed():
    return [
        # the smallest block, fp32 activations: nothing but launches and latency
        {"name": "block_tiny_f32_t32", "kind": "block", "model": "tiny", "T": 32, "skew": False},
        # one sequence's verify step (5 draft tokens) on a model with few large experts
        {"name": "block_mixtral_t5", "kind": "block", "model": "mixtral", "T": 5, "skew": False},
        # a batch of 32 such sequences
        {"name": "block_mixtral_t160", "kind": "block", "model": "mixtral", "T": 160, "skew": False},
        # a verify step on a model with many small experts, popularity of the experts falling as a power law
        {"name": "block_qwen3_30b_t64_zipf", "kind": "block", "model": "qwen3_30b", "T": 64, "skew": True},
        # a chunk of a prompt, an odd number of tokens: between verify and prefill sizes
        {"name": "block_qwen3_30b_t1000", "kind": "block", "model": "qwen3_30b", "T": 1000, "skew": False},
        # a whole prompt: the largest single call
        {"name": "block_qwen3_235b_t4096", "kind": "block", "model": "qwen3_235b", "T": 4096, "skew": False},
        # all 48 layers of a verify step for a full batch
        {"name": "stack_qwen3_30b_t256", "kind": "stack", "model": "qwen3_30b", "T": 256, "layers": 48, "skew": False},
        # the engine loop's separate calls, a small batch: the host's share of a step
        {"name": "engine_qwen3_30b_t24", "kind": "engine", "model": "qwen3_30b", "T": 24, "layers": 4, "skew": False},
        # verify attention: 32 sequences, 8 draft tokens each, up to 2048 cached tokens
        {"name": "attend_verify_s32_q8", "kind": "attend", "form": "verify", "seqs": 32, "q_len": 8, "ctx": 2048,
         "heads": 32, "kv_heads": 4, "head_dim": 128, "block": 256, "dtype": "bf16"},
        # decode attention: one token each of 64 sequences of mixed lengths
        {"name": "attend_decode_s64", "kind": "attend", "form": "decode", "seqs": 64, "q_len": 1, "ctx": 3000,
         "heads": 32, "kv_heads": 4, "head_dim": 128, "block": 256, "dtype": "bf16"},
        # prefill attention: three prompts packed one after the other
        {"name": "attend_prefill_s3", "kind": "attend", "form": "prefill", "seqs": 3, "q_len": 0, "ctx": 3000,
         "heads": 32, "kv_heads": 4, "head_dim": 128, "block": 256, "dtype": "bf16"},
        # experts that a cache miss or a model load brings in
        {"name": "load_qwen3_30b_e16", "kind": "load", "model": "qwen3_30b", "experts": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "block", "stack", "engine", "attend", "attend", "attend", "load"])
    if kind == "block":
        model = rng.choice(["tiny", "mixtral", "qwen3_30b", "qwen3_30b", "qwen3_235b"])
        most = {"tiny": 512, "mixtral": 2048, "qwen3_30b": 4096, "qwen3_235b": 4096}[model]
        return {"kind": kind, "model": model, "T": _log_int(rng, 1, most), "skew": model == "qwen3_30b" and rng.random() < 0.3}
    if kind == "stack":
        return {"kind": kind, "model": "qwen3_30b", "T": _log_int(rng, 4, 256), "layers": rng.randint(2, 40), "skew": rng.random() < 0.2}
    if kind == "engine":
        return {"kind": kind, "model": "qwen3_30b", "T": _log_int(rng, 1, 256), "layers": rng.randint(1, 6), "skew": False}
    if kind == "load":
        return {"kind": kind, "model": rng.choice(["qwen3_30b", "qwen3_235b"]), "experts": _log_int(rng, 1, 16)}
    form = rng.choice(["verify", "decode", "prefill"])
    heads, kv_heads, head_dim = rng.choice([(32, 4, 128), (32, 4, 128), (32, 8, 128), (16, 2, 128), (16, 8, 64)])
    c = {"kind": kind, "form": form, "seqs": _log_int(rng, 1, 64), "q_len": 1, "ctx": _log_int(rng, 40, 4000),
         "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "block": rng.choice([16, 64, 256, 256]),
         "dtype": rng.choice(["bf16", "bf16", "f16"])}
    if form == "verify":
        c["q_len"] = rng.randint(2, 12)
    elif form == "prefill":
        c["seqs"], c["q_len"] = rng.randint(1, 4), 0
    return c


def _active(case):
    """Experts with at least one token, for uniform routing: what a call has to read of the weights."""
    wl = _workload(case)
    return wl.E * (1.0 - (1.0 - wl.K / wl.E) ** wl.T)


def _lengths(case):
    """(cached tokens, query tokens) of each sequence: mixed lengths, a quarter of the longest and up; the first is the longest."""
    r = random.Random(case["ctx"] * 1000 + case["seqs"])
    out = []
    for i in range(case["seqs"]):
        n = case["ctx"] if i == 0 else max(1, int(case["ctx"] * r.uniform(0.25, 1.0)))
        q = n if case["form"] == "prefill" else case["q_len"]
        out.append((max(n, q), q))
    return out


def work(case):
    if case["kind"] == "load":
        wl = CONFIGS[MODELS[case["model"]]]
        n = case["experts"] * wl.H * wl.I
        return {"bytes": n * (3 * 2 + 1.59375), "flops": 0.0}
    if case["kind"] == "attend":
        ls, hd = _lengths(case), case["head_dim"]
        toks = sum(q for _, q in ls)
        kv = sum(n for n, _ in ls) + toks                   # keys and values read; the step's own written
        pairs = sum(q * n - q * (q - 1) // 2 for n, q in ls)   # visible (query, key) pairs
        return {"bytes": 2.0 * (2 * kv * case["kv_heads"] * hd + 2 * toks * case["heads"] * hd),
                "flops": 4.0 * pairs * case["heads"] * hd}
    wl = _workload(case)
    return {"bytes": float(wl.layers * wl.algorithmic_bytes(_active(case), out_bytes=4 if wl.act_dtype == torch.float32 else 2)),
            "flops": float(wl.layers * wl.algorithmic_flops())}


def tolerance(case):
    """About four times what the path differs by from itself in 64 bits (stack: from the same layers on another kernel
    plan, with other summation orders)."""
    kind = case["kind"]
    if kind == "load":
        return "exact"                                      # codes, scales and zero points are defined bit for bit
    if kind == "attend":                                    # probabilities and outputs in the storage type
        return {"rel": 1e-2, "max": 0.13} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 0.015}
    if kind == "stack":                                     # near-ties of the router resolve differently down the layers
        return {"rel": 2e-2, "max": 0.2}
    if kind == "engine":
        return {"rel": 5e-3, "max": 0.1}
    if case["model"] == "tiny":                             # fp32 outputs of fp16 operands
        return {"rel": 2.2e-3, "max": 1e-2, "differ": 0.0}
    return {"rel": 5.5e-3, "max": 0.03, "differ": 0.0}


def _layer(wl, layer):
    """Router weight, W4 bank and activations of one layer, by the recipe of ``workloads.LayerInputs``."""
    inp = LayerInputs(wl, DEV, layer)
    gate = inp.gate_weight()
    bank = odsd.W4ExpertBank(wl.E, wl.H, wl.I, DEV)
    for e, g, u, d in inp.experts():
        bank.load_expert(e, g, u, d)
    return gate, bank, inp.x()


def _layers(wl):
    """The layers of a stack: routers of their own; the experts of layer 0 in another order for each further layer,
    copied (drawing and quantising every layer's own would take most of the time)."""
    gate, bank, x = _layer(wl, 0)
    gates, banks = [gate], [bank]
    g = torch.Generator(device=DEV)
    g.manual_seed(wl.seed + 1)
    for l in range(1, wl.layers):
        gates.append(LayerInputs(wl, DEV, l).gate_weight())
        b = bank.clone()
        order = torch.randperm(wl.E, generator=g, device=DEV)
        for name in ("gu_q", "gu_sz", "dn_q", "dn_sz"):
            getattr(b, name).copy_(getattr(bank, name)[order])
        banks.append(b)
    norms = [(1.0 + 0.1 * torch.randn(wl.H, generator=g, device=DEV)).to(wl.act_dtype) for _ in range(wl.layers)]
    return gates, banks, norms, x


def _config(wl):
    return odsd.MoEConfig(hidden_size=wl.H, num_hidden_layers=wl.layers, num_experts=wl.E, num_experts_per_token=wl.K,
                          moe_intermediate_size=wl.I, norm_topk_prob=wl.renorm,
                          torch_dtype="float32" if wl.act_dtype == torch.float32 else "bfloat16")


def _prepare_attend(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    r = random.Random(seed)
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
    ls, bs, hd, kvh = _lengths(case), case["block"], case["head_dim"], case["kv_heads"]
    blocks = [-(-n // bs) for n, _ in ls]
    ids = list(range(sum(blocks)))
    r.shuffle(ids)
    seqs, at = {}, 0
    for i, (n, q) in enumerate(ls):
        # a verify step: one token that is accepted already, the others are drafts
        seqs[i] = odsd.SequenceSlots(bs, ids[at:at + blocks[i]], n, n - q + 1)
        at += blocks[i]
    build = {"verify": odsd.build_verify_context, "decode": odsd.build_decode_context, "prefill": odsd.build_prefill_context}[case["form"]]
    ctx = build(seqs, list(seqs), device=DEV)
    toks = sum(q for _, q in ls)
    mk = lambda *shape: torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).to(dt)  # noqa: E731
    return {"kind": "attend", "ctx": ctx, "q": mk(toks, case["heads"], hd), "k": mk(toks, kvh, hd), "v": mk(toks, kvh, hd),
            "k_cache": mk(sum(blocks), bs, kvh * hd), "v_cache": mk(sum(blocks), bs, kvh * hd), "kvh": kvh, "block": bs}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attend":
        return _prepare_attend(case, seed)
    if kind == "load":
        wl = CONFIGS[MODELS[case["model"]]]
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        mk = lambda n, k: (torch.randn(n, k, generator=g, device=DEV) * 0.02).to(torch.bfloat16)  # noqa: E731
        return {"kind": kind, "bank": odsd.W4ExpertBank(case["experts"], wl.H, wl.I, DEV),
                "weights": [(mk(wl.I, wl.H), mk(wl.I, wl.H), mk(wl.H, wl.I)) for _ in range(case["experts"])]}
    wl = _workload(case, seed)
    gates, banks, norms, x = _layers(wl)
    if kind == "block":
        plan = ops.MoeForwardPlan(wl.T, wl.H, wl.E, wl.K, wl.I, wl.renorm, wl.act_dtype, DEV, want_f32=False)
        return {"kind": kind, "plan": plan, "gate": gates[0], "table": banks[0].table(), "bank": banks[0], "x": x}
    x = x * RESIDUAL_SCALE
    if kind == "stack":
        return {"kind": kind, "stack": odsd.MoEOnlyStack(_config(wl), gates, norms, banks, wl.T), "x": x}
    return {"kind": kind, "runner": odsd.W4MoERunner(_config(wl), gates, banks, norms), "x": x,
            "experts": [b.all_expert_params() for b in banks]}


def run(s):
    kind = s["kind"]
    if kind == "block":
        o = s["plan"].run(s["x"], s["gate"], s["table"])
        return o.out_act, o.idx, o.w, o.counts
    if kind == "stack":
        return s["stack"].forward(s["x"])
    if kind == "engine":
        h = s["x"]
        for l, params in enumerate(s["experts"]):
            placement = odsd.ExpertPlacement(gpu_expert_params=params, cpu_expert_params={})
            h = s["runner"].forward_layer(l, h, placement).hidden_states
        return h
    if kind == "attend":
        c = s["ctx"]
        odsd.store_kvcache(s["k"], s["v"], s["k_cache"], s["v_cache"], c["slot_mapping"], c.get("verify_q_indices"))
        return odsd.attention_for_context(s["q"], s["k"], s["v"], s["k_cache"], s["v_cache"], c, s["kvh"], s["block"])
    b = s["bank"]
    for e, (gate, up, down) in enumerate(s["weights"]):
        b.load_expert(e, gate, up, down)
    return b.gu_q, b.gu_sz, b.dn_q, b.dn_sz
