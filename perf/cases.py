"""The work a speculative-decoding program hands to this package, as measurable cases.

A case is one pass through public entry points: a verification call, a draft expansion, an attention call, or one
forward of a decoder stack.  ``listed()`` holds the sizes of the repository's own benchmark configurations, ``draw``
gives others from the ranges around them, odd and ragged sizes included.
"""
from __future__ import annotations

import math
import random
from typing import Dict, List

import torch

from subspec_amd import ops, workloads as W
from subspec_amd.cache import create_kv_cache
from subspec_amd.model import Decoder, DecoderConfig, init_weights, quantize_layers

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}
VOCAB = W.QWEN_VOCAB

#: hidden size, query heads, KV heads, MLP width of a decoder layer (heads are 128 wide): the repository's default
#: decoder, a smaller and a wider one of the same family of architectures.
GEOMETRIES = {"default": (3584, 28, 4, 18944), "small": (2048, 16, 8, 5632), "wide": (4096, 32, 8, 14336)}


def listed() -> List[Dict]:
    return [
        # One decoding cycle of a single sequence, greedy target: 64 scored nodes, float32 logits.  The smallest call;
        # launches and the host side count as much as the 39 MB it reads.
        _verify("verify_greedy_1x64", trees=1, nodes=64, dtype="fp32", method="exact"),
        # Lossy verification of a batch of 32 trees behind the entropy gate, the repository's benchmark workload.
        _verify("verify_lossy_32x64", trees=32, nodes=64, dtype="bf16", method="lossy", gate="entropy", threshold=0.3, window=6),
        # The same batch with a sampling target: one draw per row.
        _verify("verify_sampled_32x64", trees=32, nodes=64, dtype="bf16", method="exact", temperature=0.8),
        # Top-16 of every row of a batch of draft probabilities, the benchmark's other half.
        {"name": "topk_2048", "kind": "topk", "rows": 2048, "vocab": VOCAB, "k": 16, "dtype": "bf16"},
        # What follows every draft level of one sequence: softmax(logits / T) of 8 leaves and the top 8 of all of them.
        {"name": "expand_8", "kind": "expand", "leaves": 8, "vocab": VOCAB, "k": 8, "dtype": "bf16", "temperature": 0.2},
        # Attention of a verification window, 8 sequences with 4096 cached rows each.
        {"name": "attention_8x64", "kind": "attention", "batch": 8, "nodes": 64, "prefix": 4096, "q_heads": 28, "kv_heads": 4,
         "dtype": "bf16"},
        # One level of the int4 draft: 8 leaves of the fifth level over a 2048-row prefix, all layers and the head.  A
        # decoding cycle runs this eight times, so it is where most of the resident cycle goes.
        _stack("draft_level_8", storage="int4", rows=8, level=5, prefix=2048),
        # The int4 draft over a whole 64-node window, as post-speculation scores the verified extension.
        _stack("draft_window_64", storage="int4", rows=64, level=0, prefix=2048),
        # The target's forward over a 64-node tree: once per cycle.
        _stack("target_window_64", storage="dense", rows=64, level=0, prefix=2048),
        # The target's forward over a tree of depth 48 with 6 nodes a level.
        _stack("target_tree_289", storage="dense", rows=289, level=0, prefix=2048),
        # Prefill of a prompt in chunks of 256 tokens: the last chunk of a 2048-token prompt.
        _prefill("prefill_chunk_256", tokens=256, start=1792),
        # Prefill of a 2048-token prompt in one piece: the largest pass.
        _prefill("prefill_2048", tokens=2048, start=0),
    ]


def draw(rng: random.Random) -> Dict:
    kind = rng.choice(["verify", "verify", "topk", "expand", "attention", "draft", "target", "prefill"])
    if kind == "verify":
        vocab = _vocab(rng)
        trees = _log_int(rng, 1, 32)
        nodes = _log_int(rng, 2, min(289, 2048 // trees))
        how = rng.choice(["greedy", "entropy", "prob", "sampled"])
        opts = {"greedy": dict(method="exact"), "sampled": dict(method="exact", temperature=rng.choice([0.2, 0.8, 1.0, 1.3])),
                "entropy": dict(method="lossy", gate="entropy", threshold=0.3, window=rng.choice([1, 2, 6])),
                "prob": dict(method="lossy", gate="prob", threshold=rng.choice([0.0, 0.05]), window=rng.choice([1, 2, 6]))}[how]
        # float32 logits come from single sequences; a batch of them is 16-bit
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"] if trees * nodes <= 512 else ["bf16", "bf16", "fp16"])
        return _verify("", trees=trees, nodes=nodes, dtype=dtype, vocab=vocab, **opts)
    if kind == "topk":
        return {"kind": "topk", "rows": _log_int(rng, 1, 2048), "vocab": _vocab(rng), "k": rng.choice([1, 4, 6, 8, 16, 32]),
                "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    if kind == "expand":
        return {"kind": "expand", "leaves": rng.randint(1, 16), "vocab": _vocab(rng), "k": rng.choice([4, 6, 8, 10, 16]),
                "dtype": rng.choice(["bf16", "bf16", "fp16"]), "temperature": rng.choice([0.2, 0.6, 1.0])}
    if kind == "attention":
        batch = rng.randint(1, 8)
        hq, hkv = rng.choice([(28, 4), (16, 8), (32, 8)])
        return {"kind": "attention", "batch": batch, "nodes": _log_int(rng, 1, min(289, 1024 // batch)),
                "prefix": _log_int(rng, 32, 4096), "q_heads": hq, "kv_heads": hkv, "dtype": rng.choice(["bf16", "bf16", "fp16"])}
    geometry = rng.choice(["default", "default", "small", "wide"])
    shape = dict(geometry=geometry, layers=_log_int(rng, 2, 24), dtype=rng.choice(["bf16", "bf16", "fp16"]))
    if kind == "prefill":
        tokens = _log_int(rng, 16, 1800)
        return _prefill("", tokens=tokens, start=rng.choice([0, rng.randint(1, 2048 - tokens)]), **shape)
    rows = _log_int(rng, 1, 64 if kind == "draft" else 289)
    return _stack("", storage="int4" if kind == "draft" else "dense", rows=rows, level=rng.randint(1, 6) if rows <= 16 else 0,
                  prefix=_log_int(rng, 32, 4096), **shape)


# ---------------------------------------------------------------------------------------------- descriptions
def _verify(name, trees, nodes, dtype, method, vocab=VOCAB, gate="prob", threshold=0.0, window=1, temperature=0.0) -> Dict:
    """``temperature`` 0: greedy target, otherwise one draw per row at that temperature."""
    return _named(name, {"kind": "verify", "trees": trees, "nodes": nodes, "vocab": vocab, "dtype": dtype, "method": method,
                         "gate": gate, "threshold": threshold, "window": window, "temperature": temperature})


def _stack(name, storage, rows, level, prefix, geometry="default", layers=28, dtype="bf16") -> Dict:
    """``level`` > 0: the rows are one level of a tree with ``rows`` nodes per level; 0: they are a whole tree."""
    return _named(name, {"kind": "stack", "storage": storage, "rows": rows, "level": level, "prefix": prefix,
                         "geometry": geometry, "layers": layers, "dtype": dtype})


def _prefill(name, tokens, start, geometry="default", layers=28, dtype="bf16") -> Dict:
    return _named(name, {"kind": "prefill", "tokens": tokens, "start": start, "geometry": geometry, "layers": layers,
                         "dtype": dtype})


def _named(name, case) -> Dict:
    return {"name": name, **case} if name else case


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _vocab(rng: random.Random) -> int:
    return rng.choice([VOCAB, VOCAB, 32000, 50257, _log_int(rng, 4096, VOCAB)])


def _config(case) -> DecoderConfig:
    hidden, hq, hkv, mlp = GEOMETRIES[case["geometry"]]
    return DecoderConfig(num_hidden_layers=case["layers"], hidden_size=hidden, num_attention_heads=hq, num_key_value_heads=hkv,
                         head_dim=128, intermediate_size=mlp, vocab_size=VOCAB)


# ---------------------------------------------------------------------------------------------- inputs
def prepare(case: Dict, seed: int) -> Dict:
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    state = {"case": case}
    if kind == "verify":
        # rows scaled to a range of entropies, a path planted in most of the trees
        cfg = W.lossy_config(seed=seed, batch=case["trees"], n=case["nodes"], vocab=case["vocab"], device=DEVICE, dtype=dtype)
        B, n = case["trees"], case["nodes"]
        state["args"] = (cfg["logits"], torch.tensor(cfg["tokens"], dtype=torch.int32, device=DEVICE),
                         torch.tensor(cfg["parents"], dtype=torch.int32, device=DEVICE))
        state["options"] = dict(verify_method=case["method"], threshold_method=case["gate"], threshold=case["threshold"],
                                window_size=case["window"])
        if case["temperature"] > 0:
            state["options"].update(do_sample=True, temperature=case["temperature"], seed=seed, offset=seed % 1000)
        # a decoding loop keeps its result tensors; the entries behind a tree's last token are never written
        zeros = lambda *shape, dtype: torch.zeros(shape, dtype=dtype, device=DEVICE)
        state["out"] = {"tokens": zeros(B, n + 1, dtype=torch.int64), "contexts": zeros(B, n + 1, dtype=torch.int64),
                        "counts": zeros(B, 4, dtype=torch.int32), "target": zeros(B, n, dtype=torch.int64),
                        "entropy": zeros(B, n, dtype=torch.float32), "child_prob": zeros(B, n, dtype=torch.float32)}
    elif kind in ("topk", "expand"):
        rows = case["rows"] if kind == "topk" else case["leaves"]
        scale = torch.rand(rows, 1, generator=gen, device=DEVICE) * 2.5 + 0.5
        logits = torch.randn(rows, case["vocab"], generator=gen, device=DEVICE) * scale
        if kind == "topk":
            state["probs"] = torch.softmax(logits, -1).to(dtype).view(rows, 1, -1)
            state["parents"] = torch.rand(rows, 1, generator=gen, device=DEVICE).to(dtype)
        else:
            state["logits"] = logits.to(dtype)
            state["parents"] = torch.rand(1, rows, generator=gen, device=DEVICE).to(dtype)
    elif kind == "attention":
        B, n, total = case["batch"], case["nodes"], case["prefix"] + case["nodes"]
        rnd = lambda *shape: torch.randn(*shape, generator=gen, device=DEVICE).to(dtype)
        parents, _, _ = _tree(host, n)
        state["q"], state["bits"] = rnd(B, case["q_heads"], n, 128), ops.ancestor_bits_tensor(parents, device=DEVICE)
        state["k"], state["v"] = rnd(B, case["kv_heads"], total, 128), rnd(B, case["kv_heads"], total, 128)
    else:
        state.update(_prepare_forward(case, seed, gen, host, dtype))
    return state


def _tree(host: torch.Generator, n: int):
    """A whole tree of ``n`` nodes: up to 64 of them as bushy as the benchmark's, more of them as deep as the
    depth-48 trees of the long configurations."""
    deep = n > 64
    return W.random_tree(host, n=n, max_depth=48 if deep else 8, max_children=6 if deep else 4, vocab=VOCAB,
                         chain_depth=min(40 if deep else 8, n - 1))


def _prepare_forward(case, seed, gen, host, dtype) -> Dict:
    cfg = _config(case)
    prefill = case["kind"] == "prefill"
    rows = case["tokens"] if prefill else case["rows"]
    prefix = case["start"] if prefill else case["prefix"]
    first = 0 if prefill or case["level"] == 0 else 1 + (case["level"] - 1) * rows
    kv = create_kv_cache("static", max_cache_len=prefix + first + rows + 64, config=cfg, device=DEVICE, dtype=dtype)
    kv.cache.data.normal_(generator=gen)
    w = init_weights(cfg, seed, DEVICE, dtype)
    # a trained stack adds small terms to a residual stream of order one: embeddings of unit size, and the two matrices
    # that write to the stream scaled down by the square root of their number (plain N(0, 0.02) stacks of this depth
    # amplify the last bit of a bf16 sum to a few percent of the logits)
    w["embed"].mul_(50.0)
    for layer in w["layers"]:
        for name in ("o_proj.weight", "down_proj.weight"):
            layer[name].mul_((2 * cfg.num_hidden_layers) ** -0.5)
    layers = w["layers"]
    if not prefill and case["storage"] == "int4":
        layers = []
        while w["layers"]:
            layers += quantize_layers([w["layers"].pop(0)])
    decoder = Decoder(cfg, w["embed"], layers, w["norm"], w["lm_head"], kv)
    tokens = torch.randint(0, cfg.vocab_size, (rows,), generator=host).to(DEVICE)
    state = {"decoder": decoder, "tokens": tokens, "prefix": prefix, "first": first, "rows": rows}
    if not prefill:
        if case["level"] == 0:
            parents, _, depths = _tree(host, rows)
        else:                                        # every level `rows` nodes, each under a random node of the level above
            parents, depths = [-1], [0]
            for d in range(1, case["level"] + 1):
                above = [i for i, x in enumerate(depths) if x == d - 1]
                parents += [above[int(torch.randint(0, len(above), (1,), generator=host))] for _ in range(rows)]
                depths += [d] * rows
        state["slots"] = first + rows
        state["bits"] = ops.ancestor_bits_tensor(parents, device=DEVICE)[first:].contiguous()
        # rotary positions and cache rows: the draft works them out for all levels of a speculation at once
        state["positions32"] = torch.tensor([prefix + d for d in depths[first:]], dtype=torch.int32, device=DEVICE)
        state["rows32"] = torch.arange(prefix + first, prefix + first + rows, dtype=torch.int32, device=DEVICE)
    return state


# ---------------------------------------------------------------------------------------------- the pass
@torch.no_grad()
def run(state: Dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "verify":
        return ops.tree_verify(*state["args"], out=state["out"], **state["options"])
    if kind == "topk":
        return ops.topk_expand(state["probs"], state["parents"], case["k"])
    if kind == "expand":
        probs = ops.softmax_temperature(state["logits"], case["temperature"]).unsqueeze(0)
        return (probs, *ops.topk_expand(probs, state["parents"], case["k"]))
    if kind == "attention":
        return ops.tree_attention(state["q"], state["k"], state["v"], state["bits"], case["prefix"])
    decoder, prefix = state["decoder"], state["prefix"]
    if kind == "prefill":
        logits = decoder.prefill(state["tokens"], prefix)
    else:
        logits = decoder.tree_forward(state["tokens"], None, state["bits"], prefix, first_slot=state["first"],
                                      n_tree_slots=state["slots"], positions32=state["positions32"], rows32=state["rows32"])
    written = prefix + state["first"]
    return logits, decoder.kv.cache.data[..., written:written + state["rows"], :]


# ---------------------------------------------------------------------------------------------- price and tolerance
def work(case: Dict) -> Dict:
    kind, es = case["kind"], SIZES[case["dtype"]]
    if kind == "verify":
        elems = case["trees"] * case["nodes"] * case["vocab"]
        return {"bytes": elems * es + case["trees"] * (case["nodes"] * 40 + 32), "flops": 4 * elems}
    if kind == "topk":
        elems = case["rows"] * case["vocab"]
        return {"bytes": elems * es + case["rows"] * (es + case["k"] * (16 + es)), "flops": elems}
    if kind == "expand":
        elems = case["leaves"] * case["vocab"]
        return {"bytes": 2 * elems * es + case["leaves"] * es + case["k"] * (16 + es), "flops": 5 * elems}
    if kind == "attention":
        B, n, hq, hkv = case["batch"], case["nodes"], case["q_heads"], case["kv_heads"]
        total = case["prefix"] + n
        return {"bytes": B * 128 * es * 2 * (hkv * total + hq * n), "flops": 4 * B * n * hq * total * 128}
    cfg = _config(case)
    H, F, Q, KV = cfg.hidden_size, cfg.intermediate_size, cfg.q_size, cfg.kv_size
    matrix = (Q + 2 * KV) * H + H * Q + 3 * F * H                       # elements of a layer's projections
    int4 = case["kind"] == "stack" and case["storage"] == "int4"
    per_layer = (matrix // 2 + matrix // 64 * 4 if int4 else matrix * es) + (2 * H + Q + 2 * KV) * es
    if case["kind"] == "prefill":
        n, before, head_rows = case["tokens"], case["start"], 1
        keys = n * before + n * (n + 1) // 2                             # (row, key) pairs under the causal mask
    else:
        n, head_rows = case["rows"], case["rows"]
        before = case["prefix"] + (0 if case["level"] == 0 else 1 + (case["level"] - 1) * n)
        keys = n * (before + n)
    bytes_ = (case["layers"] * (per_layer + 2 * KV * es * (before + n)) + n * H * es + VOCAB * H * es + head_rows * VOCAB * es)
    flops = case["layers"] * (2 * n * matrix + 4 * cfg.num_attention_heads * 128 * keys) + 2 * head_rows * VOCAB * H
    return {"bytes": bytes_, "flops": flops}


def tolerance(case: Dict):
    kind, narrow = case["kind"], case["dtype"]
    if kind == "topk":
        return "exact"                               # the order of values and indices is defined, ties included
    if kind == "verify":
        # tokens and paths are whole numbers; entropies of rows far from the gate are float32 sums (guarded rows and the
        # probabilities carry one rounding of the logits' type, which a last-bit change of the row sum can move)
        return {"rel": 1e-4 if narrow == "fp32" else 2e-3}
    if kind == "expand":
        return {"rel": 1e-3, "max": 0.02}            # one rounding per probability, moved by the last bit of a row sum
    if kind == "attention":
        return {"rel": 1e-2 if narrow == "bf16" else 2e-3}
    # a whole stack: every sum in another order (module by module against one call per layer, a prompt in two pieces
    # against one) moves the logits of 28 bf16 layers by 0.018 to 0.020, of 6 by 0.008 to 0.011; fp16 has three bits more
    return {"rel": 0.03, "max": 0.25} if narrow == "bf16" else {"rel": 0.01, "max": 0.1}
