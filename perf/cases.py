"""The work this framework is used for, as cases that can be measured.

A case is one call (or one layer's calls) that a program makes through the
public entry points: decoding compressed FP8 blocks, compressing a weight,
the layers that read the decoded or re-tiled weights in a decode step and in
a prompt, a DiT block, and one whole decode step of a small model.  Shapes
are those of the configurations in ``ecf8_amd.synth``, ``ecf8_amd.llm``,
``ecf8_amd.moe`` and ``ecf8_amd.dit``.

``listed()`` names twelve cases; ``draw(rng)`` takes one more from the same
ranges (``RANGES``); ``prepare`` / ``run`` make the inputs and run one pass;
``work``, ``tolerance`` and ``exact`` say what a pass has to move and
compute, how closely two correct implementations agree, and what a pass
returns in 64 bits.
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn

from dfloat.compress import compress_flat
from dfloat.huffman import get_nbit_codec
from dfloat.utils import get_luts_from_huffman_table
from ecf8_amd import decode as D
from ecf8_amd import llm_kernels as K
from ecf8_amd import tiled
from ecf8_amd.dit import FluxConfig, FluxPipeline, compress_blocks, fuse_dequant_blocks
from ecf8_amd.llm import Qwen3Config, Qwen3ForCausalLM, Qwen3Runner, tile_resident_weights
from ecf8_amd.synth import (QWEN3_8B_LAYER, QWEN3_MOE_EXPERT, flat_block, quantize_fp8_blockwise)

DEV = "cuda"
EPS = 1e-6
MOE = {"hidden": 2048, "inter": 768, "experts": 128, "top_k": 8}
DISTINCT_EXPERTS = 8      # experts drawn; the others are device copies of one of them
BITS = 2.577              # coded bits per exponent of block-quantized normal weights


def listed() -> list[dict]:
    return [
        # Smallest call of the decoder: one routed expert (its three Linears as
        # one compressed block), decoded in its hook.
        {"name": "decode_expert", "kind": "decode", "elements": 3 * 768 * 2048, "tpb": 512},
        # The headline call: one Qwen3-8B-shaped decoder layer, one block.
        {"name": "decode_layer", "kind": "decode", "elements": 192937984, "tpb": 512},
        # A MoE decode step that decodes only the experts 16 tokens picked.
        {"name": "decode_routed", "kind": "routed", "tokens": 16},
        # Offline direction: one 4096 x 4096 Linear compressed on the host.
        {"name": "compress_linear", "kind": "compress", "elements": 4096 * 4096},
        # An FP8 Linear (quantize + GEMM) for a batch above the decode-step
        # kernels' 16 rows: a served batch of 64 sequences.
        {"name": "linear_batch64", "kind": "linear", "rows": 64, "n": 4096, "k": 4096,
         "layout": "tiles"},
        # One decoder layer of a re-tiled model in a decode step (one graph
        # replay): 16 sequences, 640 cached positions.
        {"name": "layer_step", "kind": "step", "batch": 16, "cached": 640, "weights": "tiled"},
        # The same layer over the prompt, FP8 resident weights: 16 x 128 tokens.
        {"name": "layer_prompt", "kind": "prompt", "batch": 16, "tokens": 128},
        # The routed MLP of a re-tiled MoE layer in a decode step (one graph
        # replay): router, grouping, grouped linears, combine.
        {"name": "moe_step", "kind": "moe_step", "tokens": 16},
        # The routed MLP over one 512-token chunk of the prompt.
        {"name": "moe_prompt", "kind": "moe_prompt", "tokens": 512, "layout": "rows"},
        # Decode attention over a long context: 16 sequences, 8192 positions.
        {"name": "attention_long", "kind": "attention", "batch": 16, "cached": 8192, "group": 4},
        # One single-stream DiT block at 1024 x 1024 pixels (4096 image + 512
        # text tokens), compressed, decoded straight to bf16 by its hook.
        {"name": "dit_single", "kind": "dit", "block": "single", "grid_h": 64, "grid_w": 64,
         "text": 512, "weights": "fused"},
        # A whole decode step (2 re-tiled layers, norm, lm_head, greedy token)
        # as generation replays it: logits of 16 sequences.
        {"name": "model_step", "kind": "model", "batch": 16, "cached": 1024, "layers": 2},
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# {kind: (weight of the kind in draw(), rng -> fields)}
RANGES = {
    # blocks from a small Linear up to a whole layer; any even element count,
    # the format's chunk counts
    "decode": (3, lambda g: {"elements": 2 * _log(g, 50_000, 96_468_992),
                             "tpb": g.choice([128, 256, 512, 512, 512, 1024])}),
    # 1 token (8 experts) up to every expert
    "routed": (1, lambda g: {"tokens": _log(g, 1, 64)}),
    "compress": (1, lambda g: {"elements": 2 * _log(g, 500_000, 8_388_608)}),
    # one row up to a long prompt; widths and depths in 128s
    "linear": (3, lambda g: {"rows": _log(g, 1, 4096), "n": 128 * g.randint(4, 96),
                             "k": 128 * g.randint(4, 96), "layout": g.choice(["rows", "tiles"])}),
    "step": (2, lambda g: {"batch": g.randint(1, 16), "cached": _log(g, 1, 4096),
                           "weights": g.choice(["tiled", "fp8"])}),
    "prompt": (2, lambda g: (lambda t: {"batch": g.randint(1, max(1, min(16, 4096 // t))),
                                        "tokens": t})(_log(g, 4, 2048))),
    "moe_step": (1, lambda g: {"tokens": g.randint(1, 16)}),
    "moe_prompt": (1, lambda g: {"tokens": _log(g, 17, 1024),
                                 "layout": g.choice(["rows", "tiles"])}),
    "attention": (2, lambda g: (lambda b: {"batch": b, "cached": _log(g, 1, min(32768, 131072 // b)),
                                           "group": g.choice([4, 8])})(_log(g, 1, 64))),
    "dit": (2, lambda g: (lambda b: {"block": b, "grid_h": g.randint(16, 64),
                                     "grid_w": g.randint(16, 64), "text": g.randint(64, 512),
                                     "weights": g.choice(["fp8", "fused"]) if b == "single"
                                     else "fp8"})(g.choice(["single", "double"]))),
    "model": (1, lambda g: {"batch": g.randint(1, 16), "cached": _log(g, 8, 2048),
                            "layers": g.randint(1, 2)}),
}


def draw(rng) -> dict:
    kinds = [k for k, (w, _) in RANGES.items() for _ in range(w)]
    kind = rng.choice(kinds)
    return {"kind": kind, **RANGES[kind][1](rng)}


# ------------------------------------------------------------------ inputs


def _gen(seed: int, device=DEV) -> torch.Generator:
    return torch.Generator(device=device).manual_seed(int(seed))


def _weight(n, k, g, sigma=0.02):
    """(e4m3fn [n, k], scale_inv f32) of N(0, sigma) weights, on the GPU."""
    return quantize_fp8_blockwise(torch.randn(n, k, generator=g, device=DEV) * sigma)


def _flat(elements: int, g) -> torch.Tensor:
    """``elements`` block-quantized FP8 weights, flattened."""
    cols = 4096 if elements >= 128 * 4096 else 128
    rows = -(-elements // (128 * cols)) * 128
    return _weight(rows, cols, g)[0].reshape(-1)[:elements]


def _to_gpu(comp: dict) -> dict:
    return {k: comp[k].to(DEV) for k in ("luts", "encoded", "packed_other_4bits",
                                         "output_positions", "gaps")}


def _code(weights):
    """(code_bits, code_vals, automaton table) of one block's Huffman code."""
    counts = torch.zeros(16, dtype=torch.int64)
    for w in weights:
        e = (w.view(torch.uint8).reshape(-1) >> 3) & 0xF
        counts += torch.bincount(e.int(), minlength=16).cpu()
    counter = {int(v): int(counts[v]) for v in range(16) if int(counts[v])}
    luts = get_luts_from_huffman_table(get_nbit_codec(counter, max_n_bits=16)[2])
    return (*tiled.code_from_luts(luts), D.build_table(luts.to(DEV)))


def _dense_config(layers: int, vocab: int) -> Qwen3Config:
    return Qwen3Config(layers=layers, vocab=vocab)


def _dense_weights(seed: int) -> dict:
    """{Linear: (fp8, scale_inv)} of the one layer drawn (all layers of a
    model hold their own copies of it)."""
    g = _gen(seed)
    return {n: _weight(o, i, g, s) for n, (o, i, s) in sorted(QWEN3_8B_LAYER.items())}


def _norm_weight(shape, g):
    return (1 + 0.1 * torch.randn(shape, generator=g, device=DEV)).to(torch.bfloat16)


def _dense_norms(layers, seed):
    """Norm weights: per layer (input, post-attention, q, k), then the final one."""
    g = _gen(seed + 71)
    per = [tuple(_norm_weight(n, g) for n in (4096, 4096, 128, 128)) for _ in range(layers)]
    return per, _norm_weight(4096, g)


def _head(vocab, seed):
    """(embedding, lm_head) bf16 [vocab, 4096]."""
    g = _gen(seed + 72)
    return tuple((torch.randn(vocab, 4096, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
                 for _ in range(2))


def _dense_model(case, seed, layers=1, vocab=128):
    """A Qwen3-shaped model of ``layers`` layers, re-tiled or FP8 resident."""
    cfg = _dense_config(layers, vocab)
    with torch.device("meta"):
        model = Qwen3ForCausalLM(cfg)
    model = model.to_empty(device=DEV)
    weights, (norms, last) = _dense_weights(seed), _dense_norms(layers, seed)
    tiles = table = None
    if case.get("weights", "tiled") == "tiled" and case["kind"] != "prompt":
        bits, vals, table = _code([w for w, _ in weights.values()])
        tiles = {n: tiled.tile_encode(w, bits, vals) for n, (w, _) in weights.items()}
    with torch.no_grad():
        emb, head = _head(vocab, seed)
        model.model.embed_tokens.weight.copy_(emb)
        model.lm_head.weight.copy_(head)
        model.model.norm.weight.copy_(last)
        for layer, (n1, n2, qn, kn) in zip(model.model.layers, norms):
            layer.input_layernorm.weight.copy_(n1)
            layer.post_attention_layernorm.weight.copy_(n2)
            layer.self_attn.q_norm.weight.copy_(qn)
            layer.self_attn.k_norm.weight.copy_(kn)
            for name, (w, s) in weights.items():
                lin = layer.get_submodule(name)
                lin.weight_scale_inv = s.clone()
                lin.weight = nn.Parameter(w.clone() if tiles is None else w, requires_grad=False)
            if tiles is not None:  # what retile_layers leaves on a layer
                layer._ecf8_tiles = {n: tiled.TiledOperand(enc, weights[n][1].clone(),
                                                           *weights[n][0].shape)
                                     for n, enc in tiles.items()}
                layer._ecf8_tile_table = table
                for name in weights:
                    lin = layer.get_submodule(name)
                    lin.weight = nn.Parameter(torch.empty(0, dtype=torch.float8_e4m3fn,
                                                          device=DEV), requires_grad=False)
    if tiles is None:
        tile_resident_weights(model)
    return model


def _kv(batch, heads, length, g):
    """Cached keys (normalized heads) and values, bf16 [B, Hkv, L, 128]."""
    shape = (batch, heads, length, 128)
    return (torch.randn(shape, generator=g, device=DEV).to(torch.bfloat16),
            (torch.randn(shape, generator=g, device=DEV) * 0.5).to(torch.bfloat16))


def _graph(fn):
    """One call of ``fn`` as a HIP graph (after an eager call, which builds
    what is built lazily)."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


def _prepare_decode(case, seed):
    comp = compress_flat(_flat(case["elements"], _gen(seed)).cpu(), 8, case["tpb"])
    blk = _to_gpu(comp)
    return {"blk": blk, "table": D.build_table(blk["luts"]), "tpb": case["tpb"],
            "largest": D.largest_block(comp["output_positions"]),
            "bits": D.min_code_bits(comp["luts"]),
            "out": torch.zeros(case["elements"], dtype=torch.uint8, device=DEV)}


def _run_decode(st):
    b = st["blk"]
    return D.decode_into(st["out"], b["luts"], b["encoded"], b["packed_other_4bits"],
                         b["output_positions"], b["gaps"], table=st["table"],
                         threads_per_block=st["tpb"], max_block_elements=st["largest"],
                         min_code_bits=st["bits"])


def _expert_weights(seed):
    """The distinct experts drawn: [{Linear: (fp8, scale_inv)}]."""
    g = _gen(seed + 5)
    return [{n: _weight(o, i, g, s) for n, (o, i, s) in sorted(QWEN3_MOE_EXPERT.items())}
            for _ in range(DISTINCT_EXPERTS)]


def _flags(tokens, seed):
    """Select flags of uniform random top-8 routing."""
    g = _gen(seed + 6, "cpu")
    flags = torch.zeros(MOE["experts"], dtype=torch.int32)
    for _ in range(tokens):
        flags[torch.randperm(MOE["experts"], generator=g)[: MOE["top_k"]]] = 1
    return flags


def _prepare_routed(case, seed):
    comps = [_to_gpu(compress_flat(flat_block({n: w.cpu() for n, (w, _) in ex.items()})[0]))
             for ex in _expert_weights(seed)]
    blocks = [{k: v.clone() for k, v in comps[e % len(comps)].items()}
              for e in range(MOE["experts"])]
    n = comps[0]["packed_other_4bits"].numel() * 2
    out = torch.zeros(MOE["experts"] * n, dtype=torch.uint8, device=DEV)
    plan = D.prepare_batch(blocks, list(out.split(n)), [D.build_table(b["luts"]) for b in blocks])
    return {"select": D.BatchSelect(plan), "flags": _flags(case["tokens"], seed).to(DEV),
            "out": out}


def _run_routed(st):
    st["select"](st["flags"])
    return st["out"]


def _prepare_compress(case, seed):
    """The weights, and the buffer of a checkpoint writer that takes the
    block (its coded size depends on the weights)."""
    n = case["elements"]
    return {"flat": _flat(n, _gen(seed)).cpu(), "file": torch.zeros(n + 65536, dtype=torch.uint8)}


def _run_compress(st):
    got, off = compress_flat(st["flat"]), 0
    for k in ("luts", "output_positions", "gaps", "encoded", "packed_other_4bits"):
        t = got[k].reshape(-1)
        st["file"][off:off + t.numel()] = t
        off += t.numel()
    return st["file"]


def _linear_inputs(case, seed):
    g = _gen(seed)
    x = torch.randn(case["rows"], case["k"], generator=g, device=DEV).to(torch.bfloat16)
    return x, _weight(case["n"], case["k"], g)


def _prepare_linear(case, seed):
    x, (w, s) = _linear_inputs(case, seed)
    M, N, k = case["rows"], case["n"], case["k"]
    out = torch.zeros(M, N, dtype=torch.bfloat16, device=DEV)
    entry = (w, s) if case["layout"] == "rows" else (K.to_tiles(w), s, K.WEIGHT_TILES)
    return {"x": x, "plan": K.LinearPlan([entry], out),
            "aq": torch.zeros(K.pad16(M), k, dtype=torch.uint8,
                              device=DEV).view(torch.float8_e4m3fn),
            "as": torch.zeros(M, k // 128, device=DEV)}


def _run_linear(st):
    M = st["x"].shape[0]
    K.act_quant(st["x"], M, st["aq"], st["as"])
    return st["plan"](st["aq"], st["as"], M)


def _step_inputs(case, seed):
    B, L = case["batch"], case["cached"]
    g = _gen(seed + 3)
    x = torch.randn(B, 4096, generator=g, device=DEV)
    return x, _kv(B, 8, L + 1, g)


def _prepare_step(case, seed):
    """A decode step's layer: position ``cached`` attends to the cached
    positions before it and itself."""
    B, L = case["batch"], case["cached"]
    model = _dense_model(case, seed)
    r = Qwen3Runner(model, B, 1, L + 1)
    x, (kc, vc) = _step_inputs(case, seed)
    r.kc[0].copy_(kc)
    r.vc[0].copy_(vc)
    r.pos.fill_(L)
    layer = model.model.layers[0]

    def once():
        r.res[:B].copy_(x)
        layer(r, 0, None, False)

    return {"graph": _graph(once), "keep": (r, x, model),
            "out": {"mlp": r.down[:B], "residual": r.res[:B], "k": r.kc[0][:, :, L],
                    "v": r.vc[0][:, :, L]}}


def _run_graph(st):
    st["graph"].replay()
    return st["out"]


def _prompt_x(case, seed):
    return torch.randn(case["batch"] * case["tokens"], 4096, generator=_gen(seed + 4), device=DEV)


def _prepare_prompt(case, seed):
    B, T = case["batch"], case["tokens"]
    model = _dense_model(case, seed)
    r = Qwen3Runner(model, B, T, T)
    return {"r": r, "x": _prompt_x(case, seed), "layer": model.model.layers[0], "model": model}


def _run_prompt(st):
    r = st["r"]
    r.pos.zero_()
    r.res.copy_(st["x"])
    down = st["layer"](r, 0, None, True)
    return {"mlp": down, "residual": r.res, "k": r.kc[0], "v": r.vc[0]}


def _moe_inputs(case, seed):
    """(hidden rows bf16 [M, H], router bf16 [E, H])."""
    g = _gen(seed + 8)
    x = torch.randn(case["tokens"], MOE["hidden"], generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(MOE["experts"], MOE["hidden"], generator=g, device=DEV) * 0.02)
    return x, w.to(torch.bfloat16)


def _moe_state(case, seed):
    M, H, I, E = case["tokens"], MOE["hidden"], MOE["inter"], MOE["experts"]
    P = M * MOE["top_k"]
    x, router = _moe_inputs(case, seed)
    bf = dict(dtype=torch.bfloat16, device=DEV)

    def fp8(rows, cols):
        return torch.zeros(K.pad16(rows), cols, dtype=torch.uint8,
                           device=DEV).view(torch.float8_e4m3fn)

    return {"x": x, "router": router, "route": K.MoeRouting(M, MOE["top_k"], E, DEV),
            "gu": torch.zeros(P, 2 * I, **bf), "down": torch.zeros(P, H, **bf),
            "y": torch.zeros(M, H, **bf), "aq": fp8(M, H),
            "as": torch.zeros(M, H // 128, device=DEV), "hq": fp8(P, I),
            "hs": torch.zeros(P, I // 128, device=DEV)}


def _moe_mlp(st):
    """The routed MLP as the runner issues it."""
    M, r = st["x"].shape[0], st["route"]
    K.act_quant(st["x"], M, st["aq"], st["as"])
    K.moe_route(st["x"], st["router"], M, r)
    K.moe_group(r, M)
    st["lin_gu"](st["aq"], st["as"], r, gather=True, M=M)
    K.silu_mul_quant(st["gu"], M * r.top_k, st["hq"], st["hs"])
    st["lin_down"](st["hq"], st["hs"], r, gather=False, M=M)
    K.moe_combine(st["down"], r, M, st["y"])
    return {"y": st["y"], "weights": r.topk_w}


def _prepare_moe_step(case, seed):
    st = _moe_state(case, seed)
    drawn = []
    for ex in _expert_weights(seed):
        bits, vals, table = _code([w for w, _ in ex.values()])
        drawn.append(({n: {k: v.to(DEV) for k, v in tiled.tile_encode(w, bits, vals).items()}
                       for n, (w, _) in ex.items()}, ex, table))
    experts, tables = [], []
    for e in range(MOE["experts"]):
        enc, ex, table = drawn[e % len(drawn)]
        experts.append({n: tiled.TiledOperand({k: v.clone() for k, v in enc[n].items()},
                                              ex[n][1].clone(), *ex[n][0].shape) for n in enc})
        tables.append(D.DecodeTable(table.data.clone(), table.kind))
    st["lin_gu"] = tiled.TileMoePlan([[e["gate_proj"], e["up_proj"]] for e in experts], tables,
                                     st["gu"])
    st["lin_down"] = tiled.TileMoePlan([[e["down_proj"]] for e in experts], tables, st["down"])
    st["graph"] = _graph(lambda: _moe_mlp(st))
    st["out"] = {"y": st["y"], "weights": st["route"].topk_w}
    return st


def _prepare_moe_prompt(case, seed):
    st = _moe_state(case, seed)
    drawn = _expert_weights(seed)
    layout = K.WEIGHT_TILES if case["layout"] == "tiles" else K.WEIGHT_ROWS
    experts = []
    for e in range(MOE["experts"]):
        ex = drawn[e % len(drawn)]
        experts.append({n: (K.to_tiles(w) if layout else w.clone(), s.clone())
                        for n, (w, s) in ex.items()})
    st["lin_gu"] = K.MoeLinearPlan([[e["gate_proj"], e["up_proj"]] for e in experts], st["gu"],
                                   layout)
    st["lin_down"] = K.MoeLinearPlan([[e["down_proj"]] for e in experts], st["down"], layout)
    return st


def _attention_inputs(case, seed):
    B, L, G = case["batch"], case["cached"], case["group"]
    g = _gen(seed + 9)
    hkv = 32 // G
    qkv = torch.randn(B, (32 + 2 * hkv) * 128, generator=g, device=DEV).to(torch.bfloat16)
    qn, kn = _norm_weight(128, g), _norm_weight(128, g)
    kc, vc = _kv(B, hkv, L + 1, g)
    return qkv, qn, kn, kc, vc


def _rotary(length):
    inv = 1.0 / (1e6 ** (torch.arange(0, 128, 2, dtype=torch.float64) / 128))
    ang = torch.arange(length, dtype=torch.float64)[:, None] * inv[None]
    return torch.cos(ang).to(DEV), torch.sin(ang).to(DEV)


def _prepare_attention(case, seed):
    B, L = case["batch"], case["cached"]
    qkv, qn, kn, kc, vc = _attention_inputs(case, seed)
    cos, sin = (t.float().contiguous() for t in _rotary(L + 1))
    st = {"args": (qkv, B, 32, 32 // case["group"], qn, kn, EPS, cos, sin,
                   torch.full((1,), L, dtype=torch.int32, device=DEV), kc, vc,
                   K.attention_work(B, 32, L + 1, DEV),
                   torch.zeros(K.pad16(B), 4096, dtype=torch.uint8,
                               device=DEV).view(torch.float8_e4m3fn),
                   torch.zeros(B, 32, device=DEV),
                   torch.zeros(B, 4096, dtype=torch.bfloat16, device=DEV))}
    return st


def _run_attention(st):
    K.decode_attention_fused(*st["args"])
    qkv, B, hq, hkv, qn, kn, eps, cos, sin, pos, kc, vc, work, out_q, out_s, out_b = st["args"]
    L = kc.shape[2] - 1
    return {"q": out_q, "scale": out_s, "bf16": out_b, "k": kc[:, :, L], "v": vc[:, :, L]}


def _dit_shapes(case):
    cfg = FluxConfig(double=int(case["block"] == "double"), single=int(case["block"] == "single"))
    return cfg, (cfg.double_shapes() if cfg.double else cfg.single_shapes())


def _dit_weights(case, seed):
    g = _gen(seed + 11)
    return {n: _weight(o, i, g, s) for n, (o, i, s) in sorted(_dit_shapes(case)[1].items())}


def _dit_inputs(case, seed):
    g = _gen(seed + 12)
    n_img, n_txt = case["grid_h"] * case["grid_w"], case["text"]

    def rows(n):
        return torch.randn(1, n, 3072, generator=g, device=DEV).to(torch.bfloat16)

    return rows(n_img), rows(n_txt), torch.randn(1, 3072, generator=g,
                                                 device=DEV).to(torch.bfloat16)


def _dit_block(case, seed):
    """The pipeline that holds the one block, its other parameters drawn."""
    cfg, _ = _dit_shapes(case)
    with torch.device("meta"):
        pipe = FluxPipeline(cfg)
    pipe = pipe.to_empty(device=DEV)
    g = _gen(seed + 13)
    with torch.no_grad():
        for name, p in pipe.named_parameters():
            if p.dtype == torch.bfloat16:
                if name.split(".")[-2].startswith("norm_"):
                    p.copy_(_norm_weight(p.shape, g))
                elif name.endswith(".bias"):
                    p.copy_((torch.randn(p.shape, generator=g, device=DEV) * 0.02).bfloat16())
                else:
                    p.copy_((torch.randn(p.shape, generator=g, device=DEV) * 0.02).bfloat16())
    blk = pipe.dit.blocks[0] if cfg.double else pipe.dit.single_blocks[0]
    for name, (w, s) in _dit_weights(case, seed).items():
        lin = blk.get_submodule(name)
        lin.weight = nn.Parameter(w, requires_grad=False)
        lin.weight_scale_inv = s
    return pipe, blk


def _prepare_dit(case, seed):
    pipe, blk = _dit_block(case, seed)
    if case["weights"] == "fused":
        compress_blocks(pipe)
        fuse_dequant_blocks(pipe)
    cos, sin = pipe.dit.rope_tables(case["text"], case["grid_h"], case["grid_w"], DEV)
    img, txt, emb = _dit_inputs(case, seed)
    args = ((img, txt, emb) if case["block"] == "double"
            else (torch.cat([txt, img], dim=1), emb))
    return {"blk": blk, "args": (*args, cos, sin), "pipe": pipe}


def _run_dit(st):
    with torch.no_grad():
        return st["blk"](*st["args"])


def _model_tokens(case, seed):
    return torch.randint(0, 151936, (case["batch"],), generator=_gen(seed + 15), device=DEV)


def _model_kv(case, seed):
    g = _gen(seed + 16)
    return [_kv(case["batch"], 8, case["cached"] + 1, g) for _ in range(case["layers"])]


def _prepare_model(case, seed):
    B, L = case["batch"], case["cached"]
    model = _dense_model(case, seed, case["layers"], 151936)
    r = Qwen3Runner(model, B, 1, L + 1)
    for i, (kc, vc) in enumerate(_model_kv(case, seed)):
        r.kc[i].copy_(kc)
        r.vc[i].copy_(vc)
    start = torch.full((1,), L, dtype=torch.int32, device=DEV)
    r.pos.copy_(start)
    tok = _model_tokens(case, seed)
    r.next_tok.copy_(tok)
    r.capture()
    return {"r": r, "start": start, "tok": tok, "model": model}


def _run_model(st):
    r = st["r"]
    r.pos.copy_(st["start"])
    r.step.zero_()
    r.next_tok.copy_(st["tok"])
    r.graph.replay()
    return r.logits


_PREPARE = {"decode": _prepare_decode, "routed": _prepare_routed, "compress": _prepare_compress,
            "linear": _prepare_linear, "step": _prepare_step, "prompt": _prepare_prompt,
            "moe_step": _prepare_moe_step, "moe_prompt": _prepare_moe_prompt,
            "attention": _prepare_attention, "dit": _prepare_dit, "model": _prepare_model}
_RUN = {"decode": _run_decode, "routed": _run_routed, "compress": _run_compress,
        "linear": _run_linear, "step": _run_graph, "prompt": _run_prompt, "moe_step": _run_graph,
        "moe_prompt": _moe_mlp, "attention": _run_attention, "dit": _run_dit, "model": _run_model}


def prepare(case, seed):
    return {"run": _RUN[case["kind"]], **_PREPARE[case["kind"]](case, seed)}


def run(state):
    return state["run"](state)


# -------------------------------------------------- work of a pass, tolerance

_LAYER_N = sum(o * i for o, i, _ in QWEN3_8B_LAYER.values())
_EXPERT_N = sum(o * i for o, i, _ in QWEN3_MOE_EXPERT.values())
_CODED = 0.5 + BITS / 8 * (1 + 1 / 16)  # bytes per weight: nibble, code, a gap nibble per 8 B


def _experts_used(tokens):
    """Distinct experts that uniform top-8 routing of ``tokens`` picks, on average."""
    e, k = MOE["experts"], MOE["top_k"]
    return e * (1 - (1 - k / e) ** tokens)


def _dense_work(B, T, L, weight_bytes, layers=1):
    """A dense layer over B x T new positions after L cached ones."""
    M = B * T
    pairs = B * sum((L * T, T * (T + 1) // 2))  # (query, key) pairs of one head
    kv = B * 8 * 128 * 2 * 2
    return {"bytes": layers * (weight_bytes + kv * (L + 2 * T) + M * 4096 * (4 + 4 + 2)),
            "flops": layers * (2 * M * _LAYER_N + 4 * pairs * 32 * 128)}


def work(case):
    kind = case["kind"]
    if kind == "decode":
        return {"bytes": case["elements"] * (_CODED + 1), "flops": 0}
    if kind == "routed":
        return {"bytes": int(_flags(case["tokens"], 0).sum()) * _EXPERT_N * (_CODED + 1),
                "flops": 0}
    if kind == "compress":
        return {"bytes": case["elements"] * (_CODED + 1), "flops": 0}
    if kind == "linear":
        M, N, k = case["rows"], case["n"], case["k"]
        return {"bytes": N * k + 2 * M * (N + k), "flops": 2 * M * N * k}
    if kind in ("step", "model"):
        coded = case.get("weights", "tiled") == "tiled"
        w = _dense_work(case["batch"], 1, case["cached"], _LAYER_N * (_CODED if coded else 1),
                        case.get("layers", 1))
        if kind == "model":
            w["bytes"] += 2 * 151936 * (4096 + case["batch"])
            w["flops"] += 2 * case["batch"] * 151936 * 4096
        return w
    if kind == "prompt":
        return _dense_work(case["batch"], case["tokens"], 0, _LAYER_N)
    if kind in ("moe_step", "moe_prompt"):
        M = case["tokens"]
        per = _EXPERT_N * (_CODED if kind == "moe_step" else 1)
        return {"bytes": _experts_used(M) * per + 2 * M * 2 * 2048 + 2 * 128 * 2048,
                "flops": 2 * M * 8 * _EXPERT_N + 2 * M * 128 * 2048}
    if kind == "attention":
        B, L, hkv = case["batch"], case["cached"], 32 // case["group"]
        return {"bytes": B * (L + 1) * hkv * 128 * 2 * 2 + B * 4096 * 5,
                "flops": 4 * B * 32 * (L + 1) * 128}
    n_txt, n_img = case["text"], case["grid_h"] * case["grid_w"]
    T = n_img + n_txt
    shapes = _dit_shapes(case)[1]
    rows = {"a": n_img, "b": n_txt}
    flops = 4 * T * T * 24 * 128
    for name, (o, i, _) in shapes.items():
        m = (1 if name == "norm.linear" else T if case["block"] == "single"
             else rows[name.split(".")[1][0] if name.startswith("attn") else name[3]])
        flops += 2 * m * o * i
    n = sum(o * i for o, i, _ in shapes.values())
    return {"bytes": n * (_CODED if case["weights"] == "fused" else 1) + 2 * T * 3072 * 2,
            "flops": flops}


def tolerance(case):
    """Bytes and codes are exact.  The others round to bf16 and quantize
    activations to 3 mantissa bits between Linears, so a last-bit
    difference of a sum can move single activation codes.  About four times
    what the same path shows with its sums in another order or its
    attention in 64 bits (MI355X, relative / largest): Linear 5.5e-5 /
    0.007, prompt layer 2.1e-3 / 0.10, DiT block 3.3e-3 / 0.033, attention
    against its 64-bit result 2.6e-3 / 0.008 (the bf16 rounding)."""
    return {"decode": "exact", "routed": "exact", "compress": "exact",
            "linear": {"rel": 0.0005, "max": 0.03},
            "step": {"rel": 0.01, "max": 0.4}, "prompt": {"rel": 0.01, "max": 0.4},
            "moe_step": {"rel": 0.01, "max": 0.4}, "moe_prompt": {"rel": 0.01, "max": 0.4},
            "attention": {"rel": 0.01, "max": 0.15},
            "dit": {"rel": 0.014, "max": 0.14},
            "model": {"rel": 0.02, "max": 0.4}}[case["kind"]]


# ------------------------------------------------------------ in 64 bits


def _q64(x):
    """Activations as the FP8 Linears take them: e4m3fn codes per row and
    128 columns at scale amax / 448 (1 for an all-zero group), in 64 bits."""
    g = x.double().reshape(*x.shape[:-1], -1, 128)
    amax = g.abs().amax(-1, keepdim=True)
    s = torch.where(amax > 0, amax / 448, torch.ones_like(amax)).float().double()
    q = (g / s).float().to(torch.float8_e4m3fn).double()
    return (q * s).reshape(x.shape)


def _w64(w, s):
    o, i = w.shape
    return (w.double().view(o // 128, 128, i // 128, 128) * s.double()[:, None, :, None]).view(o, i)


def _lin64(x, ws):
    return _q64(x) @ _w64(*ws).t()


def _rms64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, cos, sin):
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _layer64(weights, norms, x, B, T, kc, vc):
    """One dense layer: x f64 [B*T, 4096] -> (residual, mlp, k, v of the new
    positions [B, 8, T, 128]); kc, vc: cached keys and values before them."""
    n1, n2, qn, kn = norms
    h = _rms64(x, n1)
    q, k, v = (_lin64(h, weights["self_attn.%s_proj" % c]).view(B, T, -1, 128).transpose(1, 2)
               for c in "qkv")
    L = 0 if kc is None else kc.shape[2]
    cos, sin = (t[L:L + T] for t in _rotary(L + T))
    q, k = _rope64(_rms64(q, qn), cos, sin), _rope64(_rms64(k, kn), cos, sin)
    o = torch.empty_like(q)
    for h8 in range(8):
        ks = k[:, h8] if kc is None else torch.cat([kc[:, h8].double(), k[:, h8]], 1)
        vs = v[:, h8] if vc is None else torch.cat([vc[:, h8].double(), v[:, h8]], 1)
        mask = torch.ones(T, L + T, dtype=torch.bool, device=DEV).triu(L + 1)
        for i in range(4 * h8, 4 * h8 + 4):
            s = (q[:, i] @ ks.transpose(1, 2)) / math.sqrt(128)
            o[:, i] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ vs
    o = o.transpose(1, 2).reshape(B * T, 4096)
    x = x + _lin64(o, weights["self_attn.o_proj"])
    h = _rms64(x, n2)
    gate, up = _lin64(h, weights["mlp.gate_proj"]), _lin64(h, weights["mlp.up_proj"])
    return x, _lin64(gate * torch.sigmoid(gate) * up, weights["mlp.down_proj"]), k, v


def _exact_linear(case, seed):
    x, ws = _linear_inputs(case, seed)
    return _lin64(x, ws)


def _exact_step(case, seed):
    x, (kc, vc) = _step_inputs(case, seed)
    L = case["cached"]
    res, mlp, k, v = _layer64(_dense_weights(seed), _dense_norms(1, seed)[0][0], x.double(),
                              case["batch"], 1, kc[:, :, :L], vc[:, :, :L])
    return {"mlp": mlp, "residual": res, "k": k[:, :, 0], "v": v[:, :, 0]}


def _exact_prompt(case, seed):
    res, mlp, k, v = _layer64(_dense_weights(seed), _dense_norms(1, seed)[0][0],
                              _prompt_x(case, seed).double(), case["batch"], case["tokens"],
                              None, None)
    return {"mlp": mlp, "residual": res, "k": k, "v": v}


def _exact_moe(case, seed):
    x, router = _moe_inputs(case, seed)
    p = torch.softmax(x.double() @ router.double().t(), -1)
    w, idx = p.topk(MOE["top_k"], dim=-1)
    w = w / w.sum(-1, keepdim=True)
    drawn = [{n: _w64(*ws) for n, ws in ex.items()} for ex in _expert_weights(seed)]
    xq, y = _q64(x), torch.zeros(x.shape, dtype=torch.float64, device=DEV)
    for j, ex in enumerate(drawn):  # experts j, j + DISTINCT_EXPERTS, ... hold these weights
        tok, slot = torch.nonzero(idx % DISTINCT_EXPERTS == j, as_tuple=True)
        gate, up = xq[tok] @ ex["gate_proj"].t(), xq[tok] @ ex["up_proj"].t()
        out = _q64(gate * torch.sigmoid(gate) * up) @ ex["down_proj"].t()
        y.index_add_(0, tok, out * w[tok, slot][:, None])
    return {"y": y, "weights": w}


def _exact_attention(case, seed):
    qkv, qn, kn, kc, vc = _attention_inputs(case, seed)
    B, L, G = case["batch"], case["cached"], case["group"]
    hkv = 32 // G
    heads = qkv.double().view(B, 32 + 2 * hkv, 128)
    cos, sin = (t[L] for t in _rotary(L + 1))
    q = _rope64(_rms64(heads[:, :32], qn), cos, sin)
    k = _rope64(_rms64(heads[:, 32:32 + hkv], kn), cos, sin)
    v = heads[:, 32 + hkv:]
    o = torch.empty(B, 32, 128, dtype=torch.float64, device=DEV)
    for h in range(hkv):
        ks = torch.cat([kc[:, h, :L].double(), k[:, h:h + 1]], 1)
        vs = torch.cat([vc[:, h, :L].double(), v[:, h:h + 1]], 1)
        s = q[:, G * h:G * (h + 1)] @ ks.transpose(1, 2) / math.sqrt(128)
        o[:, G * h:G * (h + 1)] = torch.softmax(s, -1) @ vs
    amax = o.abs().amax(-1)
    return {"q": None, "scale": torch.where(amax > 0, amax / 448, torch.ones_like(amax)),
            "bf16": o.reshape(B, 4096), "k": k, "v": v}


def _dit_attention64(q, k, v, n_q, n_k, cos, sin):
    """q, k, v [T, 24, 128] before the head norms; n_q / n_k weight rows per token."""
    def rope(x):
        x0, x1 = x[..., 0::2], x[..., 1::2]
        return torch.stack([x0 * cos - x1 * sin, x0 * sin + x1 * cos], -1).flatten(-2)

    o = torch.empty_like(q)
    for h in range(q.shape[1]):
        qh, kh = rope(_rms64(q[:, h], n_q)), rope(_rms64(k[:, h], n_k))
        o[:, h] = torch.softmax(qh @ kh.t() / math.sqrt(128), -1) @ v[:, h]
    return o.reshape(q.shape[0], -1)


def _modulate64(x, shift, scale):
    x = (x - x.mean(-1, keepdim=True)) * torch.rsqrt(x.var(-1, unbiased=False, keepdim=True) + EPS)
    return x * (1 + scale) + shift


def _silu64(x):
    return x * torch.sigmoid(x)


def _gelu64(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _exact_dit(case, seed):
    pipe, blk = _dit_block(case, seed)
    cos, sin = (t.double()[0, 0] for t in
                pipe.dit.rope_tables(case["text"], case["grid_h"], case["grid_w"], DEV))
    img, txt, emb = (t.double()[0] for t in _dit_inputs(case, seed))
    emb = _silu64(emb)

    def lin(name, x):  # a block-scaled Linear on unquantized rows
        m = blk.get_submodule(name)
        return x @ _w64(m.weight, m.weight_scale_inv).t() + m.bias.double()

    def heads(y):
        return y.view(y.shape[0], -1, 24, 128).unbind(1)

    n_txt = txt.shape[0]
    if case["block"] == "single":
        x = torch.cat([txt, img])
        shift, scale, gate = lin("norm.linear", emb).chunk(3)
        y = lin("to_qkv_mlp", _modulate64(x, shift, scale))
        q, k, v = heads(y[:, :9216])
        o = _dit_attention64(q, k, v, blk.norm_q_a.weight, blk.norm_k_a.weight, cos, sin)
        return (x + gate * lin("proj_out", torch.cat([o, _gelu64(y[:, 9216:])], -1)))[None]

    def mod(m):
        return (emb @ m.linear.weight.double().t() + m.linear.bias.double()).chunk(6)

    at = blk.attn
    sa, ca, ga, sma, cma, gma = mod(blk.norm1_a)
    sb, cb, gb, smb, cmb, gmb = mod(blk.norm1_b)
    qa, ka, va = heads(lin("attn.a_to_qkv", _modulate64(img, sa, ca)))
    qb, kb, vb = heads(lin("attn.b_to_qkv", _modulate64(txt, sb, cb)))

    def rows(a, b):  # each token's own head-norm weight
        return torch.cat([b.weight.double().expand(n_txt, 128),
                          a.weight.double().expand(img.shape[0], 128)])

    o = _dit_attention64(torch.cat([qb, qa]), torch.cat([kb, ka]), torch.cat([vb, va]),
                         rows(at.norm_q_a, at.norm_q_b), rows(at.norm_k_a, at.norm_k_b), cos, sin)
    img = img + ga * lin("attn.a_to_out", o[n_txt:])
    txt = txt + gb * lin("attn.b_to_out", o[:n_txt])
    img = img + gma * lin("ff_a.2", _gelu64(lin("ff_a.0", _modulate64(img, sma, cma))))
    txt = txt + gmb * lin("ff_b.2", _gelu64(lin("ff_b.0", _modulate64(txt, smb, cmb))))
    return img[None], txt[None]


def _exact_model(case, seed):
    weights, (norms, last) = _dense_weights(seed), _dense_norms(case["layers"], seed)
    emb, head = _head(151936, seed)
    x, L = emb[_model_tokens(case, seed)].double(), case["cached"]
    for n, (kc, vc) in zip(norms, _model_kv(case, seed)):
        res, mlp, _, _ = _layer64(weights, n, x, case["batch"], 1, kc[:, :, :L], vc[:, :, :L])
        x = res + mlp
    return _rms64(x, last) @ head.double().t()


_EXACT = {"linear": _exact_linear, "step": _exact_step, "prompt": _exact_prompt,
          "moe_step": _exact_moe, "moe_prompt": _exact_moe, "attention": _exact_attention,
          "dit": _exact_dit, "model": _exact_model}


def exact(case, seed):
    """What ``run`` returns, in 64 bits (None where the outputs are bytes)."""
    fn = _EXACT.get(case["kind"])
    if fn is None:
        return None
    with torch.no_grad():
        return fn(case, seed)
