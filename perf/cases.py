"""The work that this package is timed on: steps of quantized decoder layers as a serving program issues them.

Every case is one step through the public layers (``DecodeStackRunner``, ``QuantDecodeLayer``, the drop-in cells,
``MoELayer``, ``MLASelfAttention``) at the model shapes of ``mindformers_amd.synthetic.CONFIGS`` and of the MoE and
multi-latent-attention benchmarks: decode steps from one sequence to 256, prompts from a few dozen rows to several
thousand, mixed steps of a chunked-prefill scheduler; int8 and 4-bit weights, int8 activations, 16-bit and int8 caches.

Lengths are ragged and fixed by the case (so that its bytes and operations are known); weights, activations, cache
contents and the placement of the cache blocks come from the seed.
"""
import numpy as np
import torch

from mindformers_amd.decode_layer import QuantDecodeLayer
from mindformers_amd.modules import InferAttention, LlamaRMSNorm, MLASelfAttention, MLATransformerConfig
from mindformers_amd.modules.layers import AllQuantLinearInferCell, WeightQuantLinearCell
from mindformers_amd.modules.moe import MoELayer, QuantGroupedMLP, SharedExpertMLP, TopKRouter
from mindformers_amd import ops
from mindformers_amd.runner import DecodeStackRunner
from mindformers_amd.synthetic import CONFIGS, rope_rows
from mindformers_amd.transformer_config import TransformerConfig

DEV = "cuda"
# DeepSeek-V3 geometry of the MoE and multi-latent-attention benchmarks
MOE = dict(hidden=7168, experts=256, ffn=2048, topk=8, groups=8, group_topk=4, scale=2.5)
MLA = dict(hidden=7168, heads=128, q_lora=1536, rank=512, nope=128, rope=64, v=128, block=128)


def listed():
    return [
        # The smallest model of the package, two fp16 layers driven by the serving runner from the scheduler's host
        # arrays: what a step costs when launches and host work are all there is.
        dict(name="tiny_stack_decode", path="stack", shape="tiny_llama_w8a16", layers=2, batch=4, lo=32, hi=256),
        # One user chatting with an 8B model in 4-bit group-128 weights, through the drop-in cells.
        dict(name="chat_w4_decode", path="cells", shape="llama3_8b_w8a16", group=128, batch=1, lo=1777, hi=1777),
        # The package's headline: a batch of 64 sequences with ragged contexts, int8 weights, bf16 cache.
        dict(name="llama_decode", path="layer", shape="llama3_8b_w8a16", batch=64, lo=512, hi=4096),
        # Few sequences over long contexts on a 70B-class layer.
        dict(name="long_decode", path="layer", shape="qwen2_5_72b_w8a16", batch=16, lo=16384, hi=32768),
        # High-throughput serving with int8 activations: 256 sequences of 2048 tokens.
        dict(name="w8a8_decode", path="layer", shape="qwen2_5_7b_w8a8", batch=256, lo=2048, hi=2048),
        # Three prompts of different lengths entering an 8B model in one step, weight-only int8.
        dict(name="llama_prefill", path="prefill", shape="llama3_8b_w8a16", prompts=3, rows=4137),
        # Two prompts entering a model with int8 activations.
        dict(name="w8a8_prefill", path="prefill", shape="qwen2_5_7b_w8a8", prompts=2, rows=1531),
        # A chunked-prefill scheduler's mixed step over an int8 cache: two 512-row chunks beside 24 decoding sequences.
        dict(name="kv8_chunked", path="chunked", shape="llama3_8b_w8a16_kv8", decodes=24, chunks=2, chunk=512, lo=512,
             hi=4096),
        # A decode step of a mixture-of-experts layer, all experts resident, weight-only int8.
        dict(name="moe_decode", path="moe", tokens=128, act="none"),
        # The same layer on a prompt's rows with int8 activations.
        dict(name="moe_prefill", path="moe", tokens=2077, act="per_token"),
        # Multi-latent attention: a decode step over the latent cache, and two prompts.
        dict(name="mla_decode", path="mla_decode", batch=64, lo=512, hi=4096),
        dict(name="mla_prefill", path="mla_prefill", prompts=2, rows=2025),
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], evenly spread over its logarithm."""
    return int(round(float(lo) * (float(hi) / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["stack", "cells", "decode", "decode", "prefill", "prefill", "chunked", "moe", "moe", "mla_decode",
                       "mla_prefill"])
    if kind == "stack":
        hi = _log(rng, 32, 512)
        return dict(path="stack", shape="tiny_llama_w8a16", layers=rng.randint(1, 3), batch=_log(rng, 1, 32),
                    lo=max(1, hi // rng.randint(1, 8)), hi=hi)
    if kind == "cells":
        hi = _log(rng, 64, 8192)
        return dict(path="cells", shape="llama3_8b_w8a16", group=rng.choice([0, 64, 128]), batch=_log(rng, 1, 32),
                    lo=max(1, hi // rng.randint(1, 4)), hi=hi)
    if kind == "decode":
        shape = rng.choice(["llama3_8b_w8a16", "llama3_8b_w8a16_kv8", "qwen2_5_7b_w8a8", "qwen2_5_72b_w8a16"])
        batch = _log(rng, 1, 256)
        hi = _log(rng, 256, min(32768, 524288 // batch))
        return dict(path="layer", shape=shape, batch=batch, lo=max(1, hi // rng.randint(1, 8)), hi=hi)
    if kind == "prefill":
        shape = rng.choice(["llama3_8b_w8a16", "qwen2_5_7b_w8a8"])
        rows = _log(rng, 65, 4200)
        return dict(path="prefill", shape=shape, prompts=rng.randint(1, 4), rows=rows)
    if kind == "chunked":
        hi = _log(rng, 1024, 8192)
        return dict(path="chunked", shape=rng.choice(["llama3_8b_w8a16_kv8", "llama3_8b_w8a16"]),
                    decodes=_log(rng, 1, 48), chunks=rng.randint(1, 2), chunk=_log(rng, 64, 1024),
                    lo=max(1, hi // rng.randint(1, 8)), hi=hi)
    if kind == "moe":
        return dict(path="moe", tokens=_log(rng, 1, 2077), act=rng.choice(["none", "per_token"]))
    if kind == "mla_decode":
        hi = _log(rng, 256, 4096)
        return dict(path="mla_decode", batch=_log(rng, 1, 64), lo=max(1, hi // rng.randint(1, 8)), hi=hi)
    return dict(path="mla_prefill", prompts=rng.randint(1, 3), rows=_log(rng, 65, 2025))


# ------------------------------------------------------------------------------------------------ sizes of a case
def _spread(n, lo, hi):
    """n ragged lengths of [lo, hi], the same for every seed (golden-ratio steps)."""
    at = ((np.arange(n) + 1) * 0.6180339887498949) % 1.0
    return (lo + np.floor(at * (hi - lo + 1))).astype(np.int64)


def _split(rows, parts):
    """rows cut into ragged parts of at least one row."""
    w = 0.25 + ((np.arange(parts) + 1) * 0.6180339887498949) % 1.0
    ends = np.floor(np.cumsum(w) / w.sum() * rows).astype(np.int64)
    ends[-1] = rows
    return np.maximum(np.diff(np.concatenate([[0], ends])), 1)


def _rows_and_lengths(case):
    """(new rows per sequence, context length per sequence with the new rows)."""
    path = case["path"]
    if path in ("prefill", "mla_prefill"):
        q = _split(case["rows"], case["prompts"])
        return q, q
    if path == "chunked":
        q = np.concatenate([np.full(case["chunks"], case["chunk"]), np.ones(case["decodes"], np.int64)])
        return q, np.maximum(_spread(len(q), case["lo"], case["hi"]), q)
    lens = _spread(case["batch"], case["lo"], case["hi"])
    return np.ones(len(lens), np.int64), lens


def work(case):
    path = case["path"]
    if path == "moe":
        h, f, e, k, t = MOE["hidden"], MOE["ffn"], MOE["experts"], MOE["topk"], case["tokens"]
        active = e * (1.0 - (1.0 - k / e) ** t)                     # experts that receive a row
        per = 3 * h * f
        return dict(bytes=(active + 1) * per + 4 * e * h + 4.0 * t * h, flops=2.0 * t * (k + 1) * per + 2.0 * t * e * h)
    q, lens = _rows_and_lengths(case)
    t = int(q.sum())
    pairs = float((q * lens - q * (q - 1) / 2).sum())               # (query row, visible key) pairs
    if path.startswith("mla"):
        c = MLA
        qd, dk = c["nope"] + c["rope"], c["rank"] + c["rope"]
        proj = c["hidden"] * (c["q_lora"] + dk) + c["q_lora"] * c["heads"] * qd + c["heads"] * c["v"] * c["hidden"]
        up = c["rank"] * c["heads"] * (c["nope"] + c["v"])
        if path == "mla_decode":
            attn, cache = 2.0 * c["heads"] * (dk + c["rank"]) * pairs, 2 * dk * int(lens.sum())
        else:
            attn, cache = 2.0 * c["heads"] * (qd + c["v"]) * pairs, 2 * dk * t
        return dict(bytes=proj + 2 * up + cache + 4.0 * t * c["hidden"], flops=2.0 * t * (proj + up) + attn)
    cfg, layers = CONFIGS[case["shape"]], case.get("layers", 1)
    h, d, nh, nkv, ffn = cfg["hidden"], cfg["head_dim"], cfg["n_head"], cfg["n_kv_head"], cfg["ffn"]
    weights = h * (nh + 2 * nkv) * d + nh * d * h + 3 * h * ffn
    esz = 1 if cfg.get("kv_int8") else 2
    wbytes = weights * (0.5 if path == "cells" else 1.0)
    return dict(bytes=layers * (wbytes + int(lens.sum()) * 2 * nkv * d * esz + 4.0 * t * h),
                flops=layers * (2.0 * t * weights + 4.0 * nh * d * pairs))


def tolerance(case):
    # Measured: a step against the same step run as two smaller ones (other split and partition plans, so sums in another
    # order).  16-bit activations: rel 2.2e-3 - 3.7e-3, max 0.013 - 0.027 (one bf16 step of a value is 2^-8 of it).
    # int8 activations: rel 0.015 - 0.022, max 0.13 - 0.14, because a one-step difference of a bf16 intermediate can move
    # its quantised value by a whole int8 step.  int8 caches: rows whose 16-bit value sits at a rounding edge.
    if "w8a8" in case.get("shape", ""):
        return dict(rel=3e-2, max=0.6)
    return dict(rel=1.5e-2, max=0.1, differ=1e-3)


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _fill(t, gen, scale=1.0, clip=None):
    """N(0, scale) values, for integers rounded and clipped to +-clip."""
    flat = t.view(-1)
    for o in range(0, flat.numel(), 1 << 27):
        part = flat[o:o + (1 << 27)]
        r = torch.randn(part.numel(), generator=gen, device=DEV)
        if clip is not None:
            r.mul_(scale).round_().clamp_(-clip, clip)
        elif scale != 1.0:
            r.mul_(scale)
        part.copy_(r)
    return t


def _scales(gen, *shape, n_in, grid=32.0):
    """Scales of weights of standard deviation ``n_in ** -0.5`` whose integers have standard deviation ``grid``."""
    return (torch.rand(*shape, generator=gen, device=DEV) * 0.4 + 0.8) * (n_in ** -0.5 / grid)


def _tables(q, lens, block, seed):
    """Shuffled cache blocks: (block table [B, max_blocks], slots of the new rows, positions, number of blocks)."""
    rng = np.random.default_rng(int(seed))
    need = (lens + block - 1) // block
    nb = int(need.sum()) + 2
    perm = rng.permutation(nb).astype(np.int32)
    tables = -np.ones((len(lens), int(need.max())), np.int32)
    at = 0
    for i, n in enumerate(need):
        tables[i, :n] = perm[at:at + n]
        at += n
    seq = np.repeat(np.arange(len(q)), q)
    pos = np.concatenate([np.arange(l - n, l) for l, n in zip(lens, q)])
    slots = tables[seq, pos // block].astype(np.int64) * block + pos % block
    return tables, slots.astype(np.int32), pos, nb


def _dense_layer(cfg, gen, qwen):
    layer = QuantDecodeLayer(cfg["hidden"], cfg["n_head"], cfg["n_kv_head"], cfg["head_dim"], cfg["ffn"], 1e-5,
                             cfg["dtype"], cfg["act_quant"], qkv_bias=qwen, device=DEV)
    for name in layer.NAMES:
        w = getattr(layer, f"{name}_w")
        _fill(w, gen, 32.0, 127)
        getattr(layer, f"{name}_s").copy_(_scales(gen, w.shape[0], n_in=w.shape[1]))
        if layer.act_quant:
            getattr(layer, f"{name}_smooth").copy_(torch.rand(w.shape[1], generator=gen, device=DEV) * 1.5 + 0.5)
    if qwen:
        layer.qkv_b.copy_(torch.randn(layer.qkv_b.shape, generator=gen, device=DEV))
    for norm in (layer.attn_norm, layer.ffn_norm):
        norm.copy_(1.0 + 0.1 * torch.randn(cfg["hidden"], generator=gen, device=DEV))
    return layer.prepare()


def _caches(cfg, nb, gen):
    shape = (nb, cfg["block_size"], cfg["n_kv_head"], cfg["head_dim"])
    if cfg.get("kv_int8"):
        return [_fill(torch.empty(shape, dtype=torch.int8, device=DEV), gen, 32.0, 127) for _ in range(2)]
    return [_fill(torch.empty(shape, dtype=cfg["dtype"], device=DEV), gen) for _ in range(2)]


def _rope(cfg, pos):
    return rope_rows(torch.from_numpy(pos).to(DEV), cfg["head_dim"], cfg["theta"], cfg["dtype"], DEV)


def _prepare_stack(case, seed, gen):
    cfg = CONFIGS[case["shape"]]
    q, lens = _rows_and_lengths(case)
    tables, slots, _, nb = _tables(q, lens, cfg["block_size"], seed)
    layers = [_dense_layer(cfg, gen, False) for _ in range(case["layers"])]
    per_block = cfg["block_size"] * cfg["n_kv_head"] * cfg["head_dim"] * 2 * 2 * case["layers"]
    runner = DecodeStackRunner(layers, (nb + 1) * per_block / 2 ** 30, 0, cfg["block_size"], cfg["theta"], device=DEV)
    for c in runner.key_cache + runner.value_cache:
        _fill(c, gen)
    x = torch.randn(len(lens), cfg["hidden"], generator=gen, device=DEV).to(cfg["dtype"])
    return dict(path="stack", runner=runner, x=x, lens=[int(l) for l in lens], tables=tables, slots=slots)


def _prepare_layer(case, seed, gen):
    cfg = CONFIGS[case["shape"]]
    q, lens = _rows_and_lengths(case)
    tables, slots, pos, nb = _tables(q, lens, cfg["block_size"], seed)
    layer = _dense_layer(cfg, gen, case["shape"].startswith("qwen"))
    if cfg.get("kv_int8"):
        layer.set_kv_quant(torch.full((2, cfg["n_kv_head"] * cfg["head_dim"]), 1.0 / 32, device=DEV))
    kc, vc = _caches(cfg, nb, gen)
    cos, sin = _rope(cfg, pos)
    starts = None
    if case["path"] != "layer":
        starts = torch.from_numpy(np.concatenate([[0], np.cumsum(q)]).astype(np.int32)).to(DEV)
    x = torch.randn(int(q.sum()), cfg["hidden"], generator=gen, device=DEV).to(cfg["dtype"])
    return dict(path="layer", layer=layer, x=x, kc=kc, vc=vc, tables=torch.from_numpy(tables).to(DEV),
                lens=torch.from_numpy(lens.astype(np.int32)).to(DEV), slots=torch.from_numpy(slots).to(DEV), cos=cos,
                sin=sin, starts=starts)


def _cell4(n_in, n_out, group, gen):
    """A 4-bit deploy cell with its checkpoint's nibbles and scales."""
    cell = WeightQuantLinearCell(n_in, n_out, device=DEV, weight_bits=4, group_size=group)
    v = _fill(torch.empty(n_out, n_in, dtype=torch.int8, device=DEV), gen, 2.0, 7)
    cell.weight.copy_((v[:, 0::2] & 15) | (v[:, 1::2] << 4))
    cell.w_scale.copy_(_scales(gen, *cell.w_scale.shape, n_in=n_in, grid=2.0))
    return cell.prepare()


def _cell8(n_in, n_out, gen, act_quant=False):
    kind = AllQuantLinearInferCell if act_quant else WeightQuantLinearCell
    cell = kind(n_in, n_out, device=DEV)
    _fill(cell.weight, gen, 32.0, 127)
    cell.w_scale.copy_(_scales(gen, n_out, n_in=n_in))
    return cell.prepare()


def _prepare_cells(case, seed, gen):
    cfg = CONFIGS[case["shape"]]
    q, lens = _rows_and_lengths(case)
    tables, slots, pos, nb = _tables(q, lens, cfg["block_size"], seed)
    h, d, nh, nkv, ffn, g = cfg["hidden"], cfg["head_dim"], cfg["n_head"], cfg["n_kv_head"], cfg["ffn"], case["group"]
    att = InferAttention(nh, d, nkv, scale_value=d ** -0.5, block_size=cfg["block_size"], num_blocks=nb,
                         rotary_cos_format=2, compute_dtype=cfg["dtype"], device=DEV)
    att.is_first_iteration = False
    mgr = att.paged_attention_mgr
    _fill(mgr.key_cache, gen)
    _fill(mgr.value_cache, gen)
    cos, sin = _rope(cfg, pos)
    norms = [LlamaRMSNorm(h, 1e-5, device=DEV) for _ in range(2)]
    for n in norms:
        n.weight.data.copy_(1.0 + 0.1 * torch.randn(h, generator=gen, device=DEV))
    return dict(path="cells", att=att, norms=norms, nq=nh * d, nkv=nkv * d, qkv=_cell4(h, (nh + 2 * nkv) * d, g, gen),
                wo=_cell4(nh * d, h, g, gen), fc1=_cell4(h, 2 * ffn, g, gen), fc2=_cell4(ffn, h, g, gen),
                x=torch.randn(len(lens), h, generator=gen, device=DEV).to(cfg["dtype"]),
                tables=torch.from_numpy(tables).to(DEV), lens=torch.from_numpy(lens.astype(np.int32)).to(DEV),
                slots=torch.from_numpy(slots).to(DEV), freqs=(cos, sin, None))


def _prepare_moe(case, seed, gen):
    m, w8a8 = MOE, case["act"] != "none"
    cfg = TransformerConfig(hidden_size=m["hidden"], num_moe_experts=m["experts"], moe_ffn_hidden_size=m["ffn"],
                            moe_shared_expert_intermediate_size=m["ffn"], shared_expert_num=1, moe_router_topk=m["topk"],
                            moe_router_num_groups=m["groups"], moe_router_group_topk=m["group_topk"],
                            moe_router_topk_scaling_factor=m["scale"], moe_router_enable_expert_bias=True)
    net = MoELayer(cfg, device="meta")                              # the float experts are never materialised
    net.router = TopKRouter(cfg, device=DEV)
    _fill(net.router.weight.data, gen, 0.01)
    net.experts = QuantGroupedMLP(m["experts"], cfg, device=DEV, act_quant="per_token" if w8a8 else None)
    for w, s in ((net.experts.weight1, net.experts.w1_scale), (net.experts.weight2, net.experts.w2_scale)):
        _fill(w, gen, 32.0, 127)
        s.copy_(_scales(gen, *s.shape, n_in=w.shape[2]))
    net.experts.prepare()
    net.experts.weight1 = net.experts.weight2 = None                # the packed copies are what the layer reads
    shared = SharedExpertMLP(cfg, device="meta")
    shared.linear_fc1 = _cell8(m["hidden"], 2 * m["ffn"], gen, w8a8)
    shared.linear_fc2 = _cell8(m["ffn"], m["hidden"], gen, w8a8)
    net.shared_experts = shared
    x = torch.randn(case["tokens"], m["hidden"], generator=gen, device=DEV).to(torch.bfloat16)
    return dict(path="moe", net=net, x=x)


def _prepare_mla(case, seed, gen):
    c = MLA
    q, lens = _rows_and_lengths(case)
    tables, slots, pos, nb = _tables(q, lens, c["block"], seed)
    cfg = MLATransformerConfig(hidden_size=c["hidden"], num_attention_heads=c["heads"], q_lora_rank=c["q_lora"],
                               kv_lora_rank=c["rank"], qk_head_dim=c["nope"], qk_pos_emb_head_dim=c["rope"],
                               v_head_dim=c["v"], layernorm_epsilon=1e-6)
    net = MLASelfAttention(cfg, device=DEV)
    for name in ("linear_qkv_down_proj", "linear_q_up_proj", "linear_proj"):
        n_out, n_in = getattr(net, name).weight.shape
        setattr(net, name, _cell8(n_in, n_out, gen))
    _fill(net.linear_kv_up_proj.weight.data, gen, c["rank"] ** -0.5)
    for norm in (net.q_layernorm, net.kv_layernorm):
        norm.weight.data.copy_(1.0 + 0.1 * torch.randn(norm.weight.shape, generator=gen, device=DEV))
    net.prepare()
    net.is_prefill = case["path"] == "mla_prefill"
    cache = _fill(torch.empty(nb, c["block"], 1, c["rank"] + c["rope"], dtype=torch.bfloat16, device=DEV), gen)
    cos, sin = net.rotary_pos_emb.get_cos_sin_for_decode(torch.from_numpy(pos).to(DEV))
    x = torch.randn(int(q.sum()), c["hidden"], generator=gen, device=DEV).to(torch.bfloat16)
    lens_t = torch.from_numpy(lens.astype(np.int32)).to(DEV)
    kw = dict(rotary_pos_cos=cos, rotary_pos_sin=sin, block_tables=torch.from_numpy(tables).to(DEV),
              slot_mapping=torch.from_numpy(slots).to(DEV), key_cache=cache, batch_valid_length=lens_t)
    if net.is_prefill:
        kw["actual_seq_qlen"] = torch.from_numpy(np.cumsum(q).astype(np.int32)).to(DEV)
    return dict(path="mla", net=net, x=x, kw=kw)


def prepare(case, seed):
    gen = _gen(seed)
    with torch.no_grad():
        kind = {"stack": _prepare_stack, "cells": _prepare_cells, "moe": _prepare_moe, "mla_decode": _prepare_mla,
                "mla_prefill": _prepare_mla}.get(case["path"], _prepare_layer)
        return kind(case, seed, gen)


# ------------------------------------------------------------------------------------------------ one step
@torch.no_grad()
def run(s):
    path = s["path"]
    if path == "layer":
        out = s["layer"](s["x"], s["kc"], s["vc"], s["tables"], s["lens"], s["slots"], s["cos"], s["sin"],
                         q_starts=s["starts"])
        return out, s["kc"], s["vc"]
    if path == "stack":
        r = s["runner"]
        out = r.forward(s["x"], s["lens"], s["tables"], s["slots"], prefill=False)
        return out, r.key_cache, r.value_cache
    if path == "cells":
        qkv = s["qkv"](s["norms"][0](s["x"]))
        nq, nkv = s["nq"], s["nkv"]
        a = s["att"](qkv[:, :nq], qkv[:, nq:nq + nkv], qkv[:, nq + nkv:], s["lens"], s["tables"], s["slots"], s["freqs"])
        h = s["wo"](a, residual=s["x"])
        out = s["fc2"](ops.silu_mul(s["fc1"](s["norms"][1](h))), residual=h)
        return out, s["att"].paged_attention_mgr.key_cache, s["att"].paged_attention_mgr.value_cache
    if path == "moe":
        return s["net"](s["x"])
    return s["net"](s["x"], **s["kw"]), s["kw"]["key_cache"]
