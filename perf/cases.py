"""The work that a user of this package has it do, as cases that can be timed.

A case names a kind, a model shape and sizes; `prepare` builds what a program holds before
the call (weights, caches, plans, captured graphs, the step's inputs), `run` makes one pass
through the package's entry points, `exact` computes the same in 64 bits with plain torch.

Kinds:
  attention     one decoder layer's attention in a prefill: Attention.forward_rope (rotation of q
                and k, the KV store, varlen attention), over the paged cache for warm requests
                and over the fresh keys at ratio 0.
  layer         one whole DecoderLayer of a warm prefill (norms, projections, attention, MLP).
  decode_layer  one whole DecoderLayer of a decode step, captured as a HIP graph as the engine
                captures its decode steps.
  decode_step   a decode step of a model of a few layers through its LM head: logits.
  reuse         the all-layer copy of cached image KV with the keys re-rotated.
  vision        the vision tower with a few blocks, from pixels to embeddings.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from vlcache_amd import kernels
from vlcache_amd.config import QWEN25_VL_3B, QWEN25_VL_7B, load_model_config
from vlcache_amd.hotpath import WarmPrefillHotPath
from vlcache_amd.layers.attention import Attention
from vlcache_amd.qwen_vl import DecoderLayer, Qwen2_5_VLForConditionalGeneration, random_init_
from vlcache_amd.utils.context import reset_context, set_context
from vlcache_amd.vision import VisionTransformer, vision_config
from vlcache_amd.workloads import BLOCK_SIZE, ModelShape, WarmRequest, Workload, attention_flops

HEAD_DIM = 128
SECTION = (16, 24, 24)
MODELS = {"3b": dict(heads=16, kv=2, hidden=2048, inter=11008, layers=36, config=QWEN25_VL_3B),
          "7b": dict(heads=28, kv=4, hidden=3584, inter=18944, layers=28, config=QWEN25_VL_7B)}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # A short warm request: a 1k-token image with a little text around it; launches and latency count.
        dict(name="attention-1k-image", kind="attention", model="3b", requests=1, prefix=64, rows=32, cols=32,
             second=False, suffix=32, ratio=0.1),
        # The headline request: a 4K image, a tenth of it recomputed, the rest reused from the cache.
        dict(name="attention-4k-image", kind="attention", model="3b", requests=1, prefix=128, rows=77, cols=137,
             second=False, suffix=64, ratio=0.1),
        # A batch of four requests with two images each on the larger model, hardly anything recomputed.
        dict(name="attention-7b-two-images", kind="attention", model="7b", requests=4, prefix=64, rows=77, cols=137,
             second=True, suffix=64, ratio=0.02),
        # The first time an image is seen: the whole prompt is computed, causally, over fresh keys.
        dict(name="attention-cold-4k", kind="attention", model="3b", requests=1, prefix=128, rows=77, cols=137,
             second=False, suffix=64, ratio=0.0),
        # A decoder layer of the headline request: projections and MLP around the attention.
        dict(name="layer-4k-image", kind="layer", model="3b", requests=1, prefix=128, rows=77, cols=137,
             second=False, suffix=64, ratio=0.1),
        # Decoding behind the two-image batch: few rows, long contexts.
        dict(name="decode-7b-4x13k", kind="decode_layer", model="7b", batch=4, context=13435, max_len=16384),
        # Decoding for many users with short chats: more rows than one tile of them, short contexts.
        dict(name="decode-7b-32x2k", kind="decode_layer", model="7b", batch=32, context=2048, max_len=4096),
        # One user's decode step to its logits: the smallest work per launch.
        dict(name="decode-step-3b", kind="decode_step", model="3b", layers=4, batch=1, context=1183, max_len=4096),
        # Reusing the headline request's image in all layers at another position.
        dict(name="reuse-4k-image", kind="reuse", model="3b", layers=36, requests=1, prefix=128, rows=77, cols=137,
             second=False, suffix=64, ratio=0.1),
        # The vision tower on a 4K image, blocks that attend within windows (28 of the 32).
        dict(name="vision-4k-windows", kind="vision", rows=154, cols=274, blocks=2, full_every=0),
        # The same image, a block that attends over the whole image (4 of the 32).
        dict(name="vision-4k-whole", kind="vision", rows=154, cols=274, blocks=1, full_every=1),
        # A small image through eight blocks, the eighth over the whole image as in the public configuration.
        dict(name="vision-1k-image", kind="vision", rows=64, cols=64, blocks=8, full_every=8),
    ]


def _log(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(("attention", "attention", "layer", "decode_layer", "decode_layer", "decode_step", "reuse",
                       "vision", "vision"))
    model = rng.choice(("3b", "7b"))
    if kind in ("attention", "layer", "reuse"):
        ratio = rng.choice((0.02, 0.05, 0.1, 0.2, 0.2 if kind == "layer" else 0.5))
        if kind == "attention" and rng.random() < 0.25:
            ratio = 0.0
        case = dict(kind=kind, model=model, requests=_log(rng, 1, 4), prefix=_log(rng, 4, 512),
                    rows=_log(rng, 6, 77), cols=_log(rng, 6, 137), second=rng.random() < 0.2,
                    suffix=_log(rng, 1, 256), ratio=ratio)
        if kind == "reuse":
            case["layers"] = rng.choice((4, 12, MODELS[model]["layers"]))
        return case
    if kind == "decode_layer":
        batch = _log(rng, 1, 64)
        context = _log(rng, 64, min(16384, 131072 // batch))
        return dict(kind=kind, model=model, batch=batch, context=context,
                    max_len=4096 if context <= 4096 else 16384)
    if kind == "decode_step":
        return dict(kind=kind, model="3b", layers=rng.choice((2, 4)), batch=_log(rng, 1, 12),
                    context=_log(rng, 64, 8192), max_len=8192)
    whole = rng.random() < 0.5
    rows, cols = 2 * _log(rng, 3, 60 if whole else 77), 2 * _log(rng, 3, 100 if whole else 137)
    blocks = rng.choice((1, 2, 3))
    return dict(kind=kind, rows=rows, cols=cols, blocks=blocks, full_every=blocks if whole else 0)


# ------------------------------------------------------------------ inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _workload(case):
    m = MODELS[case["model"]]
    image = ("image", (case["rows"], case["cols"]))
    layout = [("text", case["prefix"]), image, ("text", case["suffix"])]
    if case["second"]:  # a smaller image and a line of text in front
        layout = [("text", case["prefix"]), ("image", (max(3, case["rows"] // 2), max(3, case["cols"] // 2))),
                  ("text", 64), image, ("text", case["suffix"])]
    shape = ModelShape(case["model"], case.get("layers", 1), m["heads"], m["kv"], HEAD_DIM, m["hidden"])
    request = WarmRequest(ratio=case["ratio"], cached_prefix=40, layout=tuple(layout))
    return Workload("case", shape, [request] * case["requests"])


def _model_config(case, layers):
    return load_model_config(dict(MODELS[case["model"]]["config"], num_hidden_layers=layers, vision_config=None))


def _built(make, seed):
    """A module in bf16 on the GPU with seeded N(0, 0.02) weights, as the model runner builds its model."""
    before = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device("cuda"):
            module = make()
    finally:
        torch.set_default_dtype(before)
    random_init_(module, seed=seed)
    return module.eval()


def _prefill_context(hp):
    set_context(True, hp.cu_q, hp.cu_k, 0, 0, hp.slot_mapping, None, hp.block_tables if hp.paged else None,
                attn_plan=hp.plan, cu_seqlens_q_host=hp.cu_q_host, cu_seqlens_k_host=hp.cu_k_host)


def _decode_inputs(case, seed, layers):
    """Ragged contexts (3/4 of the case's to all of it), their cache pages in a random order, the
    step's index arrays and its plan."""
    m = MODELS[case["model"]]
    b, g = case["batch"], torch.Generator().manual_seed(seed)
    lens = case["context"] - torch.arange(b) * 7919 % (case["context"] // 4 + 1)
    width = -(-case["max_len"] // BLOCK_SIZE)
    pages = -(-lens // BLOCK_SIZE)
    order = torch.randperm(int(pages.sum()), generator=g).to(torch.int32)
    table = torch.full((b, width), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(pages.tolist()):
        table[i, :n] = order[at:at + n]
        at += n
    last = lens - 1
    slots = table[torch.arange(b), last // BLOCK_SIZE] * BLOCK_SIZE + last % BLOCK_SIZE
    cache = torch.randn(2, layers, int(pages.sum()), BLOCK_SIZE, m["kv"], HEAD_DIM, generator=_generator(seed),
                        device="cuda", dtype=torch.bfloat16)
    plan = kernels.plan_decode(b, m["heads"], m["kv"], HEAD_DIM, BLOCK_SIZE, case["max_len"], "cuda")
    return SimpleNamespace(lens=lens.to(torch.int32).cuda(), table=table.cuda(), slots=slots.to(torch.int32).cuda(),
                           positions=last.repeat(3, 1).cuda(), cache=cache, plan=plan, max_len=case["max_len"])


def _decode_context(s):
    set_context(False, None, None, 1, s.max_len, s.slots, s.lens, s.table, decode_plan=s.plan)


def _captured(call):
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    reset_context()
    return graph, out


@torch.inference_mode()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "vision":
        cfg = vision_config(dict(depth=case["blocks"], fullatt_block_indexes=_whole_blocks(case)), 2048)
        tower = _built(lambda: VisionTransformer(cfg), seed)
        pixels = torch.randn(case["rows"] * case["cols"], tower.patch_dim, generator=_generator(seed + 1),
                             device="cuda", dtype=torch.bfloat16)
        return SimpleNamespace(kind=kind, tower=tower, pixels=pixels, grids=[(1, case["rows"], case["cols"])])
    m = MODELS[case["model"]]
    if kind in ("attention", "layer", "reuse"):
        hp = WarmPrefillHotPath(_workload(case), "cuda", seed=seed)
        s = SimpleNamespace(kind=kind, hp=hp)
        if kind == "attention":
            s.attn = Attention(m["heads"], HEAD_DIM, HEAD_DIM ** -0.5, m["kv"])
            s.attn.k_cache, s.attn.v_cache = hp.kv_cache[0, 0], hp.kv_cache[1, 0]
        elif kind == "layer":
            s.layer = _built(lambda: DecoderLayer(_model_config(case, 1)), seed)
            s.layer.self_attn.attn.k_cache, s.layer.self_attn.attn.v_cache = hp.kv_cache[0, 0], hp.kv_cache[1, 0]
            s.hidden, s.residual = torch.randn(2, hp.n_computed, m["hidden"], generator=_generator(seed + 1),
                                               device="cuda", dtype=torch.bfloat16).unbind(0)
        return s
    if kind == "decode_layer":
        s = _decode_inputs(case, seed, 1)
        s.kind = kind
        s.layer = _built(lambda: DecoderLayer(_model_config(case, 1)), seed)
        s.layer.self_attn.attn.k_cache, s.layer.self_attn.attn.v_cache = s.cache[0, 0], s.cache[1, 0]
        s.hidden, s.residual = torch.randn(2, case["batch"], m["hidden"], generator=_generator(seed + 1),
                                           device="cuda", dtype=torch.bfloat16).unbind(0)
        _decode_context(s)
        s.graph, s.out = _captured(lambda: s.layer(s.positions, s.hidden, s.residual))
        return s
    assert kind == "decode_step"
    s = _decode_inputs(case, seed, case["layers"])
    s.kind = kind
    s.model = _built(lambda: Qwen2_5_VLForConditionalGeneration(_model_config(case, case["layers"])), seed)
    for i, layer in enumerate(s.model.model.layers):
        layer.self_attn.attn.k_cache, layer.self_attn.attn.v_cache = s.cache[0, i], s.cache[1, i]
    s.ids = torch.randint(0, 150000, (case["batch"],), generator=_generator(seed + 1), device="cuda")
    _decode_context(s)
    s.graph, s.out = _captured(lambda: s.model(s.ids, s.positions))
    return s


# ------------------------------------------------------------------ one pass
@torch.inference_mode()
def run(s):
    if s.kind == "attention":
        _prefill_context(s.hp)
        o = s.attn.forward_rope(s.hp.positions, s.hp.q_in, s.hp.k_in, s.hp.v, s.hp.rope)
        return o, s.attn.k_cache, s.attn.v_cache
    if s.kind == "layer":
        _prefill_context(s.hp)
        hidden, residual = s.layer(s.hp.positions, s.hidden, s.residual)
        return hidden, residual, s.hp.kv_cache
    if s.kind == "decode_layer":
        s.graph.replay()
        return s.out[0], s.out[1], s.cache
    if s.kind == "decode_step":
        s.graph.replay()
        set_context(False)
        return s.model.compute_logits(s.out), s.cache
    if s.kind == "reuse":
        hp = s.hp
        kernels.rerotate_copy_kv(hp.kv_cache, hp.old_slots, hp.new_slots, hp.cos_sin, hp.seg)
        return hp.kv_cache
    return s.tower(s.pixels, s.grids)


# ------------------------------------------------------------------ what a pass cannot do without
def _layer_params(m):
    qkv = (m["heads"] + 2 * m["kv"]) * HEAD_DIM
    return m["hidden"] * (qkv + m["heads"] * HEAD_DIM + 3 * m["inter"])


def _prefill_work(case):
    m, wl = MODELS[case["model"]], _workload(case)
    n, length = wl.requests[0].n_computed * case["requests"], wl.requests[0].length * case["requests"]
    qkv, kv_row = (m["heads"] + 2 * m["kv"]) * HEAD_DIM * 2, m["kv"] * HEAD_DIM * 2 * 2
    context = length * kv_row if case["ratio"] > 0 else 0
    cos_sin_and_indices = n * (HEAD_DIM * 4 + 28)
    attn = dict(bytes=n * (qkv + m["heads"] * HEAD_DIM * 2 + kv_row) + context + cos_sin_and_indices,
                flops=attention_flops(*wl.cu_seqlens(), m["heads"], HEAD_DIM))
    return m, n, attn


def work(case):
    kind = case["kind"]
    if kind == "attention":
        return _prefill_work(case)[2]
    if kind == "layer":
        m, n, attn = _prefill_work(case)
        context = attn["bytes"] - n * (m["heads"] * 2 + 2 * m["kv"]) * HEAD_DIM * 2
        return dict(bytes=_layer_params(m) * 2 + 4 * n * m["hidden"] * 2 + context,
                    flops=2 * n * _layer_params(m) + attn["flops"])
    if kind in ("decode_layer", "decode_step"):
        m, b = MODELS[case["model"]], case["batch"]
        tokens = case["context"] * (1 + (b - 1) * 7 / 8)
        layers = case.get("layers", 1)
        params = layers * _layer_params(m)
        rows = 4 * b * m["hidden"] * 2
        if kind == "decode_step":
            params += m["hidden"] * m["config"]["vocab_size"]
            rows = b * m["config"]["vocab_size"] * 2
        return dict(bytes=params * 2 + layers * tokens * m["kv"] * HEAD_DIM * 2 * 2 + rows,
                    flops=2 * b * params + layers * 4 * tokens * m["heads"] * HEAD_DIM)
    if kind == "reuse":
        m, wl = MODELS[case["model"]], _workload(case)
        n = wl.requests[0].n_reused * case["requests"]
        return dict(bytes=n * (case["layers"] * m["kv"] * HEAD_DIM * 2 * 2 * 2 + 20), flops=0)
    n, dim, inter, pixel = case["rows"] * case["cols"], 1280, 3420, 1176
    params = case["blocks"] * dim * (4 * dim + 3 * inter) + pixel * dim + (4 * dim) ** 2 / 4 + dim * 2048
    pairs = sum((n * n if i in _whole_blocks(case) else _window_pairs(case)) for i in range(case["blocks"]))
    weights = case["blocks"] * dim * (4 * dim + 3 * inter) + pixel * dim + (4 * dim) ** 2 + 4 * dim * 2048
    return dict(bytes=2 * weights + n * pixel * 2 + n // 4 * 2048 * 2, flops=2 * n * params + 4 * pairs * dim)


def _whole_blocks(case):
    return [i for i in range(case["blocks"]) if case["full_every"] and (i + 1) % case["full_every"] == 0]


def _window_pairs(case):
    def sides(n):
        return [min(8, n - i) for i in range(0, n, 8)]
    return sum(r * r for r in sides(case["rows"])) * sum(c * c for c in sides(case["cols"]))


def tolerance(case):
    # bf16 in and out with 32-bit sums.  Measured against exact(): 0.0027 for an attention layer (the
    # roundings of q, k and the probabilities), 0.005 for a decoder layer, 0.013 for the logits of four
    # layers, 0.0007 for the re-rotated keys, 0.005 to 0.011 for one to eight vision blocks.  Two correct
    # implementations differ by up to twice that, the short ones by more where their sums' order differs.
    return {"attention": {"rel": 1e-2}, "layer": {"rel": 1.5e-2}, "decode_layer": {"rel": 1.5e-2},
            "decode_step": {"rel": 2.5e-2}, "reuse": {"rel": 3e-3}, "vision": {"rel": 2.5e-2}}[case["kind"]]


# ------------------------------------------------------------------ the same in 64 bits
def _turn(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _inv_freq(width, theta):
    return 1.0 / (theta ** (torch.arange(0, width, 2, dtype=torch.float32, device="cuda") / width))


def _rope64(x, positions):
    section = torch.repeat_interleave(torch.arange(3, device="cuda"), torch.tensor(SECTION, device="cuda"))
    angle = (positions.float()[section].t() * _inv_freq(HEAD_DIM, 1e6)).double()[:, None]
    return _turn(x.double(), angle.cos(), angle.sin())


def _attend64(q, k, v, scale, causal):
    """q [n, H, d] against k, v [m, Hkv, d]; causal: the last query sees every key."""
    (n, heads, _), m, group = q.shape, k.shape[0], q.shape[1] // k.shape[1]
    out = torch.empty(n, heads, v.shape[2], dtype=torch.float64, device="cuda")
    for h in range(heads):
        keys, values = k[:, h // group].double().t().contiguous(), v[:, h // group].double().contiguous()
        for a in range(0, n, 2048):
            score = q[a:a + 2048, h].double() @ keys * scale
            if causal:
                row = torch.arange(a, a + score.shape[0], device="cuda")[:, None]
                score.masked_fill_(torch.arange(m, device="cuda") > row + m - n, -math.inf)
            out[a:a + 2048, h] = torch.softmax(score, dim=-1) @ values
    return out


def _prefill64(hp, q, k, v):
    """(attention output, caches after the store) of a prefill's q, k, v rows before the rotation."""
    q, k, v = _rope64(q, hp.positions), _rope64(k, hp.positions), v.double()
    kc, vc = hp.kv_cache[0, 0].double(), hp.kv_cache[1, 0].double()
    kc.view(-1, *kc.shape[2:])[hp.slot_mapping.long()] = k
    vc.view(-1, *vc.shape[2:])[hp.slot_mapping.long()] = v
    out, cu_q, cu_k = [], hp.cu_q_host, hp.cu_k_host
    for i in range(len(cu_q) - 1):
        a, e, m = cu_q[i], cu_q[i + 1], cu_k[i + 1] - cu_k[i]
        if hp.paged:
            pages = hp.block_tables[i, :-(-m // BLOCK_SIZE)].long()
            keys, values = (c[pages].flatten(0, 1)[:m] for c in (kc, vc))
        else:
            keys, values = k[a:e], v[a:e]
        out.append(_attend64(q[a:e], keys, values, HEAD_DIM ** -0.5, True))
    return torch.cat(out), kc, vc


def _decode64(s, q, k, v, cache):
    q, k, v = _rope64(q, s.positions), _rope64(k, s.positions), v.double()
    kc, vc = cache[0].double(), cache[1].double()
    kc.view(-1, *kc.shape[2:])[s.slots.long()] = k
    vc.view(-1, *vc.shape[2:])[s.slots.long()] = v
    out = []
    for i, m in enumerate(s.lens.tolist()):
        pages = s.table[i, :-(-m // BLOCK_SIZE)].long()
        keys, values = (c[pages].flatten(0, 1)[:m] for c in (kc, vc))
        out.append(_attend64(q[i:i + 1], keys, values, HEAD_DIM ** -0.5, True))
    return torch.cat(out), kc, vc


def _norm64(x, module):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + module.eps) * module.weight.double()


def _linear64(x, module):
    y = x @ module.weight.double().t()
    return y if module.bias is None else y + module.bias.double()


def _mlp64(x, mlp):
    gate, up = _linear64(x, mlp.gate_up_proj).chunk(2, dim=-1)
    return _linear64(torch.nn.functional.silu(gate) * up, mlp.down_proj)


def _layer64(layer, hidden, residual, attend):
    residual = hidden if residual is None else hidden + residual
    a = layer.self_attn
    qkv = _linear64(_norm64(residual, layer.input_layernorm), a.qkv_proj)
    q, k, v = (t.unflatten(-1, (-1, HEAD_DIM)) for t in qkv.split([a.q_size, a.kv_size, a.kv_size], dim=-1))
    o, kc, vc = attend(q, k, v)
    residual = residual + _linear64(o.flatten(1), a.o_proj)
    return _mlp64(_norm64(residual, layer.post_attention_layernorm), layer.mlp), residual, kc, vc


def _vision64(case, tower, pixels):
    rows, cols, heads, width = case["rows"], case["cols"], tower.cfg.num_heads, tower.head_dim
    # Patches come merged unit by merged unit (2 x 2 patches each), units row by row.
    unit_r, unit_c, i, j = torch.meshgrid(*(torch.arange(n, device="cuda") for n in (rows // 2, cols // 2, 2, 2)),
                                          indexing="ij")
    r, c = (2 * unit_r + i).flatten(), (2 * unit_c + j).flatten()
    window = (r // 8) * (-(-cols // 8)) + c // 8
    # The published model rounds the angles, and their cosines and sines, to bf16.
    inv = _inv_freq(width // 2, 1e4)
    angle = torch.cat((r[:, None] * inv, c[:, None] * inv), dim=-1).bfloat16()
    cos, sin = angle.cos().double()[:, None], angle.sin().double()[:, None]
    x = _linear64(pixels.double(), tower.patch_embed)
    order = torch.argsort(window, stable=True)
    sizes = torch.bincount(window)
    starts = torch.cumsum(sizes, 0) - sizes
    for b, block in enumerate(tower.blocks):
        qkv = _linear64(_norm64(x, block.norm1), block.attn.qkv).unflatten(-1, (3, heads, width))
        q, k, v = _turn(qkv[:, 0], cos, sin), _turn(qkv[:, 1], cos, sin), qkv[:, 2]
        if b in _whole_blocks(case):
            o = _attend64(q, k, v, width ** -0.5, False)
        else:
            o = torch.empty_like(q)
            for size in sizes.unique().tolist():  # all windows of one size together
                at = order[starts[sizes == size][:, None] + torch.arange(size, device="cuda")]
                qw, kw, vw = (t[at].transpose(1, 2).contiguous() for t in (q, k, v))
                p = torch.softmax(qw @ kw.transpose(-1, -2).contiguous() * width ** -0.5, dim=-1)
                o[at] = (p @ vw).transpose(1, 2)
        x = x + _linear64(o.flatten(1), block.attn.proj)
        x = x + _mlp64(_norm64(x, block.norm2), block.mlp)
    x = _norm64(x, tower.merger.ln_q).view(-1, tower.merger.hidden)
    return _linear64(torch.nn.functional.gelu(_linear64(x, tower.merger.mlp[0])), tower.merger.mlp[2])


@torch.inference_mode()
def exact(case, seed):
    s = prepare(case, seed)
    if s.kind == "attention":
        return _prefill64(s.hp, s.hp.q_in, s.hp.k_in, s.hp.v)
    if s.kind == "layer":
        hidden, residual, kc, vc = _layer64(s.layer, s.hidden.double(), s.residual.double(),
                                            lambda q, k, v: _prefill64(s.hp, q, k, v))
        return hidden, residual, torch.stack((kc, vc)).unsqueeze(1)
    if s.kind == "decode_layer":
        hidden, residual, kc, vc = _layer64(s.layer, s.hidden.double(), s.residual.double(),
                                            lambda q, k, v: _decode64(s, q, k, v, s.cache[:, 0]))
        return hidden, residual, torch.stack((kc, vc)).unsqueeze(1)
    if s.kind == "decode_step":
        model, residual, caches = s.model.model, None, []
        hidden = model.embed_tokens.weight[s.ids].double()
        for i, layer in enumerate(model.layers):
            hidden, residual, kc, vc = _layer64(layer, hidden, residual,
                                                lambda q, k, v, i=i: _decode64(s, q, k, v, s.cache[:, i]))
            caches.append(torch.stack((kc, vc)))
        logits = _linear64(_norm64(hidden + residual, model.norm), s.model.lm_head)
        return logits, torch.stack(caches, dim=1)
    if s.kind == "reuse":
        hp = s.hp
        out = hp.kv_cache.double()
        flat = out.flatten(2, 3)
        delta = torch.tensor([d[0] for d in hp.deltas], device="cuda", dtype=torch.float32)[hp.seg.long()]
        angle = (delta[:, None] * _inv_freq(HEAD_DIM, 1e6)).double()[:, None]
        moved = flat[:, :, hp.old_slots]
        flat[0][:, hp.new_slots] = _turn(moved[0], angle.cos(), angle.sin())
        flat[1][:, hp.new_slots] = moved[1]
        return out
    return _vision64(case, s.tower, s.pixels)
