"""Performance cases: the work a filter or a join has this framework do.

Each case is one block of the Qwen3 fp8 forward pass, called through the
engine's own entry points as `Qwen3Pipeline.forward_chunk` calls them, or a
whole (shallow) forward pass with its readout:

  mlp      post-attention norm + quant, gate_up with the SiLU gate, down
  attn     input norm + quant, the qkv projection with q/k norm and rotary,
           the KV write, attention and the output projection, over a packed
           chunk:
             "fresh"  rows of a filter's first question: document + question,
                      behind an instruction whose pages the rows share
             "later"  a later question over documents already in the arena
             "join"   partner rows under resident anchors, tree attention
  forward  a whole chunk through several layers, and its answer logits
  readout  the final norm of the answer rows and their TRUE/FALSE scores

Geometries are Qwen3-4B and Qwen3-32B; sizes run from one short row to the
Qwen3-4B chunk budget.
"""

import math
from dataclasses import replace

import numpy as np
import torch

from quail_amd import kernels, loop
from quail_amd.arena import KVArena
from quail_amd.model import (SYNTHETIC_FALSE_IDS, SYNTHETIC_TRUE_IDS, build_random_qwen3)
from quail_amd.qwen3 import Qwen3Pipeline
from quail_amd.readout import AnswerRows
from quail_amd.specs import QWEN3_4B_FP8, QWEN3_32B_FP8

VOCAB = 32768   # covers the answer ids; the embedding's size does not change a pass
SPECS = {"4b": replace(QWEN3_4B_FP8, vocab=VOCAB), "32b": replace(QWEN3_32B_FP8, vocab=VOCAB)}
PAGE = 16


def listed():
    return [
        # one short row with its question: a filter over a handful of rows, or
        # the last row of a table
        dict(name="mlp one row", kind="mlp", model="4b", tokens=41, ue8m0=False),
        # a few rows: the end of a table, a selective later stage
        dict(name="mlp few rows", kind="mlp", model="4b", tokens=1157, ue8m0=False),
        # the GEMM sweep's size
        dict(name="mlp chunk", kind="mlp", model="4b", tokens=16384, ue8m0=False),
        # the large model, power-of-two scales, a handful of short rows
        dict(name="mlp 32b ue8m0", kind="mlp", model="32b", tokens=611, ue8m0=True),
        # one row of a filter behind a short instruction
        dict(name="attn one row", kind="attn", model="4b", path="fresh", rows=1, prefix=64, lo=150,
             hi=210, tail=24, ue8m0=False, pick=1),
        # the prefix-shared layer: 64 rows behind 256 shared tokens
        dict(name="attn shared prefix", kind="attn", model="4b", path="fresh", rows=64, prefix=256,
             lo=32, hi=256, tail=24, ue8m0=False, pick=2),
        # a full chunk of the 4,096-row filter
        dict(name="attn chunk", kind="attn", model="4b", path="fresh", rows=400, prefix=64, lo=100,
             hi=360, tail=24, ue8m0=False, pick=3),
        # the second question over a few long kept documents, the large model
        dict(name="attn later 32b", kind="attn", model="32b", path="later", rows=8, prefix=64,
             lo=1024, hi=4096, tail=24, ue8m0=False, pick=4),
        # the second question over the survivors of a chunk
        dict(name="attn later rows", kind="attn", model="4b", path="later", rows=300, prefix=64,
             lo=30, hi=500, tail=24, ue8m0=False, pick=5),
        # a join chunk: each anchor's partners behind its resident document
        dict(name="attn join", kind="attn", model="4b", path="join", rows=6, partners=40,
             prefix=48, lo=60, hi=240, tail=16, ue8m0=False, pick=6),
        # a whole small call: one row through four layers to its logits
        dict(name="forward one row", kind="forward", model="4b", layers=4, rows=1, prefix=16, lo=24,
             hi=48, tail=24, ue8m0=False, pick=7),
        # the answer rows of a full chunk
        dict(name="readout chunk", kind="readout", model="4b", rows=409),
    ]


def _spread(rng, lo, hi):
    """A whole number in [lo, hi], even over its logarithm."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "mlp", "attn", "attn", "attn", "attn", "forward", "readout"])
    model = rng.choice(["4b", "4b", "32b"])
    ue8m0 = rng.random() < 0.25
    pick = rng.randrange(1 << 20)
    if kind == "mlp":
        return dict(kind="mlp", model=model, tokens=_spread(rng, 1, 16384 if model == "4b" else 4096),
                    ue8m0=ue8m0)
    if kind == "readout":
        return dict(kind="readout", model=model, rows=_spread(rng, 1, 512))
    if kind == "forward":
        return dict(kind="forward", model="4b", layers=rng.randint(2, 4), rows=_spread(rng, 1, 24),
                    prefix=rng.randint(8, 96), lo=16, hi=rng.randint(48, 300),
                    tail=rng.randint(8, 40), ue8m0=ue8m0, pick=pick)
    path = rng.choice(["fresh", "fresh", "later", "later", "join"])
    case = dict(kind="attn", model=model, path=path, prefix=rng.randint(16, 256),
                tail=rng.randint(8, 40), ue8m0=ue8m0, pick=pick)
    if path == "fresh":
        if model == "4b":
            case.update(rows=_spread(rng, 1, 256), lo=rng.randint(16, 128), hi=rng.randint(160, 400))
        else:
            case.update(rows=_spread(rng, 1, 6), lo=rng.randint(200, 1024), hi=rng.randint(1100, 3000))
    elif path == "later":
        if model == "4b":
            case.update(rows=_spread(rng, 1, 400), lo=rng.randint(16, 128), hi=rng.randint(160, 1024))
        else:
            case.update(rows=_spread(rng, 1, 64), lo=rng.randint(200, 1024), hi=rng.randint(1100, 4096))
    else:
        case.update(rows=_spread(rng, 1, 8), partners=_spread(rng, 4, 48),
                    lo=rng.randint(16, 64), hi=rng.randint(80, 260))
        if model == "32b":
            case.update(rows=_spread(rng, 1, 4), partners=_spread(rng, 4, 16))
    return case


# ---- inputs ---------------------------------------------------------------

def _lengths(case):
    """Tokens of each document (behind the shared instruction), from the case alone."""
    rng = np.random.default_rng(case["pick"])
    own = rng.integers(case["lo"], case["hi"] + 1, size=case["rows"])
    partners = None
    if case.get("path") == "join":
        partners = rng.integers(case["lo"], case["hi"] + 1, size=case["partners"])
    return own.tolist(), partners


def _activations(gen, rows, width):
    """A residual stream: channels of unequal strength, bf16."""
    strength = torch.exp(0.5 * torch.randn(width, generator=gen, device="cuda"))
    x = torch.randn(rows, width, generator=gen, device="cuda") * strength
    return x.to(torch.bfloat16)


def _model(case, layers, seed):
    spec = SPECS[case["model"]]
    model = build_random_qwen3(spec, seed=seed, device="cuda", layers=layers,
                               ue8m0=case.get("ue8m0", False))
    gen = torch.Generator(device="cuda").manual_seed(seed + 7)
    norms = [model.model.norm]
    for layer in model.model.layers:
        norms += [layer.input_layernorm, layer.post_attention_layernorm,
                  layer.self_attn.q_norm, layer.self_attn.k_norm]
    for norm in norms:
        w = 1 + 0.1 * torch.randn(norm.weight.numel(), generator=gen, device="cuda")
        norm.weight = w.to(torch.bfloat16)
    return spec, model


def _chunk(case, spec, layers, seed):
    """The arena and one packed chunk, as the filter and join loops pack them."""
    rng = np.random.default_rng(seed)
    ids = lambda n: rng.integers(0, VOCAB, size=int(n), dtype=np.int64)  # noqa: E731
    own, partners = _lengths(case)
    prefix, tail = case["prefix"], case["tail"]
    shared = prefix // PAGE * PAGE
    room = sum(-(-(prefix + n + tail) // PAGE) for n in own) + 4
    if partners is not None:
        room = sum(-(-(prefix + n) // PAGE) for n in own) + 4
    arena = KVArena(layers, room, PAGE, spec.n_kv, spec.d_head, dtype=torch.bfloat16,
                    device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(seed + 3)
    for pool in arena.k + arena.v:   # resident keys are normed: unit variance
        pool.normal_(generator=gen)
    instruction, groups, keys = ids(prefix), [], []
    question = ids(tail)
    for i, n in enumerate(own):
        key, length = ("d", i), prefix + n
        capacity = length if partners is not None else length + tail
        borrow = (("d", 0), shared) if i and shared and partners is None else None
        if arena.activate(key, length, capacity_tokens=capacity, borrow=borrow) is None:
            raise RuntimeError("the arena is too small for the case")
        keys.append(key)
        if partners is not None:
            groups.append(dict(key=key, prefix=None, f=length,
                               suffixes=[np.concatenate([ids(p), question]) for p in partners]))
        elif case.get("path") == "later":
            groups.append(dict(key=key, prefix=None, f=length, suffixes=[question]))
        else:
            start = shared if borrow else 0
            doc = np.concatenate([instruction, ids(n)])[start:]
            groups.append(dict(key=key, prefix=doc, start=start, f=length, suffixes=[question]))
    mode = "tree" if partners is not None else "unified"
    return arena, loop.pack_chunk(torch, arena, groups, attention_mode=mode)


def prepare(case, seed):
    kind = case["kind"]
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    state = dict(kind=kind)
    if kind == "readout":
        spec, model = _model(case, 0, seed)
        rows = case["rows"]
        tokens = 2 * rows
        state.update(rows=AnswerRows(torch, model, SYNTHETIC_TRUE_IDS, SYNTHETIC_FALSE_IDS),
                     norm=model.model.norm, model=model,
                     hidden=_activations(gen, tokens, spec.hidden),
                     residual=_activations(gen, tokens, spec.hidden),
                     index=torch.randperm(tokens, generator=gen, device="cuda")[:rows])
        return state
    if kind == "forward":
        spec, model = _model(case, case["layers"], seed)
        # a trained model's residual stream is large beside what one layer
        # adds to it; the random init's embedding (0.02) is not
        model.model.embed_tokens.weight = 8 * _activations(gen, VOCAB, spec.hidden)
        arena, chunk = _chunk(case, spec, case["layers"], seed)
        pipeline = Qwen3Pipeline(model, arena, spec=spec, ue8m0=case["ue8m0"])
        state.update(model=model, pipeline=pipeline, chunk=chunk, arena=arena,
                     rows=AnswerRows(torch, model, SYNTHETIC_TRUE_IDS, SYNTHETIC_FALSE_IDS))
        return state
    spec, model = _model(case, 1, seed)
    if kind == "mlp":
        arena = KVArena(1, 1, PAGE, spec.n_kv, spec.d_head, dtype=torch.bfloat16, device="cuda")
        tokens = case["tokens"]
    else:
        arena, chunk = _chunk(case, spec, 1, seed)
        state.update(chunk=chunk)
        tokens = chunk.tokens
    pipeline = Qwen3Pipeline(model, arena, spec=spec, ue8m0=case["ue8m0"])
    state.update(model=model, engine=pipeline.engine, layer=pipeline.layers[0], arena=arena,
                 hidden=_activations(gen, tokens, spec.hidden))
    if kind == "mlp":
        state["residual"] = _activations(gen, tokens, spec.hidden)
    return state


# ---- one pass ---------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "readout":
        normed = kernels.final_norm(state["hidden"], state["residual"], state["index"],
                                    state["norm"].weight, state["norm"].variance_epsilon)
        best_true, best_false = state["rows"].logits(normed)
        bits, margin = state["rows"].bits(normed, with_margin=True)
        return [normed, best_true, best_false, bits, margin]
    if kind == "forward":
        normed = state["pipeline"].forward_chunk(state["chunk"])
        best_true, best_false = state["rows"].logits(normed)
        return [normed, best_true, best_false]
    engine, layer, hidden = state["engine"], state["layer"], state["hidden"]
    if kind == "mlp":
        # the residual stream is updated in place, as in the layer loop
        g_in, g_scale = engine.norm_quant(hidden, layer.post_attention_layernorm,
                                          state["residual"])
        d_in, d_scale = engine.gemm_silu_quant(g_in, g_scale, layer.mlp.gate_up_proj)
        return [engine.gemm(d_in, d_scale, layer.mlp.down_proj, "down"), state["residual"]]
    chunk, attn = state["chunk"], layer.self_attn
    chunk.meta["layer"] = 0
    q_in, q_scale = engine.norm_quant(hidden, layer.input_layernorm)
    o_in, o_scale = engine.qkv_project_attention(q_in, q_scale, attn, chunk.positions, chunk)
    out = engine.gemm(o_in, o_scale, attn.o_proj, "o")
    return [out, state["arena"].k[0], state["arena"].v[0]]


# ---- what a pass cannot do without -------------------------------------------

def _attn_work(case, spec):
    """(chunk tokens, (query, key) pairs, arena tokens read) of a chunk."""
    own, partners = _lengths(case)
    prefix, tail = case["prefix"], case["tail"]
    shared = prefix // PAGE * PAGE
    tokens = pairs = kv = 0
    for i, n in enumerate(own):
        length = prefix + n
        if partners is not None:
            kv += length
            for p in partners:
                c = int(p) + tail
                tokens += c
                pairs += c * length + c * (c + 1) // 2
            continue
        end = length + tail
        c = tail if case.get("path") == "later" else end - (shared if i else 0)
        tokens += c
        pairs += c * (end - c) + c * (c + 1) // 2
        kv += (end - c) if case.get("path") == "later" else 0
    return tokens, pairs, kv


def work(case):
    spec = SPECS[case["model"]]
    H, I, qkv = spec.hidden, spec.intermediate, spec.qkv_width
    q_width, kv_width = spec.n_q * spec.d_head, spec.n_kv * spec.d_head
    if case["kind"] == "readout":
        rows, n_ans = case["rows"], len(SYNTHETIC_TRUE_IDS) + len(SYNTHETIC_FALSE_IDS)
        return dict(bytes=rows * (3 * 2 * H + 9) + n_ans * 2 * H, flops=2 * rows * H * n_ans)
    mlp_weights, attn_weights = 3 * H * I, H * (qkv + q_width)
    if case["kind"] == "mlp":
        T = case["tokens"]
        return dict(bytes=mlp_weights + T * H * 2 * 4, flops=2 * T * mlp_weights)
    T, pairs, kv = _attn_work(case, spec)
    attn_bytes = attn_weights + 2 * 2 * kv_width * (kv + T)
    attn_flops = 2 * T * attn_weights + 4 * spec.n_q * spec.d_head * pairs
    if case["kind"] == "attn":
        return dict(bytes=attn_bytes + T * H * 2 * 2, flops=attn_flops)
    rows, L = case["rows"], case["layers"]
    # the last layer's output projection and MLP are needed at the answer rows only
    last = rows * (H * q_width + mlp_weights)
    flops = L * attn_flops + (L - 1) * 2 * T * mlp_weights - 2 * T * H * q_width + 2 * last
    return dict(bytes=L * (attn_bytes + mlp_weights) + T * H * 2 + rows * H * 2, flops=flops)


def tolerance(case):
    # fp8 activations are requantized inside a block: a value that another
    # summation order moves across a rounding boundary changes its e4m3 code
    # by one step. Answer bits may differ where two scores tie.
    # Attention computed by torch in fp32 over the same q, k and v (another
    # summation order, P not rounded) moves the attention block's output by
    # 0.9-1.2 % and the three-launch tree form by 1.7 %.
    if case["kind"] == "readout":
        return dict(rel=0.01, max=0.5, differ=0.005)
    if case["kind"] == "mlp":
        return dict(rel=0.01, max=0.5)
    return dict(rel=0.03, max=0.9)


# ---- the same in 64 bits -----------------------------------------------------

def _quant64(x, ue8m0):
    """1x128 e4m3 groups and their scales, multiplied out again."""
    g = x.view(x.shape[0], -1, 128)
    scale = g.abs().amax(-1, keepdim=True).clamp(min=1e-10) / 448.0
    if ue8m0:
        scale = torch.exp2(torch.ceil(torch.log2(scale)))
    q = (g / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return (q.double() * scale).view_as(x)


def _linear64(x, lin):
    w = lin.weight.double()
    s = lin.weight_scale.double().repeat_interleave(128, 0).repeat_interleave(128, 1)
    return x @ (w * s).t()


def _norm64(x, norm):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + norm.variance_epsilon) \
        * norm.weight.double()


def _rope64(x, cache, positions):
    cs = cache[positions].double()[:, None, :]
    cos, sin = cs[..., :64], cs[..., 64:]
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _softmax_rows64(q, k, v, lim):
    """q [c, n_q, d] over k, v [L, n_kv, d]; row i sees its first lim[i] keys."""
    c, n_q, d = q.shape
    n_kv = k.shape[1]
    qh = q.view(c, n_kv, n_q // n_kv, d).permute(1, 2, 0, 3)
    s = torch.matmul(qh.reshape(n_kv, -1, d), k.permute(1, 2, 0).contiguous()) / math.sqrt(d)
    s = s.view(n_kv, n_q // n_kv, c, -1)
    hidden = torch.arange(k.shape[0], device=q.device)[None, :] >= lim[:, None]
    p = torch.softmax(s.masked_fill(hidden, -math.inf), -1)
    o = torch.matmul(p.view(n_kv, -1, p.shape[-1]), v.permute(1, 0, 2).contiguous())
    return o.view(n_kv, n_q // n_kv, c, d).permute(2, 0, 1, 3).reshape(c, n_q * d)


def _attention64(chunk, x, layer, k_rows, v_rows, ue8m0, n_q, n_kv):
    """The attention block; k_rows / v_rows are the arena's rows, updated."""
    attn = layer.self_attn
    T = x.shape[0]
    qkv = _linear64(_quant64(_norm64(x, layer.input_layernorm), ue8m0), attn.qkv_proj)
    qkv = qkv.view(T, n_q + 2 * n_kv, 128)
    cache = attn.rotary_emb.cos_sin_cache
    q = _rope64(_norm64(qkv[:, :n_q], attn.q_norm), cache, chunk.positions)
    k = _rope64(_norm64(qkv[:, n_q:n_q + n_kv], attn.k_norm), cache, chunk.positions)
    v = qkv[:, n_q + n_kv:]
    out = torch.empty(T, n_q * 128, dtype=torch.float64, device=x.device)
    slot = torch.arange(PAGE, device=x.device)

    def resident(table, used):
        rows = (table.long()[:, None] * PAGE + slot).view(-1)[:used]
        return k_rows[rows], v_rows[rows]

    meta = chunk.meta
    if chunk.attention_mode == "tree":
        cu, reads = meta["cu_a"].tolist(), meta["reads"]
        which, used = meta["a_read"].tolist(), reads["used"].tolist()
        for s, (lo, hi) in enumerate(zip(cu, cu[1:])):
            kr, vr = resident(reads["table"][which[s]], used[which[s]])
            lim = kr.shape[0] + 1 + torch.arange(hi - lo, device=x.device)
            out[lo:hi] = _softmax_rows64(q[lo:hi], torch.cat([kr, k[lo:hi]]),
                                         torch.cat([vr, v[lo:hi]]), lim)
    else:
        u = meta["unified"]
        k_rows[u["dst"]], v_rows[u["dst"]] = k[u["src"]], v[u["src"]]
        cu, used = u["cu_q"].tolist(), u["used"].tolist()
        for s, (lo, hi) in enumerate(zip(cu, cu[1:])):
            kr, vr = resident(u["table"][s], used[s])
            lim = used[s] - (hi - lo) + 1 + torch.arange(hi - lo, device=x.device)
            out[lo:hi] = _softmax_rows64(q[lo:hi], kr, vr, lim)
    return _quant64(out, ue8m0)


def _mlp64(x, layer, ue8m0):
    gu = _linear64(_quant64(_norm64(x, layer.post_attention_layernorm), ue8m0),
                   layer.mlp.gate_up_proj)
    gate, up = gu.chunk(2, -1)
    return _linear64(_quant64(gate * torch.sigmoid(gate) * up, ue8m0), layer.mlp.down_proj)


def _pool_rows64(arena, layer):
    """One layer's pools as (arena row, head, element), 64 bits."""
    pages, n_kv = arena.k[layer].shape[:2]
    return (arena.k[layer].double().permute(0, 2, 1, 3).reshape(pages * PAGE, n_kv, 128),
            arena.v[layer].double().permute(0, 3, 1, 2).reshape(pages * PAGE, n_kv, 128))


def exact(case, seed):
    state = prepare(case, seed)
    spec = SPECS[case["model"]]
    if case["kind"] == "readout":
        x = (state["hidden"].double() + state["residual"].double())[state["index"]]
        normed = _norm64(x, state["norm"])
        best = _best64(normed, state["rows"])
        return [normed, best[0], best[1], None, None]
    ue8m0 = case["ue8m0"]
    if case["kind"] == "mlp":
        x = state["hidden"].double() + state["residual"].double()
        return [_mlp64(x, state["layer"], ue8m0), x]
    chunk, arena = state["chunk"], state["arena"]
    if case["kind"] == "attn":
        k_rows, v_rows = _pool_rows64(arena, 0)
        o = _attention64(chunk, state["hidden"].double(), state["layer"], k_rows, v_rows, ue8m0,
                         spec.n_q, spec.n_kv)
        pages = arena.n_pages
        return [_linear64(o, state["layer"].self_attn.o_proj),
                k_rows.view(pages, PAGE, spec.n_kv, 128).permute(0, 2, 1, 3),
                v_rows.view(pages, PAGE, spec.n_kv, 128).permute(0, 2, 3, 1)]
    pipeline = state["pipeline"]
    x = pipeline.embed.weight[chunk.input_ids].double()
    for i, layer in enumerate(pipeline.layers):
        k_rows, v_rows = _pool_rows64(arena, i)
        o = _attention64(chunk, x, layer, k_rows, v_rows, ue8m0, spec.n_q, spec.n_kv)
        x = x + _linear64(o, layer.self_attn.o_proj)
        x = x + _mlp64(x, layer, ue8m0)
    normed = _norm64(x[chunk.final_indices], pipeline.final_norm)
    best = _best64(normed, state["rows"])
    return [normed, best[0], best[1]]


def _best64(normed, rows):
    scores = normed @ rows.weights.double().t()
    true = rows.is_true.bool()
    return scores[:, true].amax(-1), scores[:, ~true].amax(-1)
