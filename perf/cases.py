"""Performance cases of the paged GPT-2 engine: its layers and whole steps, through the entry points a program calls.

GPT-2 124M in fp32 (12 layers, 768 wide, 12 heads of 64 dims, 50,257 tokens) over a paged pool of 12
layers, block size 16 unless a case says otherwise. ``listed()`` gives the cases, ``draw(rng)`` more of the same ranges;
``prepare`` makes what a program holds before the call, ``run`` is one pass, ``work`` what the pass
cannot do without, ``exact`` its result in float64 and ``tolerance`` how far a correct fp32
implementation may be from another one.

Kinds:

* ``attend``: one layer's paged attention for a step (``PagedBatch.attend``): the step's K/V written
  to the pool, decode rows and / or prompts and chunks attended.
* ``attention``: the whole attention layer (``Attention.forward``): QKV projection, attend, output
  projection.
* ``mlp``: the MLP (``MLP.forward``).
* ``head``: ``ln_f`` and the tied LM head over a small decode batch (``ops.skinny_linear``).
* ``decode_step``: a whole decode step replayed from its captured graph (``DecodeGraphs.forward``).
* ``prefill_step``: a whole prefill step (``paged_forward``).
"""

import math
import random

import torch

from tokquay_amd import GPT2, BlockAllocator, GPT2Config, Sequence, cdiv, ops
from tokquay_amd.generate import paged_forward
from tokquay_amd.graphs import DecodeGraphs
from tokquay_amd.model import MLP, Attention

CFG = GPT2Config()
C, H, L, V = CFG.n_embd, CFG.n_head, CFG.n_layer, CFG.vocab_size
D = CFG.d_head
DEVICE = "cuda"


def _attend(name, decode=0, ctx_lo=1, ctx_hi=1, prompts=0, new_lo=1, new_hi=1, start=0, block_size=16, kind="attend"):
    """``decode`` sequences feeding one token at contexts ctx_lo..ctx_hi (the new token included), and
    ``prompts`` sequences feeding new_lo..new_hi tokens each behind ``start`` cached ones."""
    case = {"kind": kind, "decode": decode, "ctx_lo": ctx_lo, "ctx_hi": ctx_hi, "prompts": prompts, "new_lo": new_lo,
            "new_hi": new_hi, "start": start, "block_size": block_size}  # fmt: skip
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # One user chatting: a single sequence part-way through its answer. Launch and latency count.
        _attend("decode_attention_1", decode=1, ctx_lo=301, ctx_hi=301),
        # The decode attention operation at the size this repository's benchmark measures alone.
        _attend("decode_attention_64", decode=64, ctx_lo=16, ctx_hi=512),
        # A full decode batch in one attention layer: 256 sequences of contexts up to the model's 1,024.
        _attend("attention_layer_decode_256", decode=256, ctx_lo=257, ctx_hi=1023, kind="attention"),
        # Chunked prefill of long prompts: four 256-token chunks behind 512 cached tokens.
        _attend("prefill_attention_chunks", prompts=4, new_lo=256, new_hi=256, start=512),
        # A large admission: 32 whole prompts of ragged lengths in one step.
        _attend("prefill_attention_32", prompts=32, new_lo=256, new_hi=1023),
        # A chunked-prefill step: chunks of new prompts beside 128 decoding sequences.
        _attend("mixed_attention", decode=128, ctx_lo=129, ctx_hi=639, prompts=4, new_lo=250, new_hi=256, start=256),
        # Attention layer of an ordinary prefill step: prompts that fill the 2,048-token step budget.
        _attend("attention_layer_prefill", prompts=13, new_lo=17, new_hi=255, kind="attention"),
        # MLP of the full decode batch.
        {"name": "mlp_256", "kind": "mlp", "rows": 256},
        # MLP of an ordinary prefill step under the 2,048-token budget (packed rows: any count).
        {"name": "mlp_1987", "kind": "mlp", "rows": 1987},
        # LM head of a small decode batch.
        {"name": "head_8", "kind": "head", "rows": 8},
        # A whole decode step of a lightly loaded server, logits out (sampling requests).
        _attend("decode_step_8", decode=8, ctx_lo=301, ctx_hi=420, kind="decode_step"),
        # A whole prefill step: a few new prompts, next-token logits out.
        _attend("prefill_step", prompts=7, new_lo=33, new_hi=511, kind="prefill_step"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attend", "attend", "attend", "attention", "attention", "mlp", "mlp", "head", "decode_step", "prefill_step"])
    if kind == "mlp":
        return {"kind": "mlp", "rows": _log_int(rng, 33, 2048)}
    if kind == "head":
        return {"kind": "head", "rows": rng.randint(1, 16)}
    case = _attend(None, kind=kind)
    if kind == "prefill_step":
        form = "prompts"
    elif kind == "decode_step":
        form = "decode"
    else:
        form = rng.choice(["decode", "prompts", "chunks", "mixed"])
        case["block_size"] = rng.choice([16, 16, 16, 32, 8])
    if form in ("decode", "mixed"):
        case["decode"] = _log_int(rng, 1, {"decode_step": 32, "attend": 256, "attention": 256}[kind])
        case["ctx_lo"] = _log_int(rng, 2, 600)
        case["ctx_hi"] = rng.randint(case["ctx_lo"], 1023)
    if form != "decode":
        case["start"] = 0 if form == "prompts" else rng.randint(1, 700)
        case["new_lo"] = _log_int(rng, 2, 256)
        case["new_hi"] = rng.randint(case["new_lo"], min(1023 - case["start"], 4 * case["new_lo"]))
        budget = 16384 if kind == "attend" and form == "prompts" else 2048  # tokens of the step
        case["prompts"] = _log_int(rng, 1, max(1, min(32, budget // case["new_hi"])))
    return case


# ------------------------------------------------------------------------------------------ shapes
def _spread(n, lo, hi, salt):
    """n lengths spread evenly over lo..hi, in a fixed shuffled order."""
    got = [lo + int((hi - lo + 1) * (i + 0.5) / n) for i in range(n)]
    random.Random(salt).shuffle(got)
    return got


def _lengths(case):
    """(cached, fed) token counts of each sequence of the step, decode rows first."""
    ctx = _spread(case["decode"], case["ctx_lo"], case["ctx_hi"], 1)
    new = _spread(case["prompts"], case["new_lo"], case["new_hi"], 2)
    return [c - 1 for c in ctx] + [case["start"]] * len(new), [1] * len(ctx) + new


def _rows(case):
    return case["rows"] if "rows" in case else sum(_lengths(case)[1])


# ------------------------------------------------------------------------------------------ inputs
def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal_(module, gen):
    """Random-init weights: matrices N(0, 0.02), LayerNorm gains near 1, biases small."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            p.normal_(0.0, 0.02, generator=gen)
            if "ln_" in name and name.endswith("weight"):
                p.add_(1.0)
    return module.requires_grad_(False)


def _sequences(case, seed, allocator):
    """The step's sequences with their cached K/V in the pool, their blocks interleaved as sequences
    that grew side by side have them."""
    cached, fed = _lengths(case)
    rng = random.Random(seed)
    seqs = []
    for i, (c, n) in enumerate(zip(cached, fed)):
        ids = [rng.randrange(V) for _ in range(c + n)]
        seqs.append(Sequence(i, ids, num_cached_tokens=c))
    grow = [s for s in seqs for _ in range(cdiv(s.num_tokens, case["block_size"]))]
    rng.shuffle(grow)
    for s in grow:  # one block at a time
        allocator.append_slot(s, (len(s.block_table) + 1) * case["block_size"])
    return seqs


def _allocator(case, gen, layers):
    """A pool with room to spare, the K/V of ``layers`` filled."""
    blocks = sum(cdiv(c + n, case["block_size"]) for c, n in zip(*_lengths(case)))
    alloc = BlockAllocator(CFG, blocks + 8, block_size=case["block_size"], device=DEVICE)
    for layer in layers:
        alloc.pool[:, layer].normal_(generator=gen)
    return alloc


LAYER = 5  # the layer whose attention the attend and attention cases run


def prepare(case, seed):
    gen = _generator(seed)
    kind = case["kind"]
    if kind == "mlp":
        mlp = _normal_(MLP(CFG).to(DEVICE), gen)
        return {"case": case, "mlp": mlp, "x": torch.randn(case["rows"], C, device=DEVICE, generator=gen)}
    if kind == "head":
        model = _normal_(GPT2(GPT2Config(n_layer=0)).to(DEVICE), gen)
        return {"case": case, "model": model, "x": torch.randn(case["rows"], C, device=DEVICE, generator=gen) * 3}
    if kind in ("attend", "attention"):
        alloc = _allocator(case, gen, [LAYER])
        seqs = _sequences(case, seed, alloc)
        batch = alloc.batch_for(seqs)
        state = {"case": case, "alloc": alloc, "batch": batch, "tables": [s.block_table for s in seqs]}
        if kind == "attend":
            state["qkv"] = torch.randn(batch.num_tokens, 3 * C, device=DEVICE, generator=gen)
        else:
            state["attention"] = _normal_(Attention(CFG).to(DEVICE), gen)
            state["x"] = torch.randn(batch.num_tokens, C, device=DEVICE, generator=gen)
        return state
    alloc = _allocator(case, gen, range(L))
    state = {"case": case, "alloc": alloc, "seqs": _sequences(case, seed, alloc)}
    with torch.device(DEVICE):
        model = GPT2(CFG)
    state["model"] = _normal_(model, gen)
    state["cached"] = [s.num_cached_tokens for s in state["seqs"]]
    if kind == "decode_step":
        state["graphs"] = DecodeGraphs(state["model"], alloc, len(state["seqs"]))
        run(state)  # a server captures a batch size's graph once
    return state


@torch.no_grad()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "mlp":
        return state["mlp"](state["x"])
    if kind == "head":
        m = state["model"]
        return ops.skinny_linear(state["x"], m.wte.weight, None, ln=(m.ln_f.weight, m.ln_f.bias, m.ln_f.eps))
    if kind == "attend":
        out = state["batch"].attend(LAYER, state["qkv"])
        return {"out": out, "pool": state["alloc"].pool[:, LAYER]}
    if kind == "attention":
        out = state["attention"](state["x"], state["batch"], LAYER)
        return {"out": out, "pool": state["alloc"].pool[:, LAYER]}
    for s, n in zip(state["seqs"], state["cached"]):  # the step again from the same cache
        s.num_cached_tokens = n
    if kind == "decode_step":
        logits = state["graphs"].forward(state["seqs"])
    else:
        logits = paged_forward(state["model"], state["alloc"], state["seqs"])
    return {"logits": logits, "pool": state["alloc"].pool}


# ------------------------------------------------------------------------------------------ work
def work(case):
    """Each input read once, each output written once (fp32), and the causal-exact flops."""
    kind, n = case["kind"], _rows(case)
    if kind == "mlp":
        return {"bytes": 4 * (8 * C * C + 5 * C + 2 * n * C), "flops": 16 * n * C * C}
    if kind == "head":
        return {"bytes": 4 * (V * C + 2 * C + n * C + n * V), "flops": 2 * n * V * C}
    cached, fed = _lengths(case)
    scores = sum(c * m + m * (m + 1) // 2 for c, m in zip(cached, fed))  # (query, visible key) pairs
    kv_read = 2 * sum(c for c in cached) * C  # the cached K/V; the new rows come with the input
    kv_written = 2 * n * C
    tables = sum(cdiv(c + m, case["block_size"]) for c, m in zip(cached, fed)) + 4 * len(fed)
    attend_floats, attend_flops = kv_read + kv_written + tables, 4 * C * scores
    if kind == "attend":
        return {"bytes": 4 * (attend_floats + 4 * n * C), "flops": attend_flops}
    if kind == "attention":
        return {"bytes": 4 * (attend_floats + 4 * C * C + 4 * C + 2 * n * C), "flops": attend_flops + 8 * n * C * C}
    weights = L * (12 * C * C + 13 * C) + V * C + 2 * C
    return {"bytes": 4 * (L * attend_floats + weights + 2 * n * C + len(fed) * V),
            "flops": L * (attend_flops + 24 * n * C * C) + 2 * len(fed) * V * C}  # fmt: skip


def tolerance(case):
    """fp32 throughout: about four times what the path was measured to differ from float64 (relative
    2-norm: 1.4e-7 to 1.1e-6 in one layer, up to 1.7e-6 through all twelve)."""
    if case["kind"] in ("decode_step", "prefill_step"):
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 4e-6, "max": 4e-5}


# ------------------------------------------------------------------------------------------ float64
def _layer_norm(x, ln):
    return torch.nn.functional.layer_norm(x, (C,), ln.weight.double(), ln.bias.double(), ln.eps)


def _linear(x, lin):
    return x @ lin.weight.double().t() + lin.bias.double()


def _mlp(x, mlp):
    return _linear(torch.nn.functional.gelu(_linear(x, mlp.c_fc), approximate="tanh"), mlp.c_proj)


def _causal(tables, cached, fed, bs, kv, qkv, order):
    """Textbook attention of each sequence's new rows; ``kv`` ``[blocks, 2, H, bs, D]`` float64 gets the
    new K/V. ``order``: the sequences in the order their rows are packed."""
    out = qkv.new_empty(qkv.size(0), C)
    at = 0
    for b in order:
        c, n = cached[b], fed[b]
        q, k, v = qkv[at : at + n].view(n, 3, H, D).unbind(1)
        pos = torch.arange(c + n, device=qkv.device)
        blk, off = torch.tensor(tables[b], device=qkv.device)[pos // bs], pos % bs
        kv[blk[c:], 0, :, off[c:]] = k
        kv[blk[c:], 1, :, off[c:]] = v
        keys, vals = kv[blk, 0, :, off], kv[blk, 1, :, off]  # [ctx, H, D]
        visible = pos[None, :] <= (c + torch.arange(n, device=qkv.device))[:, None]
        for h in range(H):
            s = (q[:, h] @ keys[:, h].t()) / math.sqrt(D)
            out[at : at + n, h * D : (h + 1) * D] = torch.softmax(s.masked_fill(~visible, -math.inf), -1) @ vals[:, h]
        at += n
    return out


def _packed_order(fed):
    """One-token rows are packed first, then the prompts (PagedBatch's row order)."""
    return [b for b, n in enumerate(fed) if n == 1] + [b for b, n in enumerate(fed) if n > 1]


@torch.no_grad()
def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "mlp":
        return _mlp(state["x"].double(), state["mlp"])
    if kind == "head":
        m = state["model"]
        return _layer_norm(state["x"].double(), m.ln_f) @ m.wte.weight.double().t()
    cached, fed = _lengths(case)
    order, bs = _packed_order(fed), case["block_size"]
    if kind in ("attend", "attention"):
        tables = state["tables"]
        kv = state["alloc"].pool[:, LAYER].double()
        if kind == "attend":
            return {"out": _causal(tables, cached, fed, bs, kv, state["qkv"].double(), order), "pool": kv}
        at = state["attention"]
        a = _causal(tables, cached, fed, bs, kv, _linear(state["x"].double(), at.c_attn), order)
        return {"out": _linear(a, at.c_proj), "pool": kv}
    m, seqs = state["model"], state["seqs"]
    pool = state["alloc"].pool.double()
    ids = [t for b in order for t in seqs[b].token_ids[cached[b] : cached[b] + fed[b]]]
    pos = [p for b in order for p in range(cached[b], cached[b] + fed[b])]
    x = m.wte.weight[torch.tensor(ids, device=DEVICE)].double() + m.wpe.weight[torch.tensor(pos, device=DEVICE)].double()
    for i, block in enumerate(m.h):
        qkv = _linear(_layer_norm(x, block.ln_1), block.attn.c_attn)
        x = x + _linear(_causal([s.block_table for s in seqs], cached, fed, bs, pool[:, i], qkv, order), block.attn.c_proj)
        x = x + _mlp(_layer_norm(x, block.ln_2), block.mlp)
    last, at = [0] * len(fed), 0
    for b in order:
        at += fed[b]
        last[b] = at - 1
    h = _layer_norm(x[torch.tensor(last, device=DEVICE)], m.ln_f)
    return {"logits": h @ m.wte.weight.double().t(), "pool": pool}
