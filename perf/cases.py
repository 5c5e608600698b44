"""The workloads whose speed this framework answers for, through the entry points its users call.

A pass is one forward of a few attention layers in model order: anchor layers (which form and pool
the scores and select) and the reuse layers behind them, in the proportion of the schedule the
framework ships head maps for (anchors 0, 2, 8, 13, 14 of 32 layers).  Four kinds:

* ``hf_prefill`` / ``hf_decode`` -- ``EfficientKascadeStrategy.attention_forward`` as a transformers
  model calls it, layer by layer: a whole prompt, or one new token against a contiguous cache.
* ``stack_prefill`` -- a prompt in chunks through ``KascadeAttentionStack.prefill_chunk`` (paged cache).
* ``stack_decode`` -- a token through ``KascadeAttentionStack``, eager or as a captured graph.
* ``paged_decode`` -- a serving engine's step over ``PagedKascadeDecoder``: the scheduler knows the
  lengths, sequences differ in length, the launches append the new rows.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from kascade_amd import budgets
from kascade_amd.stack import KascadeAttentionStack
from kascade_amd.strategy import EfficientKascadeStrategy, PagedKascadeDecoder, get_head_mapping

ANCHORS = (0, 2, 8, 13, 14)
MODEL = "Meta-Llama-3.1-8B-Instruct"      # whose head maps ship with the package (32 layers, 8 KV heads)
DEVICE = "cuda"
PAGE = 16
HEADROOM = 64                             # decode steps before a sequence goes back to its first length
# (query heads, KV heads, head_dim): the reference's shape, the benchmark's two others, the small one
SHAPES = ((32, 8, 128), (64, 8, 128), (28, 4, 128), (8, 2, 64))


def _case(name, kind, tokens, batch=1, layers=8, shape=SHAPES[0], dtype="float16", percent=10, rolling=True, **more):
    return dict(more, name=name, kind=kind, tokens=tokens, batch=batch, layers=layers, heads=shape[0],
                kv_heads=shape[1], head_dim=shape[2], dtype=dtype, percent=percent, rolling=rolling)


def listed():
    return [
        # a chat turn's prompt: everything is latency
        _case("hf_prefill_517", "hf_prefill", 517),
        # an ordinary document prompt, in the type most checkpoints come in
        _case("hf_prefill_4096_bf16", "hf_prefill", 4096, dtype="bfloat16"),
        # two prompts of an odd length at a model shape with seven query heads per KV head
        _case("hf_prefill_2x3001_28x4_bf16", "hf_prefill", 3001, batch=2, shape=SHAPES[2], dtype="bfloat16"),
        # the headline prompt length
        _case("hf_prefill_32768", "hf_prefill", 32768),
        # the longest prompt: beyond 65536 tokens the anchors pool and select in pieces
        _case("hf_prefill_131072", "hf_prefill", 131072),
        # a prompt entering a paged cache chunk by chunk
        _case("stack_prefill_16384_by_2048", "stack_prefill", 16384, layers=4, chunk=2048),
        # generation with a transformers cache: the first tokens after a short prompt, and deep into
        # a long chain of thought
        _case("hf_decode_700", "hf_decode", 700),
        _case("hf_decode_16001_bf16", "hf_decode", 16001, dtype="bfloat16"),
        # one user's generation over a paged cache, the step of a 24-layer model captured as a graph
        _case("stack_decode_16384_graph", "stack_decode", 16384, layers=24, graph=True),
        # a small serving batch launched eagerly at a larger model's shape
        _case("stack_decode_8x3000_64x8", "stack_decode", 3000, batch=8, shape=SHAPES[1], graph=False),
        # full serving batches at long context: equal lengths, and four documents of very different length
        _case("paged_decode_16x65536", "paged_decode", 65536, batch=16, spread=1.0),
        _case("paged_decode_4_ragged_524288", "paged_decode", 524288, batch=4, spread=0.25),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("hf_prefill", "hf_prefill", "hf_decode", "hf_decode", "stack_prefill", "stack_decode", "paged_decode"))
    shape = rng.choice((SHAPES[0], SHAPES[0], SHAPES[0]) + SHAPES[1:])
    more = {}
    if kind == "hf_prefill":
        tokens, batch = _log_int(rng, 160, 131072), rng.choice((1, 1, 1, 2, 3))
    elif kind == "hf_decode":
        tokens, batch = _log_int(rng, 160, 131072), rng.choice((1, 1, 1, 2, 4))
    elif kind == "stack_prefill":
        # up to eight chunks, the last one cut anywhere
        chunk = more["chunk"] = rng.choice((512, 1024, 2048, 4096))
        tokens, batch = chunk * rng.randint(1, 8) - rng.choice((0, rng.randrange(chunk // 2))), rng.choice((1, 1, 2))
    elif kind == "stack_decode":
        more["graph"] = rng.random() < 0.5
        tokens, batch = _log_int(rng, 300, 65536), _log_int(rng, 1, 16)
    else:
        more["spread"] = rng.choice((1.0, 0.5, 0.25, 0.1))
        tokens, batch = _log_int(rng, 2048, 524288), _log_int(rng, 2, 32)
    case = _case("", kind, tokens, batch=batch, layers=4 if kind == "stack_prefill" else rng.choice((4, 8)), shape=shape,
                 dtype=rng.choice(("float16", "bfloat16")), percent=rng.choice((5, 10, 10, 20)),
                 rolling=rng.random() < 0.8, **more)
    del case["name"]
    # no drawn case is larger than the largest listed one of its direction
    prefill, decode = listed()[4], listed()[11]
    top = _cost(prefill if "prefill" in kind else decode)
    while _cost(case) > top:
        case["tokens"] //= 2
    return case


# ----------------------------------------------------------------------------------- inputs
def _dtype(case):
    return torch.float16 if case["dtype"] == "float16" else torch.bfloat16


def _lengths(case):
    """The lengths of a ragged batch: falling geometrically from ``tokens`` to ``spread * tokens``."""
    B, n, spread = case["batch"], case["tokens"], case.get("spread", 1.0)
    return [max(1, int(n * spread ** (b / max(1, B - 1)))) for b in range(B)]


def _normal(gen, shape, dtype, mean=0.0):
    return torch.empty(shape, device=DEVICE, dtype=dtype).normal_(mean, 1.0, generator=gen)


def _peak(gen, keys, sinks):
    """Keys as attention meets them: every token's keys share a component out of four directions, so
    that some tokens score high for every query, and the first token of a sequence is a sink.
    keys [rows, heads, D] or any view of it; in place."""
    dirs = torch.randn(4, keys.shape[-1], device=DEVICE, generator=gen) * 2.0
    for s in range(0, keys.shape[0], 1 << 18):
        part = keys[s:s + (1 << 18)]
        u = torch.randn(part.shape[0], 4, device=DEVICE, generator=gen)
        part += (u @ dirs).to(keys.dtype).unsqueeze(1)
    keys[sinks] += 1.0


def _near(gen, x):
    """What the next layers hold: the anchor's tensor with noise of its own."""
    out = torch.empty_like(x).normal_(0.0, 0.3, generator=gen)
    return out.add_(x)


def _head_maps(case):
    """One row per layer: the shipped maps at the shape they are for, a fixed rotation otherwise."""
    G = case["kv_heads"]
    shipped = get_head_mapping(MODEL, list(ANCHORS))
    return [list(shipped[l]) if G == 8 and l < len(shipped) else [(g + l) % G for g in range(G)]
            for l in range(case["layers"])]


def _anchors(case):
    return [a for a in ANCHORS if a < case["layers"]]


def _layer_tensors(case, gen, new_tokens, kv_tokens):
    """Per layer (q [B,H,n,D] laid out token by token, as a rotary embedding leaves it; k and v
    [B,G,L,D] head-major, as a transformers cache holds them)."""
    B, H, G, D, dt = case["batch"], case["heads"], case["kv_heads"], case["head_dim"], _dtype(case)
    layers, q0, k0 = [], None, None
    for l in range(case["layers"]):
        if l in ANCHORS:
            q0 = _normal(gen, (B, new_tokens, H, D), dt, 0.5)
            k0 = _normal(gen, (B, G, kv_tokens, D), dt)
            for b in range(B):
                _peak(gen, k0[b].transpose(0, 1), [0])
            q, k = q0, k0
        else:
            q, k = _near(gen, q0), _near(gen, k0)
        layers.append((q.transpose(1, 2), k, _normal(gen, (B, G, kv_tokens, D), dt)))
    return layers


def _fill_pages(case, gen, k_pages, v_pages, block_table):
    """Contents for the caches of all layers; the first page of a sequence holds its sink."""
    sinks = (block_table[:, 0].to(torch.int64) * PAGE).tolist()
    base = None
    for l in range(case["layers"]):
        if l in ANCHORS:
            k_pages[l].normal_(0.0, 1.0, generator=gen)
            _peak(gen, k_pages[l].view(-1, *k_pages[l].shape[2:]), sinks)
            base = k_pages[l]
        else:
            k_pages[l].normal_(0.0, 0.3, generator=gen).add_(base)
        v_pages[l].normal_(0.0, 1.0, generator=gen)


def _step_inputs(case, gen):
    """q [layers,B,H,D], new keys and values [layers,B,1,G,D] of one decode step."""
    n, B, H, G, D, dt = case["layers"], case["batch"], case["heads"], case["kv_heads"], case["head_dim"], _dtype(case)
    q = _normal(gen, (n, B, H, D), dt, 0.5)
    for l in range(n):
        if l not in ANCHORS:
            anchor = max(a for a in ANCHORS if a < l)
            q[l] = _near(gen, q[anchor])
    return q, _normal(gen, (n, B, 1, G, D), dt), _normal(gen, (n, B, 1, G, D), dt)


def _stack(case, max_seqlen):
    return KascadeAttentionStack(case["layers"], _anchors(case), _head_maps(case), case["percent"], max_seqlen,
                                 batch=case["batch"], page_size=PAGE, rolling_prefill=case["rolling"], device=DEVICE,
                                 table_seed=1, kv_heads=case["kv_heads"], head_dim=case["head_dim"], dtype=_dtype(case),
                                 group_size=case["heads"] // case["kv_heads"])


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    kind, n, B = case["kind"], case["tokens"], case["batch"]
    state = {"case": case, "kind": kind}
    if kind in ("hf_prefill", "hf_decode"):
        state["layers"] = _layer_tensors(case, gen, n if kind == "hf_prefill" else 1, n)
        state["modules"] = [SimpleNamespace(layer_idx=l, is_causal=True, training=False) for l in range(case["layers"])]
        state["strategy"] = EfficientKascadeStrategy(_anchors(case), None, k=case["percent"], tile_size=32,
                                                     rolling_prefill=case["rolling"], head_mapping=_head_maps(case),
                                                     register=False)
    elif kind == "stack_prefill":
        state["stack"] = _stack(case, n)
        layers = _layer_tensors(case, gen, n, n)
        state["chunks"] = [([q.transpose(1, 2)[:, s:s + case["chunk"]] for q, _, _ in layers],
                            [k.transpose(1, 2)[:, s:s + case["chunk"]] for _, k, _ in layers],
                            [v.transpose(1, 2)[:, s:s + case["chunk"]] for _, _, v in layers])
                           for s in range(0, n, case["chunk"])]
    elif kind == "stack_decode":
        st = state["stack"] = _stack(case, n + HEADROOM)
        _fill_pages(case, gen, st.k_pages, st.v_pages, st.block_table)
        st.reset(n)
        state["inputs"] = _step_inputs(case, gen)
        if case["graph"]:
            st.capture_decode()
    else:
        lens = _lengths(case)
        G, D, dt = case["kv_heads"], case["head_dim"], _dtype(case)
        per_seq = [-(-(x + HEADROOM) // PAGE) for x in lens]
        order = torch.randperm(sum(per_seq), generator=torch.Generator().manual_seed(int(seed))).to(torch.int32)
        table = torch.zeros(B, max(per_seq), dtype=torch.int32)
        at = 0
        for b, p in enumerate(per_seq):
            table[b, :p] = order[at:at + p]
            at += p
        table = table.to(DEVICE)
        new = lambda: [torch.empty(at, PAGE, G, D, device=DEVICE, dtype=dt) for _ in range(case["layers"])]  # noqa: E731
        k_pages, v_pages = new(), new()
        _fill_pages(case, gen, k_pages, v_pages, table)
        state.update(k_pages=k_pages, v_pages=v_pages, table=table, inputs=_step_inputs(case, gen), steps=0,
                     first=torch.tensor(lens, dtype=torch.int32, device=DEVICE), max_len=max(lens) + HEADROOM)
        state["lens"] = state["first"].clone()
        state["out"] = torch.empty(case["layers"], B, case["heads"], D, device=DEVICE, dtype=dt)
        state["decoder"] = PagedKascadeDecoder(case["percent"], _head_maps(case), _anchors(case), B, state["max_len"],
                                               PAGE, DEVICE, seqlens_hint=lens, kv_heads=G, head_dim=D,
                                               group_size=case["heads"] // G)
    return state


# ------------------------------------------------------------------------------------- a pass
def run(state):
    kind, case = state["kind"], state["case"]
    if kind in ("hf_prefill", "hf_decode"):
        scaling = case["head_dim"] ** -0.5
        forward = state["strategy"].attention_forward
        return [forward(m, q, k, v, None, scaling)[0] for m, (q, k, v) in zip(state["modules"], state["layers"])]
    if kind == "stack_prefill":
        st = state["stack"]
        st.reset()
        outs = [st.prefill_chunk(*chunk) for chunk in state["chunks"]]
        return {"out": outs, "k": st.k_pages, "v": st.v_pages, "lengths": st.seqlens}
    if kind == "stack_decode":
        st = state["stack"]
        if st.length >= case["tokens"] + HEADROOM:
            st.reset(case["tokens"])
        q, k, v = state["inputs"]
        if case["graph"]:
            st.graph_q.copy_(q)
            st.graph_k.copy_(k)
            st.graph_v.copy_(v)
            out = st.replay_decode()
        else:
            out = st.decode_step(q, k, v)
        return {"out": out, "k": st.k_pages, "v": st.v_pages, "lengths": st.seqlens}
    dec, lens = state["decoder"], state["lens"]
    if state["steps"] == HEADROOM:
        lens.copy_(state["first"])
        state["steps"] = 0
    state["steps"] += 1
    q, k, v = state["inputs"]
    dec.begin_step(lens, 1)
    for l in range(case["layers"]):
        dec.forward(l, q[l], state["k_pages"][l], state["v_pages"][l], state["table"], lens, state["max_len"],
                    ragged=True, out=state["out"][l], k_new=k[l, :, 0], v_new=v[l, :, 0])
    return {"out": state["out"], "k": state["k_pages"], "v": state["v_pages"], "lengths": lens}


# ------------------------------------------------------------------------------- what it takes
def _cost(case):
    w = work(case)
    return max(w["bytes"] / 8e12, w["flops"] / 2.5e15)


def _kept(case, start):
    """Keys a query tile that starts at ``start`` takes from its list, at most."""
    if case["rolling"]:
        return min(start, budgets.rolling_budget(start, case["percent"]))
    return min(start, budgets.topk_width(case["tokens"], case["percent"]))


def work(case):
    """Prefill: causal products; a layer with an output of its own needs both products over the keys
    it attends to, an anchor also the scores of all keys (twice: a row's probabilities, which are
    what is pooled, need the row's sum first).  Decode: the K and V rows attended to, and for an
    anchor all K rows."""
    H, G, D, B, n = case["heads"], case["kv_heads"], case["head_dim"], case["batch"], case["tokens"]
    anchors = len(_anchors(case))
    reuse_like = case["layers"] - 1                       # every layer but the first ends in a sparse pass
    if "prefill" in case["kind"]:
        pairs = n * (n + 1) / 2
        step = max(32, n // 2048 // 32 * 32)              # sampled tile starts: the budget is smooth
        starts = range(0, n, step)
        sparse = sum((_kept(case, s) + 16.5) * min(step, n - s) for s in starts)
        one = 2.0 * D * H * B
        flops = one * (2 * pairs + pairs + (anchors - 1) * 2 * pairs + reuse_like * 2 * sparse)
        rows = B * n * D * 2
        moved = rows * (2 * H + 2 * G)
        if case["kind"] == "stack_prefill":
            moved += rows * 2 * G
        return {"bytes": case["layers"] * moved, "flops": flops}
    lens = _lengths(case)
    row = G * D * 2
    dense = sum(lens) * row
    kept = [min(x, max(128, budgets.decode_budget(x, case["percent"]))) for x in lens]
    sparse = sum(kept) * (2 * row + G * 4)
    small = case["layers"] * B * D * 2 * (2 * H + 2 * G)
    nbytes = 2 * dense + (anchors - 1) * dense + reuse_like * sparse + small
    return {"bytes": nbytes, "flops": 2.0 * H / G * nbytes / 2}


def tolerance(case):
    """Outputs are rounded to the element type, probabilities too before they meet V.  Pooled scores
    are fp16 for both types: tokens within a step of the selection's threshold may trade places,
    which fp16 outputs show as about as much again."""
    return {"rel": 1e-2} if case["dtype"] == "bfloat16" else {"rel": 4e-3}
