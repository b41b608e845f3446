"""The work that a user of this framework has it do, as measurable cases.

Three ways in, all public:

* ``layer`` - decode steps over a few layers of a model whose contexts are in the cache, as
  ``model.Decoder`` and a serving stack with a token budget run them: one ``ops.DecodeLayer`` for all
  layers, a ``Batch`` and a threshold hint per layer, K/V store and attention in one ``step`` call, or
  ``ops.qkv_store`` and the layer call (``proj``), or a selection cache per layer (``cache``).
* ``chunk`` - a chunk of a long prompt over a few layers: ``ops.PrefillChunk.step``.
* ``serve`` - whole requests through the patched attention (``patch()``, a ``ModelRunner``, a retriever
  per request, ``RadixAttention.forward`` in EXTEND and then in DECODE mode) on the projection's output as
  the attention module splits it; several requests are prefilled one by one and decoded together.

A pass starts by putting the lengths (and the free-page counts) back, as a scheduler that hands the
layer the lengths of the step does, so that it can be repeated.  Queries, keys and values are normal;
a query drifts from step to step, and the rows of a chunk have a part in common, as a model's do.
Sizes are those of the shipped configurations: sink 128, local window 512, top-k 2048 (4096 for the
longest contexts), chunks of 512 rows, tables of 1048576 tokens.
"""

import random

import torch

from tokenselect_amd import ops
from tokenselect_amd.patcher import sglang_standins as stack
from tokenselect_amd.patcher import token_retrieval

D = 128
N_INIT, N_LOCAL = 128, 512
CHUNK = 512
MAX_TOKENS = 1048576
STEP_DRIFT = 0.95     # cosine of a query with the one of the step before
CACHE_DRIFT = 0.97    # with the selection cache: an entry serves three more steps, then falls below 0.898
CACHE_SERVES = 3

# (query heads, KV heads, rope base) of one layer, and hidden size where it is not the query heads' width:
# whole models and their tensor-parallel ranks.
SHAPES = {
    "llama3-8b": (32, 8, 5e5),
    "qwen2-7b": (28, 4, 1e6),
    "llama3.2-3b": (24, 8, 5e5),
    "qwen2-1.5b": (12, 2, 1e6),
    "llama3-8b tp4": (8, 2, 5e5),
    "llama3-8b tp8": (4, 1, 5e5),
    "qwen2-7b tp2": (14, 2, 1e6),
}


def _layer(shape, batch, lo, hi, layers, steps=2, page=1, k=2048, pool=-1, proj=False, cache=False):
    return {"path": "layer", "shape": shape, "batch": batch, "lo": lo, "hi": hi, "layers": layers,
            "steps": steps, "page": page, "k": k, "pool": pool, "proj": proj, "cache": cache}


def _chunk(shape, length, rows, layers, page=1, k=2048, pool=-1):
    return {"path": "chunk", "shape": shape, "length": length, "rows": rows, "layers": layers,
            "page": page, "k": k, "pool": pool}


def _serve(shape, batch, lo, hi, layers, new, k=2048, pool=-1):
    return {"path": "serve", "shape": shape, "batch": batch, "lo": lo, "hi": hi, "layers": layers,
            "new": new, "k": k, "pool": pool}


def _named(name, case):
    return {"name": name, **case}


def listed():
    return [
        # A chat turn: a short prompt and a few tokens, everything attended to densely.
        _named("serve short", _serve("llama3-8b", 1, 300, 300, layers=2, new=8)),
        # A document question: the prompt in 62 chunks, the last of them ragged, then the answer's tokens.
        _named("serve 31k", _serve("qwen2-7b", 1, 31599, 31599, layers=1, new=16)),
        # Three requests of different lengths prefilled one by one, then decoded together.
        _named("serve batch", _serve("llama3-8b", 3, 700, 5200, layers=2, new=8)),
        # Decode while the context is still short: dense.
        _named("decode 1x2k", _layer("qwen2-7b", 1, 2003, 2003, layers=8)),
        # One request at the length many deployments allow, on the reference's per-token table.
        _named("decode 1x32k", _layer("qwen2-7b", 1, 32768, 32768, layers=8)),
        # The headline: one request of 128K tokens on pages of 16.
        _named("decode 1x128k", _layer("llama3-8b", 1, 131072, 131072, layers=2, page=16)),
        # A long-context evaluation: votes max-pooled over a window.
        _named("decode 1x100k pooled", _layer("llama3-8b", 1, 100003, 100003, layers=2, pool=15)),
        # An ordinary serving batch, the QKV projection with the store as its epilogue.
        _named("decode 8x8k", _layer("llama3-8b", 8, 3000, 16000, layers=4, proj=True)),
        # A large ragged batch, and few very long requests: more scores than one selection launch holds.
        _named("decode 16x68k", _layer("llama3-8b", 16, 4096, 131072, layers=1, page=16)),
        _named("decode 4x256k", _layer("llama3-8b", 4, 262144, 262144, layers=1, steps=1, page=16, k=4096)),
        # Selections reused while the query hardly moves.
        _named("cached 4x64k", _layer("llama3-8b", 4, 65536, 65536, layers=1, steps=8, cache=True)),
        # A chunk of a long prompt.
        _named("chunk 512 at 128k", _chunk("llama3-8b", 131072, 512, layers=2)),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    path = rng.choice(("layer", "layer", "layer", "cached", "chunk", "serve"))
    pool = rng.choice((-1, -1, -1, rng.randint(5, 128)))
    if path == "serve":
        batch = rng.choice((1, 1, 2, 4))
        lo = _log(rng, 100, 32000 // batch)
        hi = lo if batch == 1 else _log(rng, lo, 32000 // batch)
        return _serve(rng.choice(list(SHAPES)), batch, lo, hi, layers=1 if hi > 4000 else 2,
                      new=rng.randint(4, 16), pool=pool)
    if path == "chunk":
        length = _log(rng, 600, 200000)
        return _chunk(rng.choice(list(SHAPES)), length, rng.choice((CHUNK, CHUNK, rng.randint(2, CHUNK))),
                      layers=2, page=rng.choice((1, 1, 16)), pool=pool)
    if path == "cached":
        batch = rng.choice((1, 2, 4, 8))
        hi = _log(rng, 4000, 262144 // batch)
        return _layer(rng.choice(("llama3-8b", "qwen2-7b", "llama3.2-3b")), batch, max(4000, hi // 2), hi,
                      layers=1, steps=8, page=rng.choice((1, 16)), cache=True)
    batch = _log(rng, 1, 32)
    most = min(262144, 1048576 // batch)
    hi = _log(rng, 600, most)
    lo = rng.choice((hi, _log(rng, 500, hi)))
    shape = rng.choice(list(SHAPES))
    return _layer(shape, batch, lo, hi, layers=1 if hi * batch > 262144 else 4 if hi * batch < 32768 else 2,
                  steps=1 if hi * batch > 524288 else 2, page=rng.choice((1, 16, 16, 64)),
                  k=rng.choice((2048, 2048, 1024, 4096)), pool=pool,
                  proj=batch <= 8 and shape in ("llama3-8b", "qwen2-7b") and rng.random() < 0.3)


# --------------------------------------------------------------------------- what a case stands for
def _lengths(case):
    """The requests' lengths before the pass: given by the case alone."""
    rng = random.Random("%d %d %d" % (case["batch"], case["lo"], case["hi"]))
    got = [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])]
    got[0], got[-1] = (case["hi"], case["lo"]) if case["batch"] > 1 else (case["hi"], case["hi"])
    return got


def _jumps(case):
    """[steps][batch]: whether a request's query is a new one at a step (selection cache)."""
    rng = random.Random("jumps %d %d" % (case["batch"], case["hi"]))
    return [[t == 0 or rng.random() < 0.1 for _ in range(case["batch"])] for t in range(case["steps"])]


def _config(case):
    heads, kv_heads, base = SHAPES[case["shape"]]
    return ops.LayerConfig(num_heads=heads, num_kv_heads=kv_heads, page_size=case.get("page", 1), n_init=N_INIT,
                           n_local=N_LOCAL, top_k=case["k"], pool_kernel=case["pool"], rope_theta=base)


def _hidden(case):
    return 4096 if case["shape"] == "llama3-8b" else 3584


# --------------------------------------------------------------------------- layer
def _contexts(case, gen, lengths, extra):
    """Pools and tables of every layer: `lengths[b]` tokens cached and room for `extra` more per request."""
    cfg = _config(case)
    ps, dev = cfg.page_size, "cuda"
    held = [-(-n // ps) for n in lengths]
    fresh = -(-extra // ps) + 1
    total = sum(held) + fresh * len(lengths)
    width = max(held) + fresh
    order = torch.randperm(total, generator=gen, device=dev).to(torch.int32)
    table = torch.zeros((len(lengths), width), dtype=torch.int32, device=dev)
    at = 0
    for b, n in enumerate(held):
        table[b, :n] = order[at:at + n]
        at += n
    layers = range(case["layers"])

    def pools():
        return [torch.randn((total * ps, cfg.num_kv_heads, D), generator=gen, device=dev, dtype=torch.bfloat16)
                for _ in layers]

    s = {"cfg": cfg, "k_pools": pools(), "v_pools": pools(), "tables": [table.clone() for _ in layers]}
    lens = torch.tensor(lengths, dtype=torch.int32, device=dev)
    s["lens_before"] = lens.repeat(case["layers"], 1).contiguous()
    s["lens"] = s["lens_before"].clone()
    s["pages"] = [None for _ in layers]
    if ps > 1:
        free = order[at:]
        s["free_before"] = torch.full((case["layers"], 1), free.shape[0], dtype=torch.int32, device=dev)
        s["free"] = s["free_before"].clone()
        s["pages"] = [ops.PagePool(free.clone(), s["free"][l], torch.zeros(1, dtype=torch.int32, device=dev))
                      for l in layers]
    s["slots"] = order[at:] if ps == 1 else None
    return s


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _prepare_layer(case, gen):
    lengths, steps, layers, batch = _lengths(case), case["steps"], case["layers"], case["batch"]
    s = _contexts(case, gen, lengths, steps)
    cfg = s["cfg"]
    s["lengths"] = lengths
    row = cfg.num_kv_heads * D
    if s["slots"] is not None:
        s["slots"] = s["slots"][:steps * batch].view(steps, batch).contiguous()
    drift = CACHE_DRIFT if case["cache"] else STEP_DRIFT
    jumps = _jumps(case) if case["cache"] else None
    width = _hidden(case) if case["proj"] else cfg.num_heads * D
    q, x = [], _randn(gen, layers, batch, width)
    for t in range(steps):
        new = _randn(gen, layers, batch, width)
        step = drift * x + (1 - drift * drift) ** 0.5 * new
        if jumps is not None:
            step = torch.where(torch.tensor(jumps[t], device="cuda").view(1, -1, 1), new, step)
        x = step
        q.append(x.to(torch.bfloat16))
    s["q"] = [[q[t][l].contiguous() for l in range(layers)] for t in range(steps)]
    if case["proj"]:
        n_out = (cfg.num_heads + 2 * cfg.num_kv_heads) * D
        s["w"] = [(_randn(gen, n_out, width) * width ** -0.5).to(torch.bfloat16) for _ in range(layers)]
    else:
        s["kv"] = _randn(gen, steps, layers, 2, batch, row).to(torch.bfloat16)
    max_len = max(lengths) + steps
    s["layer"] = ops.DecodeLayer(cfg, batch, max_len, torch.device("cuda"))
    s["hints"] = torch.zeros((layers, batch), dtype=torch.int32, device="cuda")
    s["caches"] = [ops.SelectionCache.allocate(cfg, batch, "cuda") if case["cache"] else None for _ in range(layers)]
    s["out"] = torch.empty((steps, layers, batch, cfg.num_heads * D), dtype=torch.bfloat16, device="cuda")
    return s


def _run_layer(case, s):
    s["lens"].copy_(s["lens_before"])
    if "free" in s:
        s["free"].copy_(s["free_before"])
    if case["cache"]:
        for cache in s["caches"]:
            cache.cache_len.zero_()
    cfg, layer = s["cfg"], s["layer"]
    for t in range(case["steps"]):
        host = torch.tensor([n + t + 1 for n in s["lengths"]], dtype=torch.int32)
        longest = max(s["lengths"]) + t + 1
        loc = None if s["slots"] is None else s["slots"][t]
        for l in range(case["layers"]):
            bt = ops.Batch(s["lens"][l], s["tables"][l], longest, host_seq_lens=host, hint=s["hints"][l])
            k_pool, v_pool, out = s["k_pools"][l], s["v_pools"][l], s["out"][t, l]
            if case["proj"]:
                q = ops.qkv_store(cfg, s["q"][t][l], s["w"][l], None, loc, k_pool, v_pool, s["tables"][l],
                                  s["lens"][l], pages=s["pages"][l])
                layer(q, k_pool, v_pool, bt, s["caches"][l], out=out)
            else:
                layer.step(s["q"][t][l], s["kv"][t, l, 0], s["kv"][t, l, 1], loc, k_pool, v_pool, bt,
                           s["caches"][l], out=out, pages=s["pages"][l])
    return {"out": s["out"], "lens": s["lens"], "tables": s["tables"]}


# --------------------------------------------------------------------------- chunk
def _prepare_chunk(case, gen):
    before, rows, layers = case["length"], case["rows"], case["layers"]
    s = _contexts(case, gen, [before], rows)
    cfg = s["cfg"]
    s["longest"] = before + rows
    if s["slots"] is not None:
        s["slots"] = s["slots"][:rows].contiguous()
    row = cfg.num_kv_heads * D
    common = _randn(gen, layers, 1, cfg.num_heads * D)
    s["q"] = (common + _randn(gen, layers, rows, cfg.num_heads * D)).to(torch.bfloat16)
    s["kv"] = _randn(gen, layers, 2, rows, row).to(torch.bfloat16)
    s["chunk"] = ops.PrefillChunk(cfg, before + rows, torch.device("cuda"), max_rows=CHUNK)
    s["out"] = torch.empty((layers, rows, cfg.num_heads * D), dtype=torch.bfloat16, device="cuda")
    return s


def _run_chunk(case, s):
    s["lens"].copy_(s["lens_before"])
    if "free" in s:
        s["free"].copy_(s["free_before"])
    for l in range(case["layers"]):
        bt = ops.Batch(s["lens"][l], s["tables"][l], s["longest"])
        s["chunk"].step(s["q"][l], s["kv"][l, 0], s["kv"][l, 1], s["slots"], s["k_pools"][l], s["v_pools"][l], bt,
                        out=s["out"][l], pages=s["pages"][l])
    return {"out": s["out"], "lens": s["lens"], "tables": s["tables"]}


# --------------------------------------------------------------------------- serve
def _prepare_serve(case, gen):
    heads, kv_heads, base = SHAPES[case["shape"]]
    layers, prompts, new = case["layers"], _lengths(case), case["new"]
    token_retrieval.patch(rope_base=base, rope_scale=1, rope_model="ROPE_LLAMA", max_n_tokens=MAX_TOKENS,
                          top_k=case["k"], n_init=N_INIT, n_local=N_LOCAL, kernel_size=case["pool"])
    rows = sum(prompts) + len(prompts) * new
    pool = stack.TokenToKVPool(rows, torch.bfloat16, kv_heads, D, layers, "cuda")
    runner = stack.ModelRunner(model_config=stack.ModelConfig(layers, D, heads, kv_heads), token_to_kv_pool=pool,
                               dtype=torch.bfloat16)
    slots = torch.randperm(rows, generator=gen, device="cuda").to(torch.int32)
    width = (heads + 2 * kv_heads) * D
    common = torch.zeros((layers, 1, width), device="cuda")
    common[:, :, :heads * D] = _randn(gen, layers, 1, heads * D)
    s = {"pool": pool, "owner": runner.req_to_token_retriever, "requests": 0,
         "sizes": (heads * D, kv_heads * D, kv_heads * D),
         "attn": [stack.RadixAttention(heads, D, D ** -0.5, kv_heads, layer_id=l) for l in range(layers)]}
    s["prompt_qkv"] = [[(_randn(gen, n, width) + common[l]).to(torch.bfloat16) for l in range(layers)]
                       for n in prompts]
    s["token_qkv"] = [[(_randn(gen, len(prompts), width) + common[l]).to(torch.bfloat16) for l in range(layers)]
                      for _ in range(new)]
    at, s["prompt_slots"] = 0, []
    for n in prompts:
        s["prompt_slots"].append(slots[at:at + n])
        at += n
    s["token_slots"] = slots[at:].view(new, len(prompts))
    return s


def _run_serve(case, s):
    pool, owner, outs = s["pool"], s["owner"], []
    first = s["requests"]
    s["requests"] += case["batch"]
    names = tuple("request %d" % (first + b) for b in range(case["batch"]))
    retrievers = []
    for b in range(case["batch"]):
        retriever = owner.get_token_retriever(names[0]) if case["batch"] == 1 else owner.new_token_retriever()
        meta = stack.InputMetadata(stack.ForwardMode.EXTEND, retriever, pool, s["prompt_slots"][b])
        for l, attn in enumerate(s["attn"]):
            q, k, v = s["prompt_qkv"][b][l].split(s["sizes"], dim=-1)
            outs.append(attn.forward(q, k, v, meta))
        retrievers.append(retriever)
    running = retrievers[0] if case["batch"] == 1 else owner.get_batch_token_retriever(names, retrievers)
    for t in range(case["new"]):
        meta = stack.InputMetadata(stack.ForwardMode.DECODE, running, pool, s["token_slots"][t],
                                   batch_size=case["batch"])
        for l, attn in enumerate(s["attn"]):
            q, k, v = s["token_qkv"][t][l].split(s["sizes"], dim=-1)
            outs.append(attn.forward(q, k, v, meta))
    return {"out": outs, "k": pool.k_buffer, "v": pool.v_buffer}


# --------------------------------------------------------------------------- the interface
_PATHS = {"layer": (_prepare_layer, _run_layer), "chunk": (_prepare_chunk, _run_chunk),
          "serve": (_prepare_serve, _run_serve)}


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    state = _PATHS[case["path"]][0](case, gen)
    state["case"] = case
    return state


def run(state):
    return _PATHS[state["case"]["path"]][1](state["case"], state)


def _call(case, length, rows, hit=False):
    """(bytes, flops) of one layer call of one request that holds `length` tokens, `rows` of them new: the new
    rows read and stored, the candidates' keys read once, the selected rows read once, the output written."""
    heads, kv_heads, _ = SHAPES[case["shape"]]
    kept = N_INIT + case["k"] + N_LOCAL
    sparse = length > kept
    attended = kept if sparse else length
    row = kv_heads * D * 2
    moved = rows * (4 * row + 2 * heads * D * 2) + attended * (2 * row + 4)
    pairs = rows * attended - rows * (rows - 1) // 2
    flops = 4 * heads * D * pairs
    if sparse and not hit:
        candidates = length - N_INIT - N_LOCAL
        moved += candidates * row + 4 * -(-candidates // case.get("page", 1))
        flops += 2 * heads * D * candidates
    return moved, flops


def work(case):
    """One pass: every call of it reads its inputs once and writes its outputs once (the keys of a context are
    read again by each step and each chunk: a new query has to see them)."""
    calls, layers = [], case["layers"]
    extra_bytes = extra_flops = 0
    if case["path"] == "chunk":
        calls.append(_call(case, case["length"] + case["rows"], case["rows"]))
    elif case["path"] == "serve":
        for n in _lengths(case):
            for start in range(0, n, CHUNK):
                rows = min(CHUNK, n - start)
                calls.append(_call(case, start + rows, rows))
            calls += [_call(case, n + t + 1, 1) for t in range(case["new"])]
    else:
        lengths = _lengths(case)
        jumps = _jumps(case) if case["cache"] else None
        since = [0] * len(lengths)
        for t in range(case["steps"]):
            for b, n in enumerate(lengths):
                hit = False
                if jumps is not None:
                    hit = not jumps[t][b] and since[b] < CACHE_SERVES
                    since[b] = since[b] + 1 if hit else 0
                calls.append(_call(case, n + t + 1, 1, hit))
        if case["proj"]:
            heads, kv_heads, _ = SHAPES[case["shape"]]
            weights = (heads + 2 * kv_heads) * D * _hidden(case)
            extra_bytes = case["steps"] * 2 * weights
            extra_flops = case["steps"] * case["batch"] * 2 * weights
    return {"bytes": layers * (sum(c[0] for c in calls) + extra_bytes),
            "flops": layers * (sum(c[1] for c in calls) + extra_flops)}


def tolerance(case):
    """bf16 outputs of sums in fp32.  A selection may also settle a near-tie at the k-th vote the other way
    (fp32 votes added up in another order): one of some 2688 averaged rows changes, sqrt(2 / 2688) = 0.027 of
    that selection's output and less of a pass's.  Lengths, tables and stored rows are copied: the same."""
    return {"rel": 2e-2, "differ": 0.0}
