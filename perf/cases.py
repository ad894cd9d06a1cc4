"""The performance cases of the two attention paths and of the decoder around them.

A case is a dict of plain values; `prepare` makes what a program that uses the package has in hand
before the call (inputs from the seed alone, weights, caches, recordings), `run` takes one pass through
the public entry points, `work` counts the bytes and operations that a pass cannot do without, and
`tolerance` says how far two correct implementations of it may lie apart.

Kinds of cases

    prefill        `summary_attn_func` of one layer over whole prompts (periodic summary rows in line)
    index          `compute_block_sparsity`: a prompt length that was not seen before pays it once per
                   window size of the model
    decode         one decode step of one layer: `ksa_decode` with a row range per sequence, or
                   `decode_attention_forward` on the cache's strided views
    pre_attention  q / k norm + rotary embedding + layout write behind the fused projection of one layer
    model_prefill  `KsaQwen3ForCausalLM.prefill`
    model_step     one greedy step of the decoder inside a chunk: `decode_step_graph` + the token choice
"""
from __future__ import annotations

import math

import torch

import ksa_amd
from ksa_amd.model import KsaQwen3Config, KsaQwen3ForCausalLM, init_weights

CHUNK, SUMMARY = 128, 8       # text tokens and summary tokens per chunk
UNBOUNDED = 1 << 20           # window of a "full attention" layer, in chunks
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
STEP_TOKENS = 4096            # prompt length of the listed decode-step cases


def listed():
    return [
        # A short chat prompt: two chunks and a rest.  Launches and host work count.
        dict(name="prefill-300", kind="prefill", batch=1, tokens=300, q_heads=32, kv_heads=8, head_dim=128,
             window=4, dtype="bf16"),
        # The smallest benchmark configuration: 32 chunks, 16 query heads; one short launch.
        dict(name="prefill-4k", kind="prefill", batch=1, tokens=4096, q_heads=16, kv_heads=8, head_dim=128,
             window=4, dtype="bf16"),
        # A long document, one layer of the 4B shape.
        dict(name="prefill-32k", kind="prefill", batch=1, tokens=32768, q_heads=32, kv_heads=8, head_dim=128,
             window=4, dtype="bf16"),
        # The long-context benchmark configuration: over 95 % of the tile pairs are empty.
        dict(name="prefill-128k", kind="prefill", batch=1, tokens=131072, q_heads=32, kv_heads=8, head_dim=128,
             window=4, dtype="bf16"),
        # A layer with an unbounded window over a batch of prompts that end inside a chunk, in fp16.
        dict(name="prefill-dense-ragged", kind="prefill", batch=3, tokens=9001, q_heads=32, kv_heads=8,
             head_dim=128, window=UNBOUNDED, dtype="f16"),
        # The block index of the long-context configuration.
        dict(name="index-128k", kind="index", tokens=131072, window=4),
        # One sequence at 16k tokens of context, as the model code calls it (views of the cache).
        dict(name="decode-b1-16k", kind="decode", batch=1, tokens=16384, q_heads=32, kv_heads=8, head_dim=128,
             window=4, query_tokens=1, views=True, dtype="bf16"),
        # The decode benchmark configuration: 64 sequences of 128k tokens at different places of a chunk.
        dict(name="decode-b64-128k", kind="decode", batch=64, tokens=131072, q_heads=32, kv_heads=8, head_dim=128,
             window=4, query_tokens=1, views=False, dtype="bf16"),
        # Behind the fused projection of a 32k prompt; keys and values go straight to their cache rows.
        dict(name="pre-attention-32k", kind="pre_attention", batch=1, tokens=32768, q_heads=32, kv_heads=8,
             head_dim=128, dtype="bf16"),
        # Prompt processing of one group of layers (3 windowed : 1 unbounded) of the 4B shape, two users.
        dict(name="model-prefill-2x3000", kind="model_prefill", batch=2, tokens=3000, layers=4),
        # Token generation for one user and for a small batch, two groups of layers of the 4B shape and its
        # output head.
        dict(name="model-step-b1", kind="model_step", batch=1, tokens=STEP_TOKENS, layers=8),
        dict(name="model-step-b8", kind="model_step", batch=8, tokens=STEP_TOKENS, layers=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("prefill",) * 6 + ("index",) * 2 + ("decode",) * 4 + ("pre_attention",) * 2
                      + ("model_prefill", "model_step", "model_step"))
    dtype = rng.choice(("bf16", "bf16", "bf16", "f16"))
    q_heads, kv_heads = rng.choice(((32, 8), (32, 8), (32, 8), (16, 8), (8, 8), (32, 4)))
    if kind == "prefill":
        case = dict(kind=kind, batch=rng.choice((1, 1, 2, 3, 8)), tokens=_log_int(rng, 130, 131072),
                    q_heads=q_heads, kv_heads=kv_heads, head_dim=rng.choice((128, 128, 128, 128, 64, 256)),
                    window=rng.choice((4, 4, 4, 1, 3, 16, UNBOUNDED)), dtype=dtype)
        most = work(listed()[3])["flops"]
        while work(case)["flops"] > most:
            case["tokens"] = case["tokens"] // 2 + 1
        return case
    if kind == "index":
        return dict(kind=kind, tokens=_log_int(rng, 2000, 131072), window=rng.choice((4, 4, 1, 8)))
    if kind == "decode":
        case = dict(kind=kind, batch=_log_int(rng, 1, 64), tokens=_log_int(rng, 200, 131072), q_heads=q_heads,
                    kv_heads=kv_heads, head_dim=rng.choice((128, 128, 128, 64, 256)),
                    window=rng.choice((4, 4, 3, 16)), query_tokens=rng.choice((1, 1, 1, 1, SUMMARY)),
                    views=rng.random() < 0.5, dtype=dtype)
        most = work(listed()[7])["bytes"]
        while work(case)["bytes"] > most:
            case["batch"] = max(1, case["batch"] // 2)
            if case["batch"] == 1:
                case["tokens"] = case["tokens"] // 2 + 1
        return case
    if kind == "pre_attention":
        return dict(kind=kind, batch=rng.choice((1, 2, 4)), tokens=_log_int(rng, 300, 32768), q_heads=q_heads,
                    kv_heads=kv_heads, head_dim=rng.choice((128, 128, 128, 64)), dtype=dtype)
    if kind == "model_prefill":
        batch = rng.choice((1, 2, 4))
        return dict(kind=kind, batch=batch, tokens=_log_int(rng, 100, 6000 // batch), layers=4)
    return dict(kind=kind, batch=_log_int(rng, 1, 64), tokens=_log_int(rng, 300, STEP_TOKENS), layers=rng.choice((4, 8)))


# ---- sizes ----------------------------------------------------------------------------------------

def _rows(tokens):
    """(rows with the summary tokens in line, summary rows) of a prompt."""
    summaries = tokens // CHUNK * SUMMARY
    return tokens + summaries, summaries


def _visible_pairs(tokens, W):
    """(query row, key) pairs that attend each other: text rows see the text of their chunk and of W chunks
    before it and the summaries of all earlier chunks, summary rows see their own chunk, causally."""
    total = 0
    chunks, rest = divmod(tokens, CHUNK)
    for c in range(chunks + (1 if rest else 0)):
        n = CHUNK if c < chunks else rest
        total += n * (min(c, W) * CHUNK + max(0, c - W) * SUMMARY) + n * (n + 1) // 2
        if c < chunks:
            total += SUMMARY * CHUNK + SUMMARY * (SUMMARY + 1) // 2
    return total


def _cache_layout(case):
    """Rows of the ring-buffer cache of a windowed layer: (capacity, row behind the chunk, last attended row)."""
    W, done = case["window"], case["tokens"] // CHUNK
    n_sum = done * SUMMARY
    ring = W * CHUNK
    cap = SUMMARY + CHUNK + ring + n_sum + max(512, n_sum + 256)
    head = SUMMARY + CHUNK
    if done >= W:
        end = head + ring + n_sum - min(W * SUMMARY, n_sum)
    else:
        end = head + done * CHUNK
    return cap, head, end


def _chunk_fill(case, b):
    """Rows of the current chunk of sequence b, 1 .. CHUNK, spread over the chunk."""
    return 1 + (case["tokens"] + 37 * b) % CHUNK


def _model_config(layers):
    return KsaQwen3Config(num_hidden_layers=layers,
                          summary_sliding_chunk_num=[UNBOUNDED if i % 4 == 3 else 4 for i in range(layers)])


def _layer_params(cfg):
    D = cfg.head_dim
    nq, nkv = cfg.num_attention_heads * D, cfg.num_key_value_heads * D
    return cfg.hidden_size * (2 * nq + 2 * nkv + 3 * cfg.intermediate_size)


def work(case):
    kind = case["kind"]
    if kind == "prefill":
        rows, _ = _rows(case["tokens"])
        D, b = case["head_dim"], case["batch"]
        return {"bytes": b * rows * D * 2 * (2 * case["q_heads"] + 2 * case["kv_heads"]),
                "flops": 4 * D * case["q_heads"] * b * _visible_pairs(case["tokens"], case["window"])}
    if kind == "index":
        rows, summaries = _rows(case["tokens"])
        M, N = -(-rows // 128), -(-(rows + summaries) // 64)
        return {"bytes": 2 * 4 * (M + M * N), "flops": 0}
    if kind == "decode":
        _, head, end = _cache_layout(case)
        if case["views"]:
            rows = case["batch"] * (end - head + _chunk_fill(case, 0))
        else:
            rows = sum(end - head + _chunk_fill(case, b) for b in range(case["batch"]))
        D, Q = case["head_dim"], case["query_tokens"]
        return {"bytes": 2 * D * (2 * rows * case["kv_heads"] + 2 * case["batch"] * Q * case["q_heads"]),
                "flops": 4 * D * rows * case["q_heads"] * Q}
    if kind == "pre_attention":
        rows, _ = _rows(case["tokens"])
        D = case["head_dim"]
        return {"bytes": 2 * D * rows * (2 * case["batch"] * (case["q_heads"] + 2 * case["kv_heads"]) + 2), "flops": 0}
    cfg = _model_config(case["layers"])
    D, b = cfg.head_dim, case["batch"]
    params = case["layers"] * _layer_params(cfg)
    head = cfg.vocab_size * cfg.hidden_size
    wide = case["layers"] // 4
    if kind == "model_prefill":
        rows, _ = _rows(case["tokens"])
        pairs = (case["layers"] - wide) * _visible_pairs(case["tokens"], 4) + wide * _visible_pairs(case["tokens"], UNBOUNDED)
        return {"bytes": 2 * (params + head) + case["layers"] * 2 * 2 * b * rows * cfg.num_key_value_heads * D,
                "flops": 2 * b * rows * params + 2 * b * head + 4 * D * cfg.num_attention_heads * b * pairs}
    done, rest = divmod(_step_tokens(case), CHUNK)
    small = rest + 1 + (4 * CHUNK + (done - 4) * SUMMARY if done >= 4 else done * CHUNK)
    rows = (case["layers"] - wide) * small + wide * (_step_tokens(case) + 1)
    return {"bytes": 2 * (params + head) + 2 * 2 * b * rows * cfg.num_key_value_heads * D,
            "flops": 2 * b * (params + head) + 4 * D * cfg.num_attention_heads * b * rows}


def _step_tokens(case):
    """Prompt length of a decode-step case: a step at the last token of a chunk is another kind of step."""
    n = case["tokens"]
    return n - 2 if n % CHUNK >= CHUNK - 2 else n


def tolerance(case):
    # About four times the distance to the same path in 64 bits, or between two orders of summation.
    kind = case["kind"]
    if kind == "index":
        return "exact"
    if kind in ("model_prefill", "model_step"):
        # logits and cache rows behind layers of 16-bit roundings: two forms of the MLP that differ in the order
        # of their fp32 sums lie 0.8 % apart behind 4 layers, 1.25 % behind 8, 1.5 % behind 12 and 3.2 %
        # behind 36 (random weights), which is why the cases stay at 8 layers
        return {"rel": 3e-2}
    if kind == "pre_attention":
        # (the fp32 sum of squares decides a rounding now and then: one unit in the last place)
        return {"rel": 1e-4, "max": 5e-2} if case["dtype"] == "bf16" else {"rel": 4e-5, "max": 8e-3}
    # attention against the same in 64 bits: 2.2e-3 in bf16, 2.7e-4 in fp16
    return {"rel": 9e-3 if case["dtype"] == "bf16" else 1.2e-3}


# ---- states -----------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(shape, dtype, g):
    """N(0, 1) values, drawn slice by slice along the first dimension (no fp32 copy of the whole)."""
    t = torch.empty(shape, dtype=dtype, device="cuda")
    flat = t.view(-1)
    step = 1 << 26
    for i in range(0, flat.numel(), step):
        n = min(step, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, generator=g, device="cuda").to(dtype)
    return t


def prepare(case, seed):
    return {"prefill": _prepare_prefill, "index": _prepare_index, "decode": _prepare_decode,
            "pre_attention": _prepare_pre_attention, "model_prefill": _prepare_model_prefill,
            "model_step": _prepare_model_step}[case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _prepare_prefill(case, seed):
    g = _generator(seed)
    rows, _ = _rows(case["tokens"])
    dt, b, D = DTYPES[case["dtype"]], case["batch"], case["head_dim"]
    # queries and keys come from an RMSNorm over the head dimension: elements of unit scale
    q = _normal((b, rows, case["q_heads"], D), dt, g)
    k = _normal((b, rows, case["kv_heads"], D), dt, g)
    v = _normal((b, rows, case["kv_heads"], D), dt, g)
    pos = (torch.arange(rows, device="cuda") % (CHUNK + SUMMARY)) >= CHUNK
    return dict(run=_run_prefill, q=q, k=k, v=v, pos=pos, window=case["window"])


def _run_prefill(s):
    out, _ = ksa_amd.summary_attn_func(s["q"], s["k"], s["v"], CHUNK, SUMMARY, s["window"], summary_pos=s["pos"])
    return out


def _prepare_index(case, seed):
    rows, summaries = _rows(case["tokens"])
    # another seed: another layer's window
    return dict(run=_run_index, rows=rows, keys=rows + summaries, window=case["window"] + int(seed) % 4)


def _run_index(s):
    return tuple(ksa_amd.compute_block_sparsity(s["rows"], s["keys"], CHUNK, SUMMARY, s["window"]))


class _Module:
    """What `decode_attention_forward` takes of an attention module."""

    def __init__(self, groups):
        self.num_key_value_groups = groups


def _prepare_decode(case, seed):
    g = _generator(seed)
    dt, b, D = DTYPES[case["dtype"]], case["batch"], case["head_dim"]
    cap, head, end = _cache_layout(case)
    kc = _normal((b, case["kv_heads"], cap, D), dt, g)
    vc = _normal((b, case["kv_heads"], cap, D), dt, g)
    q = _normal((b, case["q_heads"], case["query_tokens"], D), dt, g)
    if case["views"]:
        a = head - _chunk_fill(case, 0)
        return dict(run=_run_decode_views, q=q, kc=kc, vc=vc, start=a, end=end, scale=D ** -0.5,
                    module=_Module(case["q_heads"] // case["kv_heads"]))
    start = torch.tensor([head - _chunk_fill(case, i) for i in range(b)], dtype=torch.int32, device="cuda")
    stop = torch.full((b,), end, dtype=torch.int32, device="cuda")
    return dict(run=_run_decode_ranges, q=q, kc=kc, vc=vc, start=start, end=stop)


def _run_decode_views(s):
    k, v = s["kc"][:, :, s["start"]:s["end"]], s["vc"][:, :, s["start"]:s["end"]]
    return ksa_amd.decode_attention_forward(s["module"], s["q"], k, v, None, scaling=s["scale"])[0]


def _run_decode_ranges(s):
    return ksa_amd.ksa_decode(s["q"], s["kc"], s["vc"], s["start"], s["end"])


def _prepare_pre_attention(case, seed):
    g = _generator(seed)
    rows, _ = _rows(case["tokens"])
    dt, b, D, Hq, Hkv = DTYPES[case["dtype"]], case["batch"], case["head_dim"], case["q_heads"], case["kv_heads"]
    qkv = _normal((b, rows, (Hq + 2 * Hkv) * D), dt, g)
    q = qkv[..., :Hq * D].view(b, rows, Hq, D)
    k = qkv[..., Hq * D:(Hq + Hkv) * D].view(b, rows, Hkv, D)
    v = qkv[..., (Hq + Hkv) * D:].view(b, rows, Hkv, D)
    inv = 1e6 ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float32) / D)
    angle = torch.arange(rows, device="cuda", dtype=torch.float32)[:, None] * inv[None]
    angle = torch.cat((angle, angle), dim=-1)[None]
    slots = [torch.zeros(b, Hkv, rows + 1024, D, dtype=dt, device="cuda")[:, :, :rows].transpose(1, 2) for _ in range(2)]
    weights = [(1 + 0.1 * torch.randn(D, generator=g, device="cuda")).to(dt) for _ in range(2)]
    return dict(run=_run_pre_attention, q=q, k=k, v=v, wq=weights[0], wk=weights[1], cos=angle.cos().to(dt),
                sin=angle.sin().to(dt), k_out=slots[0], v_out=slots[1])


def _run_pre_attention(s):
    return ksa_amd.pre_attention(s["q"], s["k"], s["v"], s["wq"], s["wk"], s["cos"], s["sin"], 1e-6,
                                 k_out=s["k_out"], v_out=s["v_out"])


def _model(case, seed):
    cfg = _model_config(case["layers"])
    model = KsaQwen3ForCausalLM(cfg, init_weights(cfg, "cuda", torch.bfloat16, seed=int(seed)))
    return cfg, model


def _prepare_model_prefill(case, seed):
    cfg, model = _model(case, seed)
    ids = torch.randint(0, cfg.vocab_size, (case["batch"], case["tokens"]), generator=_generator(seed), device="cuda")
    return dict(run=_run_model_prefill, model=model, ids=ids)


def _run_model_prefill(s):
    logits, cache = s["model"].prefill(s["ids"])
    return [logits] + [t for layer in range(len(cache)) for t in cache.get_attention_kv(layer)]


# the cache's host-side cursors: putting them back rewinds a step inside a chunk
_CURSORS = ("_text_len", "_chunk_buf_len", "cur_chunk_sizes", "true_tokens")


def _prepare_model_step(case, seed):
    cfg, model = _model(case, seed)
    ids = torch.randint(0, cfg.vocab_size, (case["batch"], _step_tokens(case)), generator=_generator(seed), device="cuda")
    logits, cache = model.prefill(ids)
    token = model.ops.argmax(logits[:, 0])[:, None]
    cursors = {name: list(getattr(cache, name)) for name in _CURSORS}
    state = dict(run=_run_model_step, model=model, cache=cache, token=token, cursors=cursors)
    _run_model_step(state)      # the step's recording, which a program makes once per cache
    return state


def _run_model_step(s):
    model, cache = s["model"], s["cache"]
    for name, values in s["cursors"].items():   # the same step of the same sequence again
        setattr(cache, name, list(values))
    logits = model.decode_step_graph(s["token"], cache)
    # the next token of the program's loop; not among the outputs, since it may tip between two logits that
    # lie closer to each other than the rounding of the layers
    s["next"] = model.ops.argmax(logits[:, 0])[:, None]
    # what the step has added to the cache, in a windowed and in an unbounded layer
    written = []
    for layer in (len(cache) - 2, len(cache) - 1):
        k, v = cache.get_attention_kv(layer)
        row = slice(-1, None) if cache.is_large_window[layer] else slice(0, 1)
        written += [k[:, :, row], v[:, :, row]]
    return [logits] + written
