"""What a program does with this framework, as cases that can be timed.

Three kinds of call, each through a public entry point:

- "attend": one decode attention over paged K/V on the caller's device
  buffers (tinyinfer_amd.backend.paged_attention_decode, its allocation-free
  form, and the fast arithmetic's form for many rows);
- "forward": one chunk forward of a device context (mp_hip_forward) with
  resident weights and filled K/V pages: `decode` sequences of one new token
  each and `prefill` sequences of `chunk` new tokens each, in the fast or the
  exact arithmetic;
- "serve": an Engine that takes requests sharing a prompt prefix, prefills and
  decodes them to their end.

Every model has the SmolLM2-135M layer (hidden 576, 9 query and 3 KV heads of
64, SwiGLU 1536, tied head); "layers" and "vocabulary" of a case say how much
of the 30-layer, 49,152-token model its context holds. Contexts and prompt
lengths are spread evenly over [shortest, longest] in a fixed shuffled order.
Weights are N(0, 0.02), RMSNorm weights near 1, token ids uniform, and the
K/V already in the pages has the size that such weights give it.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from tinyinfer_amd import backend as mp
from tinyinfer_amd.host import Engine, Runner, Weights

PAGE = 16
HIDDEN, INNER, HEADS, KV_HEADS, DIM = 576, 1536, 9, 3, 64
KVW = KV_HEADS * DIM
GROUP = HEADS // KV_HEADS
EPS, THETA = 1e-5, 100000.0
LAYER_WEIGHTS = HIDDEN * (HIDDEN + 2 * KVW) + HIDDEN * HIDDEN + 3 * HIDDEN * INNER
KV_STD = 0.48  # 0.02 * sqrt(576): what a normalised row times N(0, 0.02) weights gives

F32P = ctypes.POINTER(ctypes.c_float)
I32P = ctypes.POINTER(ctypes.c_int32)


def _attend(name, arithmetic, rows, shortest, longest):
    return dict(name=name, kind="attend", arithmetic=arithmetic, rows=rows, shortest=shortest, longest=longest)


def _forward(name, arithmetic, layers, vocabulary, decode=0, shortest=0, longest=0, prefill=0, chunk=0, used=0):
    return dict(name=name, kind="forward", arithmetic=arithmetic, layers=layers, vocabulary=vocabulary, decode=decode,
                shortest=shortest, longest=longest, prefill=prefill, chunk=chunk, used=used)


def _serve(name, layers, vocabulary, requests, prefix, unique, new_tokens):
    return dict(name=name, kind="serve", layers=layers, vocabulary=vocabulary, requests=requests, prefix=prefix,
                unique=unique, new_tokens=new_tokens)


def listed():
    return [
        # The single attention operation at its usual size, one row of 503 tokens: a call's latency.
        _attend("attend_exact_503", "exact", 1, 503, 503),
        # A long document's row in a program that may not allocate.
        _attend("attend_noalloc_16640", "noalloc", 1, 16640, 16640),
        # Eight long documents decoding together.
        _attend("attend_fast_8_long", "fast", 8, 14337, 16639),
        # One user chatting: the next token of the whole model.
        _forward("decode_1", "fast", 30, 49152, decode=1, shortest=191, longest=191),
        # A server's ordinary step: 64 ragged sequences, the whole model, logits kept for sampling.
        _forward("decode_64", "fast", 30, 49152, decode=64, shortest=256, longest=2175),
        # The widest batch, 256 sequences of about a thousand tokens.
        _forward("decode_256", "fast", 8, 4096, decode=256, shortest=1024, longest=1087),
        # One request's prompt chunk while nothing else runs: time to the first token.
        _forward("prefill_1x256", "fast", 8, 4096, prefill=1, chunk=256, used=768),
        # Long prompts prefilling together, in the middle of 16k tokens.
        _forward("prefill_8x512", "fast", 4, 4096, prefill=8, chunk=512, used=8192),
        # Continuous batching: decoding sequences and the ragged last chunks of new prompts in one step.
        _forward("mixed_29_3x61", "fast", 8, 4096, decode=29, shortest=1000, longest=1127, prefill=3, chunk=61,
                 used=1003),
        # The reference's own arithmetic, bit for bit: a batch decoding.
        _forward("exact_decode_64", "exact", 4, 4096, decode=64, shortest=256, longest=2175),
        # The same for a prompt chunk.
        _forward("exact_prefill_1x256", "exact", 4, 4096, prefill=1, chunk=256, used=256),
        # A whole small service: a shared prompt prefix, copy-on-write of its tail, prefill, decode, host scheduling.
        _serve("serve_8_shared", 8, 4096, 8, 1000, 64, 8),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    case = _drawn(rng)
    del case["name"]
    return case


def _drawn(rng):
    pick = rng.random()
    if pick < 0.12:
        length = _log(rng, 17, 16640)
        return _attend("", rng.choice(["exact", "noalloc"]), 1, length, length)
    if pick < 0.24:
        longest = _log(rng, 40, 16640)
        return _attend("", "fast", _log(rng, 1, min(256, 280000 // longest)), max(1, int(longest * rng.uniform(0.1, 1))),
                       longest)
    if pick < 0.56:
        rows = _log(rng, 1, 256)
        longest = _log(rng, 64, min(8000, 280000 // rows))
        return _forward("", "fast", rng.randint(2, 8), 4096, decode=rows,
                        shortest=max(1, int(longest * rng.uniform(0.2, 1))), longest=longest)
    if pick < 0.78:
        sequences = _log(rng, 1, 8)
        return _forward("", "fast", rng.randint(2, 4), 4096, prefill=sequences, chunk=_log(rng, 5, 512),
                        used=rng.choice([0, rng.randint(1, 4096), rng.randint(1, 8192)]))
    if pick < 0.88:
        longest = _log(rng, 64, 2100)
        return _forward("", "fast", rng.randint(2, 6), 4096, decode=_log(rng, 1, 128),
                        shortest=max(1, int(longest * rng.uniform(0.2, 1))), longest=longest,
                        prefill=rng.randint(1, 4), chunk=_log(rng, 5, 256), used=rng.randint(0, 2000))
    if pick < 0.97:
        if rng.random() < 0.5:
            longest = _log(rng, 64, 2175)
            return _forward("", "exact", rng.randint(2, 4), 4096, decode=_log(rng, 1, 64),
                            shortest=max(1, int(longest * rng.uniform(0.2, 1))), longest=longest)
        return _forward("", "exact", rng.randint(2, 4), 4096, prefill=1, chunk=_log(rng, 5, 256),
                        used=rng.randint(0, 512))
    return _serve("", rng.randint(2, 6), 4096, rng.randint(1, 8), rng.randint(40, 1000), rng.randint(3, 64),
                  rng.randint(2, 8))


# ---- lengths and pages ----------------------------------------------------


def _spread(shortest, longest, rows):
    """Lengths over [shortest, longest], in an order that is not sorted."""
    return [shortest + int((longest - shortest + 0.999) * ((0.5 + 0.6180339887 * i) % 1.0)) for i in range(rows)]


def _pages(tokens):
    return -(-tokens // PAGE)


def _sequences(case):
    """(committed tokens, new tokens) per sequence of a forward case."""
    return [(n, 1) for n in _spread(case["shortest"], case["longest"], case["decode"])] + \
        [(case["used"] + 5 * i if case["prefill"] > 1 and case["chunk"] % PAGE else case["used"], case["chunk"])
         for i in range(case["prefill"])]


def _lengths(case):
    return _spread(case["shortest"], case["longest"], case["rows"])


def _generator(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(1000003 * seed + 17)


def _tables(gen, lengths, spare):
    """A page table per row, out of a shuffled pool with `spare` times the pages needed."""
    counts = [_pages(n) for n in lengths]
    blocks = math.ceil(spare * sum(counts))
    order = torch.randperm(blocks, generator=gen, device="cuda", dtype=torch.int64).to(torch.int32)
    return list(torch.split(order[: sum(counts)], counts)), blocks


# ---- weights --------------------------------------------------------------

SLOTS = (("input_norm", (HIDDEN,)), ("q", (HIDDEN, HIDDEN)), ("k", (HIDDEN, KVW)), ("v", (HIDDEN, KVW)),
         ("o", (HIDDEN, HIDDEN)), ("post_norm", (HIDDEN,)), ("gate", (HIDDEN, INNER)), ("up", (HIDDEN, INNER)),
         ("down", (INNER, HIDDEN)))


def _weights(gen, layers, vocabulary):
    """{"embedding", "final_norm", "layers": [{slot: tensor}]} on the GPU, projections [in, out]."""
    def normal(shape):
        return torch.randn(shape, generator=gen, device="cuda") * 0.02

    def norm():
        return 1.0 + 0.1 * torch.randn(HIDDEN, generator=gen, device="cuda")

    return {"embedding": normal((vocabulary, HIDDEN)), "final_norm": norm(),
            "layers": [{n: norm() if len(s) == 1 else normal(s) for n, s in SLOTS} for _ in range(layers)]}


def _model(layers, vocabulary, context):
    return dict(layers=layers, hidden=HIDDEN, intermediate=INNER, heads=HEADS, kv_heads=KV_HEADS,
                vocabulary=vocabulary, context=context, rms_epsilon=EPS, rope_theta=THETA, tied=1, eos=0)


class _Pool:
    """A device context's K or V pool as a tensor that keeps the context alive."""

    def __init__(self, owner, pointer, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (pointer, False), "version": 2}


def _pools(context):
    """The K and V pools [block, layer, KV head, 16, 64, 4 | 4, 64, 4] in the device's page order."""
    k, v, n = context.kv_pools()
    shape = (context.max_blocks, n // (context.max_blocks * PAGE * KVW), KV_HEADS, PAGE * DIM)
    return [torch.as_tensor(_Pool(context, p, shape), device="cuda") for p in (k, v)]


# ---- the state before the call --------------------------------------------


def _prepare_attend(case, seed):
    gen = _generator(seed)
    lengths = _lengths(case)
    tables, blocks = _tables(gen, lengths, 1.25)
    stride = max(t.numel() for t in tables)
    table = torch.zeros((len(tables), stride), dtype=torch.int32, device="cuda")
    for row, t in zip(table, tables):
        row[: t.numel()] = t
    shape = (blocks, 1, PAGE * KVW)
    q = torch.randn((len(lengths), HEADS * DIM), generator=gen, device="cuda")
    keys = torch.randn(shape, generator=gen, device="cuda")
    values = torch.randn(shape, generator=gen, device="cuda")
    return dict(case=case, q=q, keys=keys, values=values, table=table, out=torch.empty_like(q),
                lengths=np.asarray(lengths, dtype=np.int32), stride=stride)


def _prepare_forward(case, seed):
    gen = _generator(seed)
    sequences = _sequences(case)
    longest = max(used + count for used, count in sequences)
    weights = _weights(gen, case["layers"], case["vocabulary"])
    tables, blocks = _tables(gen, [used + count for used, count in sequences], 1.25)
    context = mp.HipBackend(_model(case["layers"], case["vocabulary"], longest + 64), PAGE, blocks,
                            max_sequences=len(sequences),
                            arithmetic=mp.ARITHMETIC_FAST if case["arithmetic"] == "fast" else mp.ARITHMETIC_EXACT)
    context.upload(-1, mp.TENSOR_EMBEDDING, weights["embedding"].cpu().numpy())
    context.upload(-1, mp.TENSOR_FINAL_NORM, weights["final_norm"].cpu().numpy())
    for i, layer in enumerate(weights["layers"]):
        for slot, (name, _) in enumerate(SLOTS):
            context.upload(i, slot, layer[name].cpu().numpy())
    for i, t in enumerate(tables):
        context.table_write(i, 0, t.cpu().numpy())
    context.sync()
    pools = _pools(context)
    for pool in pools:
        pool.copy_(torch.randn(pool.shape, generator=gen, device="cuda").mul_(KV_STD))
    rows = sum(count for _, count in sequences)
    tokens = torch.randint(case["vocabulary"], (rows,), generator=gen, device="cuda").to(torch.int32).cpu().numpy()
    logits = torch.empty((len(sequences), case["vocabulary"]), dtype=torch.float32, pin_memory=True)
    argmax = torch.empty(len(sequences), dtype=torch.int32)
    torch.cuda.synchronize()
    steps = (mp.SeqStep * len(sequences))(*[mp.SeqStep(i, u, c) for i, (u, c) in enumerate(sequences)])
    return dict(case=case, context=context, steps=steps, count=len(sequences), tokens=tokens, logits=logits,
                argmax=argmax, pools=pools, tables=tables, sequences=sequences,
                call=(context.handle, steps, len(sequences), tokens.ctypes.data_as(I32P),
                      ctypes.cast(logits.data_ptr(), F32P), ctypes.cast(argmax.data_ptr(), I32P), None))


def _prompts(case, seed):
    """The shared prefix and each request's whole prompt, with different first own tokens."""
    rng = np.random.default_rng(seed)
    vocabulary = case["vocabulary"]
    prefix = rng.integers(0, vocabulary, case["prefix"]).astype(np.int32)
    own = rng.integers(0, vocabulary, (case["requests"], case["unique"])).astype(np.int32)
    own[:, 0] = rng.permutation(vocabulary)[: case["requests"]]
    return prefix, [np.concatenate([prefix, o]) for o in own]


def _prepare_serve(case, seed):
    prefix, prompts = _prompts(case, seed)
    context = len(prompts[0]) + case["new_tokens"] + 64
    weights = Weights.synthetic(_model(case["layers"], case["vocabulary"], context), seed=seed)
    pages = _pages(len(prefix)) + sum(_pages(len(p) + case["new_tokens"]) for p in prompts)
    blocks = math.ceil(1.25 * pages)
    runner = Runner(weights, context=context, block_tokens=PAGE, max_blocks=blocks, prefix_cache_blocks=blocks, kind=2)
    runner.keep_logits()
    engine = Engine(runner, max_batch_size=32, token_budget=2048, prefill_chunk=64, context=context)
    engine.set_batching(True)
    return dict(case=case, engine=engine, runner=runner, weights=weights, prefix=prefix, prompts=prompts, served=0)


def prepare(case, seed):
    return {"attend": _prepare_attend, "forward": _prepare_forward, "serve": _prepare_serve}[case["kind"]](case, seed)


# ---- the call -------------------------------------------------------------


def _run_attend(state):
    case = state["case"]
    stream = torch.cuda.current_stream().cuda_stream
    q, keys, values = state["q"].data_ptr(), state["keys"].data_ptr(), state["values"].data_ptr()
    table, out = state["table"].data_ptr(), state["out"].data_ptr()
    if case["arithmetic"] == "fast":
        mp.paged_attention_decode_fast(q, keys, values, table, state["stride"], state["lengths"], 0, 1, HEADS,
                                       KV_HEADS, out, stream)
    else:
        call = mp.paged_attention_decode if case["arithmetic"] == "exact" else mp.paged_attention_decode_noalloc
        call(q, keys, values, table, int(state["lengths"][0]), 0, 1, PAGE, HEADS, KV_HEADS, DIM, out, stream)
    return state["out"]


def _run_forward(state):
    context = state["context"]
    status = context.lib.mp_hip_forward(*state["call"])
    if status:
        raise mp.BackendError(status, context.lib.mp_hip_last_error(context.handle).decode())
    out = {"logits": state["logits"], "argmax": state["argmax"]}
    if state["case"]["prefill"]:
        # A prompt's K/V is what its chunk leaves behind.
        out["keys"], out["values"] = state["pools"]
    return out


def _run_serve(state):
    case, engine, runner = state["case"], state["engine"], state["runner"]
    tag = state["served"]
    state["served"] += 1
    # The prefix's own request publishes it; the others reuse its pages.
    engine.submit(f"{tag}.prefix", state["prefix"], 1)
    while not engine.idle():
        engine.step()
    ids = [f"{tag}.{i}" for i in range(case["requests"])]
    for rid, prompt in zip(ids, state["prompts"]):
        engine.submit(rid, prompt, case["new_tokens"])
    tokens = {rid: [] for rid in ids}
    while not engine.idle():
        engine.step()
        for event in engine.poll_events():
            if event["id"] in tokens:
                tokens[event["id"]].append(event["token"])
    logits = np.stack([runner.kept_logits(rid) for rid in ids])
    runner.clear()
    return {"tokens": np.asarray([tokens[rid] for rid in ids], dtype=np.int64), "logits": logits}


def run(state):
    return {"attend": _run_attend, "forward": _run_forward, "serve": _run_serve}[state["case"]["kind"]](state)


# ---- what a pass cannot do without ----------------------------------------


def _forward_work(sequences, layers, vocabulary, heads_out):
    rows = sum(c for _, c in sequences)
    # Query-key pairs of every row; K/V of every attended token is read once per sequence.
    pairs = sum(c * u + c * (c + 1) // 2 for u, c in sequences)
    tokens = sum(u + c for u, c in sequences)
    flops = layers * (2 * rows * LAYER_WEIGHTS + 4 * HEADS * DIM * pairs) + 2 * heads_out * vocabulary * HIDDEN
    bytes_ = 4 * (layers * LAYER_WEIGHTS + vocabulary * HIDDEN + heads_out * vocabulary +
                  layers * 2 * KVW * (tokens + rows))
    return bytes_, flops


def work(case):
    if case["kind"] == "attend":
        tokens = sum(_lengths(case))
        return {"bytes": 4 * (2 * KVW * tokens + 2 * case["rows"] * HEADS * DIM), "flops": 4 * HEADS * DIM * tokens}
    if case["kind"] == "forward":
        sequences = _sequences(case)
        b, f = _forward_work(sequences, case["layers"], case["vocabulary"], len(sequences))
        return {"bytes": b, "flops": f}
    # The prefix once, every request's own tokens as one chunk, then single tokens.
    args, n = (case["layers"], case["vocabulary"]), case["requests"]
    total = [list(_forward_work([(0, case["prefix"])], *args, 1))]
    total.append(_forward_work([(case["prefix"], case["unique"])] * n, *args, n))
    for i in range(case["new_tokens"] - 1):
        total.append(_forward_work([(case["prefix"] + case["unique"] + i, 1)] * n, *args, n))
    return {"bytes": sum(t[0] for t in total), "flops": sum(t[1] for t in total)}


def tolerance(case):
    # The exact arithmetic promises the reference's bits.
    if case.get("arithmetic") in ("exact", "noalloc"):
        return "exact"
    # 32-bit sums in another order: one attention, and up to 30 layers of them.
    if case["kind"] == "attend":
        return {"rel": 1e-6, "max": 2e-5}
    # Ties of the two largest logits may go either way.
    return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}


# ---- the same in 64 bits, in plain torch ----------------------------------


def _pages64(pool_keys, pool_values, table, tokens):
    """K and V [KV head, token, 64] in 64 bits of one layer's pages in the device's page order."""
    at = table.long()
    k = pool_keys[at].double().view(-1, KV_HEADS, DIM // 4, PAGE, 4).permute(1, 0, 3, 2, 4)
    v = pool_values[at].double().view(-1, KV_HEADS, PAGE // 4, DIM, 4).permute(1, 0, 2, 4, 3)
    return [x.reshape(KV_HEADS, -1, DIM)[:, :tokens] for x in (k, v)]


def _attention64(q, k, v, first):
    """q [rows, heads, 64] at positions first.. over k, v [KV heads, tokens, 64]."""
    rows, tokens = q.shape[0], k.shape[1]
    hidden = torch.arange(tokens, device=q.device)[None, :] > first + torch.arange(rows, device=q.device)[:, None]
    out = []
    for h in range(HEADS):
        s = (q[:, h] @ k[h // GROUP].T.contiguous()) * DIM ** -0.5
        out.append(torch.softmax(s.masked_fill(hidden, -math.inf), dim=1) @ v[h // GROUP])
    return torch.stack(out, dim=1).reshape(rows, HEADS * DIM)


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS) * w


def _rope64(x, positions):
    half = DIM // 2
    # The angles as the model defines them, in 32 bits.
    power = torch.tensor(THETA, dtype=torch.float32) ** (torch.arange(0, DIM, 2, dtype=torch.float32) / DIM)
    angle = positions.float().cpu()[:, None] / power[None, :]
    cos, sin = (f(angle).to(x.device).double()[:, None, :] for f in (torch.cos, torch.sin))
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _chunk64(weights, tokens, used, history):
    """Last-row logits of one sequence's chunk; history[layer] is its [K, V], extended in place."""
    x = weights["embedding"][tokens.long()].double()
    rows = x.shape[0]
    positions = torch.arange(used, used + rows, device=x.device)
    for layer, w in enumerate(weights["layers"]):
        n = _rms64(x, w["input_norm"].double())
        q, k, v = (n @ w[s].double() for s in ("q", "k", "v"))
        q = _rope64(q.view(rows, HEADS, DIM), positions)
        k = _rope64(k.view(rows, KV_HEADS, DIM), positions)
        keys, values = history[layer]
        keys = torch.cat([keys, k.transpose(0, 1)], dim=1)
        values = torch.cat([values, v.view(rows, KV_HEADS, DIM).transpose(0, 1)], dim=1)
        history[layer] = [keys, values]
        x = x + _attention64(q, keys, values, used) @ w["o"].double()
        n = _rms64(x, w["post_norm"].double())
        gate = n @ w["gate"].double()
        x = x + (gate / (1 + torch.exp(-gate)) * (n @ w["up"].double())) @ w["down"].double()
    last = _rms64(x[-1:], weights["final_norm"].double())
    return (last @ weights["embedding"].double().T.contiguous())[0]


def _exact_attend(case, seed):
    state = _prepare_attend(case, seed)
    out = []
    for r, n in enumerate(state["lengths"].tolist()):
        table = state["table"][r, : _pages(n)]
        if case["arithmetic"] == "fast":
            k, v = _pages64(state["keys"][:, 0], state["values"][:, 0], table, n)
        else:  # the reference's page order [slot][KV head][64]
            k, v = (p[table.long(), 0].double().view(-1, KV_HEADS, DIM)[:n].transpose(0, 1)
                    for p in (state["keys"], state["values"]))
        out.append(_attention64(state["q"][r].double().view(1, HEADS, DIM), k, v, n - 1))
    return torch.cat(out)


def _exact_forward(case, seed):
    # The weights are the generator's first draws in _prepare_forward too.
    weights = _weights(_generator(seed), case["layers"], case["vocabulary"])
    state = _prepare_forward(case, seed)
    pools = state["pools"]
    after = [p.double() for p in pools] if case["prefill"] else None
    logits, at = [], 0
    tokens = torch.from_numpy(state["tokens"]).cuda()
    for (used, count), table in zip(state["sequences"], state["tables"]):
        history = [_pages64(pools[0][:, l], pools[1][:, l], table, used) for l in range(case["layers"])]
        logits.append(_chunk64(weights, tokens[at: at + count], used, history))
        at += count
        if after is None:
            continue
        positions = torch.arange(used, used + count, device="cuda")
        blocks, slots = table.long()[positions // PAGE], positions % PAGE
        for l in range(case["layers"]):
            # Indexing with two index tensors puts their dimension first: [count, KV head, ...].
            k = after[0][:, l].view(-1, KV_HEADS, DIM // 4, PAGE, 4)
            v = after[1][:, l].view(-1, KV_HEADS, PAGE // 4, DIM, 4)
            new_k, new_v = (h[:, used:].transpose(0, 1) for h in history[l])
            k[blocks, :, :, slots] = new_k.reshape(count, KV_HEADS, DIM // 4, 4)
            v[blocks, :, slots // 4, :, slots % 4] = new_v
    out = {"logits": torch.stack(logits), "argmax": None}
    if after is not None:
        out["keys"], out["values"] = after
    return out


def _exact_serve(case, seed):
    prefix, prompts = _prompts(case, seed)
    config = _model(case["layers"], case["vocabulary"], len(prompts[0]) + case["new_tokens"] + 64)
    given = Weights.synthetic(config, seed=seed)
    names = {"input_norm": "input_layernorm", "post_norm": "post_attention_layernorm", "q": "self_attn.q_proj",
             "k": "self_attn.k_proj", "v": "self_attn.v_proj", "o": "self_attn.o_proj", "gate": "mlp.gate_proj",
             "up": "mlp.up_proj", "down": "mlp.down_proj"}

    def tensor(name, shape):
        return torch.from_numpy(given.tensor(name)).cuda().view(shape)

    weights = {"embedding": tensor("model.embed_tokens.weight", (case["vocabulary"], HIDDEN)),
               "final_norm": tensor("model.norm.weight", (HIDDEN,)),
               "layers": [{n: tensor(f"model.layers.{l}.{names[n]}.weight", s) for n, s in SLOTS}
                          for l in range(case["layers"])]}
    logits = []
    empty = torch.zeros((KV_HEADS, 0, DIM), dtype=torch.float64, device="cuda")
    for prompt in prompts:
        history = [[empty, empty] for _ in range(case["layers"])]
        used, chunk = 0, torch.from_numpy(prompt).cuda()
        for _ in range(case["new_tokens"]):
            last = _chunk64(weights, chunk, used, history)
            used += chunk.numel()
            chunk = torch.argmax(last).view(1)
        logits.append(last)
    return {"tokens": None, "logits": torch.stack(logits)}


def exact(case, seed):
    return {"attend": _exact_attend, "forward": _exact_forward, "serve": _exact_serve}[case["kind"]](case, seed)
