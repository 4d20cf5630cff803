"""The work this engine is measured by: prompts read in, tokens decoded, both at once, and requests
through the engine's own loop, at the layer sizes of the 4B presets.

A case is a dict of plain values. ``kind`` says what one pass does:

* ``read``: prompts go through the step function in steps of at most ``budget`` tokens; the logits
  at every prompt's last token come back.
* ``decode``: requests whose context is in the cache decode ``steps`` tokens each, one step of the
  whole batch after the other; the logits of every step come back. The next pass goes on where this
  one stopped, as a running request does; after ``ROOM`` tokens the contexts are read in anew.
* ``mix``: requests come in one after another, prompts are read in portions beside the tokens of
  those that decode already (a step holds at most ``budget`` tokens); the logits after every prompt
  and of every decoded token come back.
* ``score``: requests with given continuations through ``Engine.add_request`` and ``Engine.step``:
  scheduler, step function, sampler; tokens and their log-probabilities come back.

The ids that requests go on with are given in every kind, so that two implementations that differ
by rounding read the same tokens. Weights are seeded and random, in bfloat16, N(0, 0.02) as in the
repository's own benchmark but for the matrices (and norms) that lead back into the residual stream:
those are smaller, so that a layer changes the stream by a few per cent of itself, as in a trained
model, and does not replace it, which would amplify rounding from layer to layer. ``exact`` draws the
same weights and computes the models in float64.
"""

from __future__ import annotations

import hashlib
import math
import random

import torch

DEVICE = "cuda:0"
PAGE = 16
ROOM = 1536      # tokens a ``decode`` request may grow by before its context is read in anew
# standard deviations of the matrices that lead back into the residual stream
BACK = {"o": 1e-4, "o_proj": 1e-4, "down": 1e-5, "down_proj": 1e-5}
WARM_STEPS = 3   # decode steps that ``prepare`` runs: the first ones of a size are slower than the rest


def listed():
    qwen, deginex, roserax = "qwen3_4b", "deginex_4b_moe", "roserax_4b"
    return [
        # one user waits for the next word: every weight is read for one token, launches count
        _decode("decode 1", qwen, 1, 2049, 2049, 4),
        # the repository's headline: a batch of eight behind 2,048-token prompts
        _decode("decode 8", qwen, 8, 2049, 2049, 8),
        # a busy server: contexts of very unequal lengths
        _decode("decode 48 ragged", qwen, 48, 131, 2601, 4),
        # time to the first token of an ordinary prompt
        _read("read 2048", qwen, 1, 2048, 2048, 2048),
        # a long document, read in portions over a growing history; its length divides by nothing
        _read("read 8191 in portions", qwen, 1, 8191, 8191, 2048),
        # continuous batching: portions of prompts beside decoding requests
        {"name": "continuous batching", "kind": "mix", "model": qwen, "dtype": "bfloat16", "requests": 10,
         "shortest": 77, "longest": 1501, "steps": 12, "budget": 512},
        # short prompts and given continuations through the engine's own loop
        {"name": "score 6 short requests", "kind": "score", "model": qwen, "dtype": "bfloat16", "requests": 6,
         "shortest": 19, "longest": 307, "steps": 16, "budget": 2048},
        # the true 32-bit mode, short prompts and a few tokens: what checks of numerics run
        {"name": "float32 2 requests", "kind": "mix", "model": qwen, "dtype": "float32", "requests": 2,
         "shortest": 93, "longest": 261, "steps": 6, "budget": 512},
        # routed experts over several residual streams
        _read("experts read 3 prompts", deginex, 3, 301, 1151, 2048),
        _decode("experts decode 8", deginex, 8, 1025, 1025, 8),
        # latent attention, retention, windows and experts
        _read("latent read 2047", roserax, 1, 2047, 2047, 2048),
        _decode("latent decode 8", roserax, 8, 1025, 1025, 8),
    ]


def draw(rng):
    """One more case of the ranges above."""
    spread = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    kind = rng.choice(("read", "read", "decode", "decode", "mix", "score"))
    model = rng.choice(("qwen3_4b", "qwen3_4b", "deginex_4b_moe", "roserax_4b"))
    if kind == "read":
        requests = rng.choice((1, 1, 2, 5))
        longest = spread(65, 2900)
        return _read(None, model, requests, max(17, longest // rng.choice((1, 2, 7))), longest, 2048)
    if kind == "decode":
        requests = spread(1, 40)
        longest = spread(70, 2600 if requests <= 16 else 1200)
        return _decode(None, model, requests, max(33, longest // rng.choice((1, 1, 3, 9))), longest, rng.choice((3, 5)))
    dtype = "float32" if rng.random() < 0.3 else "bfloat16"
    longest = spread(40, 220 if dtype == "float32" else 900)
    case = {"kind": kind, "model": "qwen3_4b" if dtype == "float32" else model, "dtype": dtype,
            "requests": rng.randint(1, 2 if dtype == "float32" else 7), "shortest": max(11, longest // rng.choice((1, 2, 5))),
            "longest": longest, "steps": rng.randint(3, 5 if dtype == "float32" else 9), "budget": rng.choice((256, 512, 2048))}
    return case


def _case(name, kind, model, requests, shortest, longest, **more):
    case = {"kind": kind, "model": model, "dtype": "bfloat16", "requests": requests, "shortest": shortest,
            "longest": longest, **more}
    return case if name is None else {"name": name, **case}


def _read(name, model, requests, shortest, longest, budget):
    return _case(name, "read", model, requests, shortest, longest, budget=budget)


def _decode(name, model, requests, shortest, longest, steps):
    return _case(name, "decode", model, requests, shortest, longest, steps=steps)


def lengths(case):
    """Prompt lengths, from the shortest to the longest with equal ratios, in a mixed order."""
    n, lo, hi = case["requests"], case["shortest"], case["longest"]
    out = [hi] if n == 1 else [int(round(lo * (hi / lo) ** (i / (n - 1)))) for i in range(n)]
    random.Random(n).shuffle(out)
    return out


# ------------------------------------------------------------------ inputs
def drawn(seed, name, shape):
    """A weight as stored: bfloat16 on the device, from the seed and its own name."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int.from_bytes(hashlib.sha256(f"{seed}/{name}".encode()).digest()[:7], "little"))
    x = torch.randn(shape, generator=gen, dtype=torch.float32, device=DEVICE)
    leaf = name.removesuffix(".weight").rsplit(".", 1)[-1]
    if "norm" in leaf:
        x = (3e-4 if leaf in ("norm1b", "norm2b") else 1.0) * (1.0 + 0.1 * x)
    elif ".hc" in name:  # coefficients of several residual streams: near one, near the identity
        x = 0.1 * x + (torch.eye(shape[0], device=DEVICE) if name.endswith(".mix") else 1.0)
    else:
        x = BACK.get(leaf, 0.02) * x
    return x.to(torch.bfloat16)


class Weights:
    """The tensors a model declares, by name, as a model folder would hold them."""

    def __init__(self, decls, seed):
        self.shapes = {d.file_name: tuple(d.shape) for d in decls}
        self.seed = seed

    def names(self):
        return sorted(self.shapes)

    def has(self, name):
        return name in self.shapes

    def shape(self, name):
        return self.shapes[name]

    def dtype(self, name):
        return torch.bfloat16

    def get(self, name, device=DEVICE):
        return drawn(self.seed, name, self.shapes[name]).to(device)


def ids_of(case, seed, vocab):
    """Per request: its prompt and the ids it goes on with."""
    gen = torch.Generator().manual_seed(seed * 7919 + 11)
    take = lambda n: torch.randint(0, vocab, (n,), generator=gen).tolist()  # noqa: E731
    more = {"read": 0, "decode": WARM_STEPS + ROOM}.get(case["kind"], case.get("steps", 0))
    return [(take(n), take(more)) for n in lengths(case)]


# ------------------------------------------------------------------ the engine at work
class State:
    def __init__(self, case, seed):
        from qwen3_runtime_amd.config.engine import EngineConfig
        from qwen3_runtime_amd.engine.engine import Engine
        from qwen3_runtime_amd.engine.factory import build_model, load
        from qwen3_runtime_amd.registry import preset_config

        self.case = case
        raw = preset_config(case["model"])
        _, model = build_model(raw)
        vocab = model.plan.vocab_size
        self.requests = ids_of(case, seed, vocab)
        pages = sum(-(-(len(p) + len(m) + 2) // PAGE) + 1 for p, m in self.requests)
        config = EngineConfig(page_size=PAGE, num_pages=pages, max_num_seqs=len(self.requests), dtype=case["dtype"],
                              max_num_batched_tokens=case.get("budget", 2048), device=DEVICE)
        self.engine = Engine(config, load(None, config, source=Weights(model.tensor_decls(), seed), raw_config=raw))
        self.runner, self.cache = self.engine.runner, self.engine.cache
        self.passes = self.done = 0


def prepare(case, seed):
    s = State(case, seed)
    if case["kind"] == "decode":
        _begin(s)
    else:  # a server that has served before: the same sizes, other ids
        kept = s.requests
        s.requests = ids_of(case, seed + 1_000_003, s.runner.vocab_size)
        for _ in range(1 if case["kind"] == "read" else 2):
            run(s)
        s.requests = kept
    torch.cuda.synchronize()
    return s


def run(s):
    return {"read": _run_read, "decode": _run_decode, "mix": _run_mix, "score": _run_score}[s.case["kind"]](s)


def _steps_of(prompts, budget):
    """Prompts in order, cut into steps of at most ``budget`` tokens: lists of (request, from, to)."""
    steps, left = [[]], budget
    for i, p in enumerate(prompts):
        at = 0
        while at < len(p):
            n = min(left, len(p) - at)
            steps[-1].append((i, at, at + n))
            at, left = at + n, left - n
            if left == 0:
                steps.append([])
                left = budget
    return [step for step in steps if step]


def _admit(s):
    rids = [f"{s.passes}.{i}" for i in range(len(s.requests))]
    s.passes += 1
    for rid in rids:
        s.cache.admit(rid)
    return rids


def _read_prompts(s, rids, budget, wanted=True):
    """All prompts into the cache; the logits at their last tokens, in the requests' order."""
    from qwen3_runtime_amd.engine.batch import StepEntry

    prompts = [p for p, _ in s.requests]
    rows = []
    for step in _steps_of(prompts, budget):
        entries = [StepEntry(rids[i], prompts[i][a:b], [b - a - 1] if wanted and b == len(prompts[i]) else [])
                   for i, a, b in step]
        logits = s.runner.step(entries)
        if logits is not None:
            rows.append(logits)
    return rows


def _run_read(s):
    rids = _admit(s)
    rows = _read_prompts(s, rids, s.case["budget"])
    for rid in rids:
        s.cache.release(rid)
    return rows[0] if len(rows) == 1 else torch.cat(rows)


def _decode_step(s, rids):
    from qwen3_runtime_amd.engine.batch import StepEntry

    at = s.done
    s.done += 1
    return s.runner.step([StepEntry(rid, [m[at]], [0]) for rid, (_, m) in zip(rids, s.requests)])


def _begin(s):
    s.rids, s.done = _admit(s), 0
    _read_prompts(s, s.rids, 2048, wanted=False)
    for _ in range(WARM_STEPS):
        _decode_step(s, s.rids)


def _run_decode(s):
    steps = s.case["steps"]
    if s.done + steps > WARM_STEPS + ROOM:
        for rid in s.rids:
            s.cache.release(rid)
        _begin(s)
    # a replayed step's logits lie in the step's own buffer: whoever keeps them copies them
    return torch.stack([_decode_step(s, s.rids).clone() for _ in range(steps)])


def _run_mix(s):
    from qwen3_runtime_amd.engine.batch import StepEntry

    rids, budget, steps = _admit(s), s.case["budget"], s.case["steps"]
    at, out, live = [0] * len(rids), [[] for _ in rids], list(range(len(rids)))
    while live:
        left, entries, who = budget, [], []
        for i in live:
            prompt, more = s.requests[i]
            if at[i] >= len(prompt):
                tokens, want = [more[at[i] - len(prompt)]], [0]
            else:
                tokens = prompt[at[i]: at[i] + left]
                want = [len(tokens) - 1] if tokens and at[i] + len(tokens) == len(prompt) else []
            if not tokens or left <= 0:
                break
            left -= len(tokens)
            entries.append(StepEntry(rids[i], tokens, want))
            who.append(i)
        logits = s.runner.step(entries)
        row, logits = 0, None if logits is None else logits.clone()
        for i, e in zip(who, entries):
            at[i] += len(e.tokens)
            if e.want:
                out[i].append(logits[row])
                row += 1
            if at[i] == len(s.requests[i][0]) + steps:
                s.cache.release(rids[i])
                live.remove(i)
    return torch.stack([row for rows in out for row in rows])


def _run_score(s):
    engine = s.engine
    reqs = [engine.request(engine.add_request(p, max_tokens=len(m), forced_tokens=m)) for p, m in s.requests]
    while not engine.is_finished():
        engine.step()
    return {"tokens": torch.tensor([r.output_tokens for r in reqs]),
            "logprobs": torch.tensor([r.logprobs for r in reqs], dtype=torch.float32)}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    """Every step reads the weights it uses, the cache of its requests' visible tokens, and writes
    logits; operations are the products' and the attention's, as the model's parts count them."""
    from qwen3_runtime_amd.engine.factory import build_model
    from qwen3_runtime_amd.registry import preset_config

    _, model = build_model(preset_config(case["model"]))
    width = 4 if case["dtype"] == "float32" else 2
    total = {"bytes": 0.0, "flops": 0.0}

    def step(spans, rows):
        cost = model.step_cost(spans, rows, width)
        total["flops"] += cost.flop
        total["bytes"] += cost.total_weight_bytes + 4.0 * rows * model.plan.vocab_size
        for spec in model.plan.caches:
            if spec.paged:
                seen = sum(min(kv, spec.window + spec.keep_first) if spec.window else kv for _, kv in spans)
                total["bytes"] += seen * spec.elements_per_token() * width
            else:
                total["bytes"] += 2.0 * len(spans) * math.prod(spec.shape) * 4

    sizes, steps = lengths(case), case.get("steps", 0)
    if case["kind"] == "decode":
        for k in range(steps):
            step([(1, n + WARM_STEPS + k + 1) for n in sizes], len(sizes))
    else:
        for part in _steps_of([range(n) for n in sizes], case["budget"]):
            step([(b - a, b) for _, a, b in part], sum(b == sizes[i] for i, a, b in part))
        for k in range(steps - (case["kind"] == "score")):
            step([(1, n + k + 1) for n in sizes], len(sizes))
    return total


def tolerance(case):
    """About four times the distance from float64 that was measured: 0.002 to 0.003 for bfloat16
    logits (the roundings of activations, and of the final norm above all), 0.0001 for log-probabilities,
    1.7e-6 for float32."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5}
    return {"rel": 5e-4} if case["kind"] == "score" else {"rel": 0.01}


# ------------------------------------------------------------------ the same in float64
def exact(case, seed):
    from qwen3_runtime_amd.registry import preset_config

    raw = preset_config(case["model"])
    vocab = raw.get("vocab_size") or raw["vocab"]
    form = {"qwen3_4b": _qwen3, "deginex_4b_moe": _deginex, "roserax_4b": _roserax}[case["model"]]
    seqs, wanted = [], []
    for p, m in ids_of(case, seed, vocab):
        if case["kind"] == "decode":
            n = WARM_STEPS + case["steps"]
            seqs.append(p + m[:n])
            wanted.append(list(range(len(p) + WARM_STEPS, len(p) + n)))
        elif case["kind"] == "score":
            seqs.append(p + m[:-1])
            wanted.append(list(range(len(p) - 1, len(p) + len(m) - 1)))
        else:
            seqs.append(p + m)
            wanted.append(list(range(len(p) - 1, len(p) + len(m))))
    with torch.no_grad():
        hidden, table = form(raw, lambda name, *shape: drawn(seed, name, shape).double(), seqs, wanted)
        logits = [h @ table.T for h in hidden]
        if case["kind"] == "decode":
            return torch.stack(logits, dim=1)
        if case["kind"] == "score":
            tokens = torch.tensor([m for _, m in ids_of(case, seed, vocab)], device=DEVICE)
            return {"tokens": tokens, "logprobs": torch.stack(
                [x.log_softmax(-1).gather(1, t[:, None])[:, 0] for x, t in zip(logits, tokens)])}
        return torch.cat(logits)


def _rms(x, w, eps):
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w + b


def _turn(x, base):
    """Rotation of the last dimension by position (first half against second), x [T, heads, D]."""
    t, _, d = x.shape
    freq = base ** (-torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)
    angle = torch.arange(t, dtype=torch.float64, device=x.device)[:, None, None] * freq
    a, b = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1)


def _attend(q, k, v, scale, hidden_from=None, cap=None, sink=False):
    """Causal attention of one sequence, q [T, Hq, D], k [T, Hk, D], v [T, Hk, Dv]; ``hidden_from`` is a
    mask of (query, key) pairs beyond the causal one that are not seen."""
    t, nq, nk = q.shape[0], q.shape[1], k.shape[1]
    group, out = nq // nk, q.new_empty(t, nq, v.shape[2])
    unseen = torch.ones(t, t, dtype=torch.bool, device=q.device).triu(1)
    if hidden_from is not None:
        i = torch.arange(t, device=q.device)
        unseen |= hidden_from(i[:, None], i[None, :])
    for h in range(nk):
        s = torch.matmul(q[:, h * group: (h + 1) * group].transpose(0, 1), k[:, h].T).mul_(scale)
        if cap is not None:
            s = s.div_(cap).tanh_().mul_(cap)
        s.masked_fill_(unseen, -math.inf)
        if sink:
            s = torch.cat([s, s.new_zeros(*s.shape[:2], 1)], -1)
        p = s.softmax(-1)
        out[:, h * group: (h + 1) * group] = torch.matmul(p[..., :t], v[:, h]).transpose(0, 1)
    return out.reshape(t, -1)


def _silu(x):
    return x * torch.sigmoid(x)


def _each(seqs, x, f):
    """``f`` over the rows of every sequence."""
    return torch.cat([f(part) for part in x.split([len(s) for s in seqs])])


def _rows(seqs, wanted, x):
    return [part[w] for part, w in zip(x.split([len(s) for s in seqs]), wanted)]


def _qwen3(c, w, seqs, wanted):
    h, d, eps, ff = c["hidden_size"], c["head_dim"], c["rms_norm_eps"], c["intermediate_size"]
    nq, nk = c["num_attention_heads"], c["num_key_value_heads"]
    table = w("model.embed_tokens.weight", c["vocab_size"], h)
    x = table[torch.tensor([t for s in seqs for t in s], device=DEVICE)]
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        a = p + "self_attn."
        n = _rms(x, w(p + "input_layernorm.weight", h), eps)
        q = _rms((n @ w(a + "q_proj.weight", nq * d, h).T).view(-1, nq, d), w(a + "q_norm.weight", d), eps)
        k = _rms((n @ w(a + "k_proj.weight", nk * d, h).T).view(-1, nk, d), w(a + "k_norm.weight", d), eps)
        v = (n @ w(a + "v_proj.weight", nk * d, h).T).view(-1, nk, d)
        qkv = torch.cat([q, k, v], 1)
        y = _each(seqs, qkv, lambda z: _attend(_turn(z[:, :nq], c["rope_theta"]), _turn(z[:, nq: nq + nk], c["rope_theta"]),
                                               z[:, nq + nk:], d ** -0.5))
        x = x + y @ w(a + "o_proj.weight", h, nq * d).T
        n = _rms(x, w(p + "post_attention_layernorm.weight", h), eps)
        x = x + (_silu(n @ w(p + "mlp.gate_proj.weight", ff, h).T) * (n @ w(p + "mlp.up_proj.weight", ff, h).T)) \
            @ w(p + "mlp.down_proj.weight", h, ff).T
    norm = w("model.norm.weight", h)
    return [_rms(r, norm, eps) for r in _rows(seqs, wanted, x)], table


def _experts(n, w, p, mlp, index, weight):
    """Sum of the chosen experts' outputs, expert by expert over its own rows."""
    h, ff, out = n.shape[1], mlp["expert"]["ff"], torch.zeros_like(n)
    for e in range(mlp["router"]["experts"]):
        rows, which = torch.nonzero(index == e, as_tuple=True)
        if rows.numel():
            g, u, d = (w(f"{p}e{e}.{part}", *shape) for part, shape in (("gate", (ff, h)), ("up", (ff, h)), ("down", (h, ff))))
            y = (_silu(n[rows] @ g.T) * (n[rows] @ u.T)) @ d.T
            out.index_add_(0, rows, y * weight[rows, which][:, None])
    return out


def _deginex(c, w, seqs, wanted):
    h, eps, streams = c["width"], c["norm"]["eps"], c["streams"]
    table = w("embed", c["vocab"], h)
    x = table[torch.tensor([t for s in seqs for t in s], device=DEVICE)].repeat(streams, 1, 1)

    def mixer(n, p, m):
        nq, nk, d, chunk = m["heads"], m["kv_heads"], m["dim"], m["mask"]["size"]
        q, k, v = ((n @ w(p + s, heads * d, h).T).view(-1, heads, d) for s, heads in (("q", nq), ("k", nk), ("v", nk)))
        qkv = torch.cat([_rms(q, None, eps), _rms(k, None, eps), v], 1)
        y = _each(seqs, qkv, lambda z: _attend(z[:, :nq], z[:, nq: nq + nk], z[:, nq + nk:], m["scale"], cap=m["softcap"],
                                               hidden_from=lambda i, j: i // chunk != j // chunk))
        return (y * torch.sigmoid(n @ w(p + "g", nq * d, h).T)) @ w(p + "o", h, nq * d).T

    def feed_forward(n, p, m):
        if m["kind"] == "dense":
            return (_silu(n @ w(p + "gate", m["ff"], h).T) * (n @ w(p + "up", m["ff"], h).T)) @ w(p + "down", h, m["ff"]).T
        router = m["router"]
        z = n @ w(p + "router", router["experts"], h).T + w(p + "router.b", router["experts"])
        best, index = z.topk(router["top"], -1)
        return _experts(n, w, p, m, index, best.softmax(-1))

    for i, layer in enumerate(c["layers"]):
        for q, sub, prefix, m in ((1, mixer, f"l{i}.mix.", layer["mixer"]), (2, feed_forward, f"l{i}.mlp.", layer["mlp"])):
            into, mix, back = (w(f"l{i}.hc{q}.{s}", *shape) for s, shape in (("in", (streams,)), ("mix", (streams, streams)),
                                                                           ("out", (streams,))))
            n = _layer_norm(torch.tensordot(into, x, 1), w(f"l{i}.norm{q}", h), w(f"l{i}.norm{q}.b", h), eps)
            x = torch.tensordot(mix.T, x, 1) + back[:, None, None] * sub(n, prefix, m)
    last = w("final.norm", h), w("final.norm.b", h), eps
    return [_layer_norm(r, *last) for r in _rows(seqs, wanted, x.sum(0))], table


def _roserax(c, w, seqs, wanted):
    h, eps = c["width"], c["norm"]["eps"]
    table = w("embed", c["vocab"], h)
    x = table[torch.tensor([t for s in seqs for t in s], device=DEVICE)] * c["embedding"]["scale"]

    def heads(n, p, count, d):
        return (n @ w(p, count * d, h).T).view(-1, count, d)

    def window(n, p, m):
        nq, nk, d, size, keep = m["heads"], m["kv_heads"], m["dim"], m["mask"]["size"], m["mask"]["keep_first"]
        qkv = torch.cat([_rms(heads(n, p + "q", nq, d), w(p + "q.norm", d), eps),
                         _rms(heads(n, p + "k", nk, d), w(p + "k.norm", d), eps), heads(n, p + "v", nk, d)], 1)
        return _each(seqs, qkv, lambda z: _attend(z[:, :nq], z[:, nq: nq + nk], z[:, nq + nk:], m["scale"], sink=True,
                                                  hidden_from=lambda i, j: (i - j >= size) & (j >= keep))) \
            @ w(p + "o", h, nq * d).T

    def latent(n, p, m):
        nq, d, r, rank, dv, base = m["heads"], m["dim"], m["rot_dim"], m["kv_rank"], m["vdim"], m["rot"]["base"]
        q = _rms(n @ w(p + "dq", m["q_rank"], h).T, w(p + "dq.norm", m["q_rank"]), eps)
        q = (q @ w(p + "uq", nq * (d + r), m["q_rank"]).T).view(-1, nq, d + r)
        down = n @ w(p + "dkv", rank + r, h).T
        lat = _rms(down[:, :rank], w(p + "dkv.norm", rank), eps)
        k, v = ((lat @ w(p + s, nq * size, rank).T).view(-1, nq, size) for s, size in (("uk", d), ("uv", dv)))

        def one(z):
            q, k, v, k_rot = z[:, : nq * (d + r)], z[:, nq * (d + r): -nq * dv - r], z[:, -nq * dv - r: -r], z[:, None, -r:]
            q, k, v = q.view(-1, nq, d + r), k.view(-1, nq, d), v.view(-1, nq, dv)
            q = torch.cat([q[..., :d], _turn(q[..., d:], base)], -1)
            k = torch.cat([k, _turn(k_rot, base).expand(-1, nq, -1)], -1)
            return _attend(q, k, v, m["scale"])

        y = _each(seqs, torch.cat([q.flatten(1), k.flatten(1), v.flatten(1), down[:, rank:]], 1), one)
        return (y * torch.sigmoid(n @ w(p + "g", nq * dv, h).T)) @ w(p + "o", h, nq * dv).T

    def retention(n, p, m):
        count, d, base, decay = m["heads"], m["dim"], m["rot"]["base"], m["decay"]
        qkv = torch.cat([heads(n, p + "q", count, d), heads(n, p + "k", count, d) * d ** -0.5, heads(n, p + "v", count, d)], 1)

        def one(z):  # what the recurrence S <- decay S + k v^T sums up to: (q k^T, decayed by the distance) v
            q, k, v = _turn(z[:, :count], base), _turn(z[:, count: 2 * count], base), z[:, 2 * count:]
            i = torch.arange(z.shape[0], dtype=torch.float64, device=z.device)
            gap = i[:, None] - i[None, :]
            return torch.stack([((q[:, j] @ k[:, j].T) * (decay[j] ** gap.clamp(min=0)).masked_fill(gap < 0, 0.0)) @ v[:, j]
                                for j in range(count)], 1)

        y = _rms(_each(seqs, qkv, one), None, eps).flatten(1)
        return (y * _silu(n @ w(p + "g", count * d, h).T)) @ w(p + "o", h, count * d).T

    def feed_forward(n, p, m):
        if m["kind"] == "dense":
            return torch.relu(n @ w(p + "up", m["ff"], h).T).square() @ w(p + "down", h, m["ff"]).T
        router = m["router"]
        s = (n @ w(p + "router", router["experts"], h).T).softmax(-1)
        groups, keep = router["groups"]["count"], router["groups"]["keep"]
        best = s.view(s.shape[0], groups, -1).amax(-1).topk(keep, -1).indices
        stays = torch.zeros(s.shape[0], groups, dtype=torch.bool, device=s.device).scatter_(1, best, True)
        index = s.masked_fill(~stays.repeat_interleave(s.shape[1] // groups, 1), -1.0).topk(router["top"], -1).indices
        return _experts(n, w, p, m, index, s.gather(1, index))

    mixers = {"attention": window, "latent_attention": latent, "retention": retention}
    for i, layer in enumerate(c["layers"]):
        p = f"l{i}."
        y = mixers[layer["type"]](_rms(x, w(p + "norm1", h), eps), p + "mix.", layer["mixer"])
        x = x + _rms(y, w(p + "norm1b", h), eps)
        y = feed_forward(_rms(x, w(p + "norm2", h), eps), p + "mlp.", layer["mlp"])
        x = x + _rms(y, w(p + "norm2b", h), eps)
    norm = w("final.norm", h)
    return [_rms(r, norm, eps) * c["logit_scale"] for r in _rows(seqs, wanted, x)], table
