"""The work that a serving engine has this library do, as cases that can be
timed and compared: attention layers (decode, speculative verify, chunked
prefill and their mixture, each appending its new keys and values first), the
o_proj product that consumes them, the move of sequences out of the pool and
back, and a captured decode step of a whole model's layers.

A case is a dict of plain values.  ``listed()`` names the fixed ones,
``draw(rng)`` gives more of the same ranges, ``prepare(case, seed)`` makes what
a program holds before the call, ``run(state)`` is one pass through the public
entry points, ``exact(case, seed)`` the same results in 64 bits from plain
torch, ``work(case)`` the bytes and operations that a pass cannot do without,
and ``tolerance(case)`` how far another correct implementation may be off.
"""

import math
import random

import numpy as np
import torch

from flint_amd import ops
from flint_amd.pool import ArenaSpec, KvPool, RowMeta
from flint_amd.rope import Rope

# The model shapes of this repository's benchmark and tests:
# query heads, KV heads, head_dim, hidden size (o_proj's output), rope theta.
MODELS = {
    "qwen2-0.5b": (14, 2, 64, 896, 1e6),
    "llama3-8b": (32, 8, 128, 4096, 5e5),
    "qwen3-8b": (32, 8, 128, 4096, 1e6),
    "gemma2-9b": (16, 8, 256, 3584, 1e4),
    "qwen2.5-32b": (40, 8, 128, 5120, 1e6),
}
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f16": 2, "bf16": 2}


def _attn(name, model, **kw):
    """One attention layer: `batch` sequences with contexts spread
    log-uniformly over [ctx_lo, ctx_hi] that each append `rows` tokens, and
    `chunks` prefill chunks of `chunk` tokens after `prefix` cached ones."""
    case = {"name": name, "kind": "attn", "model": model, "kv": "f16", "page": 16, "x": "f16", "y": "f16",
            "batch": 0, "ctx_lo": 0, "ctx_hi": 0, "rows": 1, "chunks": 0, "chunk": 0, "prefix": 0, "window": 0,
            "softcap": 0.0, "rope": False, "norm": False, "gate": False, "fork": False}
    case.update(kw)
    return case


def listed():
    return [
        # A few short conversations on a small model: one layer is a few
        # microseconds, so latency is all there is.  f32 activations.
        _attn("small batch decode", "qwen2-0.5b", batch=4, ctx_lo=128, ctx_hi=512, x="f32", y="f32"),
        # One user's chat in the reference's own storage (bf16 keys in pages of
        # 32, f32 activations): the call of a local engine.
        _attn("one sequence decode", "llama3-8b", batch=1, ctx_lo=2500, ctx_hi=2500, kv="bf16", page=32, x="f32",
              y="f32", rope=True),
        # The benchmark's headline shape: a full decode batch.
        _attn("full batch decode", "llama3-8b", batch=32, ctx_lo=4096, ctx_hi=4096),
        # Speculative decoding: four drafts a sequence, verified at once; a
        # global layer with soft-capped logits.
        _attn("draft verify", "gemma2-9b", batch=16, ctx_lo=8192, ctx_hi=8192, rows=4, softcap=50.0),
        # Documents: four contexts of 131072 tokens, each forked once.
        _attn("long context decode", "qwen2.5-32b", batch=4, ctx_lo=131060, ctx_hi=131060, fork=True),
        # Continuous batching: ragged decode rows beside fresh 512-token
        # chunks, with q/k norm and rotation.
        _attn("continuous batch", "qwen3-8b", batch=64, ctx_lo=256, ctx_hi=16384, chunks=8, chunk=512, rope=True,
              norm=True),
        # A prompt from its first token, alone.
        _attn("prompt prefill", "llama3-8b", chunks=1, chunk=4096, rope=True),
        # A ragged chunk after a cached prefix, sliding window and soft-cap,
        # head_dim 256.
        _attn("chunk after prefix", "gemma2-9b", chunks=1, chunk=777, prefix=3001, window=4096, softcap=50.0,
              y="f32"),
        # The attention's consumer at decode and at prefill.
        {"name": "o_proj decode", "kind": "gemm", "rows": 32, "n": 4096, "k": 4096, "x": "bf16", "w": "bf16",
         "acc": True},
        {"name": "o_proj prefill", "kind": "gemm", "rows": 1500, "n": 5120, "k": 5120, "x": "bf16", "w": "bf16",
         "acc": True},
        # Preemption: sequences copied out of the pool and into new pages.
        {"name": "swap out and in", "kind": "swap", "model": "llama3-8b", "layers": 4, "batch": 6, "ctx_lo": 300,
         "ctx_hi": 4000, "page": 16},
        # A serving loop's decode step: page allocation, plan, and for every
        # layer append + attention + o_proj, captured once and replayed.
        {"name": "captured decode step", "kind": "step", "model": "llama3-8b", "layers": 32, "batch": 8,
         "ctx_lo": 300, "ctx_hi": 3000, "kv": "f16", "page": 16},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "verify", "mixed", "prefill", "prefill", "gemm", "gemm", "swap", "step"])
    if kind == "gemm":
        model = rng.choice(sorted(MODELS))
        nq, _, hd, hidden, _ = MODELS[model]
        return {"kind": "gemm", "rows": _log_int(rng, 1, 6000), "n": hidden, "k": nq * hd,
                "x": rng.choice(["bf16", "bf16", "f16", "f32"]), "w": rng.choice(["bf16", "bf16", "f16"]),
                "acc": rng.random() < 0.7}
    if kind == "swap":
        lo = _log_int(rng, 20, 2000)
        return {"kind": "swap", "model": rng.choice(sorted(MODELS)), "layers": rng.randint(1, 8),
                "batch": rng.randint(1, 12), "ctx_lo": lo, "ctx_hi": 2 * lo + rng.randint(0, 99),
                "page": rng.choice([16, 32])}
    if kind == "step":
        lo = _log_int(rng, 60, 2000)
        return {"kind": "step", "model": rng.choice(["qwen2-0.5b", "llama3-8b"]), "layers": rng.choice([8, 16, 24]),
                "batch": _log_int(rng, 1, 24), "ctx_lo": lo, "ctx_hi": lo + _log_int(rng, 1, 1000),
                "kv": rng.choice(["f16", "bf16"]), "page": rng.choice([16, 32])}
    model = rng.choice(sorted(MODELS))
    case = _attn("", model, kv=rng.choice(["f16", "f16", "bf16"]), page=rng.choice([16, 16, 32]),
                 x=rng.choice(["f32", "f16"]), y=rng.choice(["f32", "f16"]))
    del case["name"]
    if model == "gemma2-9b":
        case.update(softcap=50.0, window=rng.choice([0, 4096]))
    elif model == "qwen3-8b":
        case.update(rope=True, norm=True, gate=rng.random() < 0.2)
    else:
        case.update(rope=rng.random() < 0.5)
    if kind in ("decode", "verify", "mixed"):
        case["batch"] = _log_int(rng, 1, 64)
        longest = min(65536, 120000 // case["batch"])
        lo = _log_int(rng, 32, longest)
        case.update(ctx_lo=lo, ctx_hi=rng.randint(lo, min(longest, 8 * lo)))
        if kind == "verify":
            case["rows"] = rng.randint(2, 4)
    if kind == "mixed":
        case.update(chunks=rng.randint(1, 4), chunk=_log_int(rng, 60, 600))
    if kind == "prefill":
        case.update(chunks=rng.choice([1, 1, 2, 4]), chunk=_log_int(rng, 40, 1500),
                    prefix=rng.choice([0, 0, _log_int(rng, 16, 6000)]))
    return case


# ------------------------------------------------------------------- inputs


def _rng_of(case):
    """Sizes within a case's ranges follow from the case alone."""
    return random.Random("/".join(f"{k}={case[k]}" for k in sorted(case) if k != "name"))


def _gen(seed, *more):
    g = torch.Generator(device="cuda")
    g.manual_seed(hash((int(seed),) + tuple(int(x) for x in more)) & 0x7FFFFFFFFFFF)
    return g


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, device="cuda", generator=g) * scale


def _spread(rng, n, lo, hi):
    return [min(hi, max(lo, _log_int(rng, lo, hi))) for _ in range(n)]


def _sequences(case):
    """(cached tokens, new tokens) of each sequence, decode rows first."""
    seqs = [(n, case["rows"]) for n in _spread(_rng_of(case), case["batch"], case["ctx_lo"], case["ctx_hi"])]
    if case["fork"]:
        seqs += seqs
    return seqs + [(case["prefix"], case["chunk"])] * case["chunks"]


def _cached(case, seed, s, n):
    """Keys and values of sequence s's cached tokens, [kv_heads, n, head_dim]
    in the pool's type.  A fork's are its source's."""
    _, nkv, hd, _, _ = MODELS[case["model"]]
    if case["fork"]:
        s %= case["batch"]
    g = _gen(seed, 1, s)
    return tuple(_randn(g, nkv, n, hd).to(DTYPES[case["kv"]]) for _ in range(2))


def _new(case, seed, m):
    """Queries (spread so that some keys stand out), new keys and values and
    the output gate of a call's m rows."""
    nq, nkv, hd, _, _ = MODELS[case["model"]]
    g, dt = _gen(seed, 2), DTYPES[case["x"]]
    q = _randn(g, m, nq, hd, scale=1.5).to(dt)
    k, v = (_randn(g, m, nkv, hd).to(dt) for _ in range(2))
    gate = _randn(g, m, nq, hd).to(dt) if case["gate"] else None
    return q, k, v, gate


def _tables(model, max_pos):
    _, _, hd, _, theta = MODELS[model]
    angle = np.arange(max_pos)[:, None] / np.power(theta, 2.0 * np.arange(hd // 2) / hd)
    return np.cos(angle).astype(np.float32), np.sin(angle).astype(np.float32)


def _norms(case, seed):
    if not case["norm"]:
        return None, None
    hd = MODELS[case["model"]][2]
    g = _gen(seed, 3)
    return tuple(1.0 + 0.1 * torch.randn(hd, device="cuda", generator=g) for _ in range(2))


EPS = 1e-6


def _pool(model, kv, page, lens, layers, budgets=None):
    """A pool over a zero-filled caller-owned arena."""
    _, nkv, hd, _, _ = MODELS[model]
    budgets = budgets or lens
    pages = sum(-(-n // page) for n in lens)
    arena = torch.zeros(layers * 2 * (pages * page * nkv * hd + 128) + 2048, dtype=DTYPES[kv], device="cuda")
    pool = KvPool(ArenaSpec(list(budgets), pages), nkv, hd, layers=layers, page_len=page, kv_dtype=kv, arena=arena)
    return pool, arena


def _scatter_pages(pool, lens, page, rng):
    """Allocates the sequences' tokens piece by piece in random order, as a
    busy engine's pool would hold them."""
    piece = max(page, -(-max(sum(lens), 1) // 4096 // page) * page)
    order = [s for s, n in enumerate(lens) for _ in range(-(-n // piece))]
    rng.shuffle(order)
    have = [0] * len(lens)
    for s in order:
        n = min(piece, lens[s] - have[s])
        pool.alloc(s, have[s], n)
        have[s] += n


def prepare(case, seed):
    return {"attn": _prepare_attn, "gemm": _prepare_gemm, "swap": _prepare_swap, "step": _prepare_step}[case["kind"]](
        case, seed)


def _prepare_attn(case, seed):
    model = case["model"]
    nq, _, hd, _, _ = MODELS[model]
    seqs = _sequences(case)
    page, src = case["page"], case["batch"] if case["fork"] else len(seqs)
    total = [c + n for c, n in seqs]
    # a fork owns the pages of its last, partial page and what it appends
    own = total[:src] + [2 * page] * (len(seqs) - src)
    pool, arena = _pool(model, case["kv"], page, own, 1, budgets=total)
    if case["fork"]:
        _scatter_pages(pool, [c for c, _ in seqs[:src]], page, _rng_of(case))
    else:
        _scatter_pages(pool, total, page, _rng_of(case))
    for s in range(src):
        n = seqs[s][0]
        if n:
            k, v = _cached(case, seed, s, n)
            ops.kv_scatter(pool, 0, s, 0, n, k, v)
    for s in range(src, len(seqs)):
        pool.fork(s - src, s, seqs[s][0])
    if case["fork"]:
        for s, (c, n) in enumerate(seqs):
            pool.alloc(s, c, n)
    pool.sync()
    positions = [c + i for c, n in seqs for i in range(n)]
    owners = [s for s, (_, n) in enumerate(seqs) for _ in range(n)]
    m = len(owners)
    rows = RowMeta(m)
    rows.write(positions, owners, m)
    q, k, v, gate = _new(case, seed, m)
    y = torch.zeros(m, nq, hd, dtype=DTYPES[case["y"]], device="cuda")
    rope = None
    if case["rope"]:
        cos, sin = _tables(model, max(total))
        qn, kn = _norms(case, seed)
        rope = Rope(cos, sin, hd, q_norm=qn, k_norm=kn, eps=EPS)
    spec = ops.AttnSpec(q_heads=nq, window=case["window"], scale=ops.default_scale(hd), m=m, causal=True, seq=None,
                        args=rows, softcap=case["softcap"])
    return {"kind": "attn", "pool": pool, "arena": arena, "rows": rows, "spec": spec, "q": q, "k": k, "v": v,
            "gate": gate, "y": y, "rope": rope}


def _prepare_gemm(case, seed):
    g = _gen(seed, 4)
    x = _randn(g, case["rows"], case["k"]).to(DTYPES[case["x"]])
    w = _randn(g, case["n"], case["k"], scale=0.02).to(DTYPES[case["w"]])
    y = _randn(g, case["rows"], case["n"])
    return {"kind": "gemm", "x": x, "w": w, "y": y, "rows": case["rows"], "acc": case["acc"]}


def _swap_lens(case):
    return _spread(_rng_of(case), case["batch"], case["ctx_lo"], case["ctx_hi"])


def _prepare_swap(case, seed):
    _, nkv, hd, _, _ = MODELS[case["model"]]
    lens = _swap_lens(case)
    pool, arena = _pool(case["model"], "f16", case["page"], lens + lens, case["layers"])
    _scatter_pages(pool, lens + lens, case["page"], _rng_of(case))
    g = _gen(seed, 5)
    for layer in range(case["layers"]):
        for s, n in enumerate(lens):
            k, v = (_randn(g, nkv, n, hd).half() for _ in range(2))
            ops.kv_scatter(pool, layer, s, 0, n, k, v)
    out = [(s, layer, 0, n) for layer in range(case["layers"]) for s, n in enumerate(lens)]
    back = [(len(lens) + s, layer, 0, n) for s, layer, _, n in out]
    total = sum(n for _, _, _, n in out) * nkv * hd
    k, v = (torch.zeros(total, dtype=torch.float16, device="cuda") for _ in range(2))
    return {"kind": "swap", "pool": pool, "arena": arena, "out": out, "back": back, "k": k, "v": v}


def _step_lens(case):
    return _spread(_rng_of(case), case["batch"], case["ctx_lo"], case["ctx_hi"])


def _step_inputs(case, seed, layer):
    """q, k, v of the step's rows and o_proj's weights of one layer."""
    nq, nkv, hd, hidden, _ = MODELS[case["model"]]
    g, b = _gen(seed, 6, layer), case["batch"]
    q = _randn(g, b, nq, hd, scale=1.5).half()
    k, v = (_randn(g, b, nkv, hd).half() for _ in range(2))
    w = _randn(g, hidden, nq * hd, scale=0.02).to(torch.bfloat16)
    return q, k, v, w


def _step_cached(case, seed, layer, s, n):
    _, nkv, hd, _, _ = MODELS[case["model"]]
    g = _gen(seed, 7, layer, s)
    return tuple(_randn(g, nkv, n, hd).to(DTYPES[case["kv"]]) for _ in range(2))


def _prepare_step(case, seed):
    model, b, layers = case["model"], case["batch"], case["layers"]
    nq, _, hd, hidden, _ = MODELS[model]
    lens = _step_lens(case)
    total = [n + 1 for n in lens]
    pool, arena = _pool(model, case["kv"], case["page"], total, layers)
    _scatter_pages(pool, lens, case["page"], _rng_of(case))
    for layer in range(layers):
        for s, n in enumerate(lens):
            k, v = _step_cached(case, seed, layer, s, n)
            ops.kv_scatter(pool, layer, s, 0, n, k, v)
    inputs = [_step_inputs(case, seed, layer) for layer in range(layers)]
    x0 = _randn(_gen(seed, 8), b, hidden)
    h, y = torch.zeros_like(x0), torch.zeros(layers, b, nq * hd, dtype=torch.bfloat16, device="cuda")
    cos, sin = _tables(model, max(total))
    rope = Rope(cos, sin, hd)
    rows = RowMeta(b)
    rows.write(lens, list(range(b)), b)
    spec = ops.AttnSpec(q_heads=nq, window=0, scale=ops.default_scale(hd), m=b, causal=True, seq=None, args=rows)
    plan = ops.DevicePlan(pool, max_m=b, q_heads=nq, append=True)
    plan.set_pos_limit(rope.max_pos)

    def body():
        h.copy_(x0)
        pool.alloc_rows(rows, b)
        plan.build(spec, inputs[0][0], y[0])
        for layer, (q, k, v, w) in enumerate(inputs):
            plan.step(layer, q, y[layer], k_src=k, v_src=v, rope=rope)
            ops.gemm_acc(y[layer], w, h, b, True)

    body()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            body()
    torch.cuda.current_stream().wait_stream(side)
    return {"kind": "step", "pool": pool, "arena": arena, "rows": rows, "positions": lens, "seqs": list(range(b)),
            "graph": graph, "h": h, "y": y, "keep": (plan, inputs, rope, x0)}


# ---------------------------------------------------------------- one pass


def run(state):
    kind = state["kind"]
    if kind == "attn":
        ops.attn_step(state["pool"], 0, state["spec"], state["q"], state["y"], gate=state["gate"], k_src=state["k"],
                      v_src=state["v"], rope=state["rope"])
        return {"y": state["y"], "pool": state["arena"]}
    if kind == "gemm":
        ops.gemm_acc(state["x"], state["w"], state["y"], state["rows"], state["acc"])
        return state["y"]
    if kind == "swap":
        ops.kv_gather_batch(state["pool"], state["out"], state["k"], state["v"])
        ops.kv_scatter_batch(state["pool"], state["back"], state["k"], state["v"])
        return {"k": state["k"], "v": state["v"], "pool": state["arena"]}
    state["rows"].write(state["positions"], state["seqs"])
    state["graph"].replay()
    return {"h": state["h"], "y": state["y"], "pool": state["arena"]}


# --------------------------------------------------------- in 64 bits


def _rotate64(x, cos, sin, weight):
    """x [m, heads, hd] normalised (with a weight) and rotated, in f64."""
    x = x.double()
    if weight is not None:
        x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()
    half = x.shape[-1] // 2
    a, b = x[..., :half], x[..., half:]
    c, s = cos[:, None, :], sin[:, None, :]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _encode(x, kv):
    """Values as the pool stores them: f16 by rounding, bf16 by truncation."""
    if kv == "f16":
        return x.half().double()
    return (x.float().view(torch.int32) & -65536).view(torch.float32).double()


def _attend64(q, k, v, first, window, softcap):
    """Causal attention in f64: q [m, nq, hd] at positions first.., k and v
    [nkv, n, hd]."""
    m, nq, hd = q.shape
    nkv, n, _ = k.shape
    g = nq // nkv
    kt = k.transpose(1, 2).contiguous()
    out = torch.empty(m, nq, hd, dtype=torch.float64, device=q.device)
    t = torch.arange(n, device=q.device)
    for r in range(0, m, 256):
        qr = q[r:r + 256]
        b = qr.shape[0]
        s = torch.matmul(qr.view(b, nkv, g, hd).permute(1, 2, 0, 3).reshape(nkv, g * b, hd).contiguous(), kt)
        s = s / math.sqrt(hd)
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        pos = first + r + torch.arange(b, device=q.device)
        seen = t[None, :] <= pos[:, None]
        if window:
            seen &= t[None, :] + window > pos[:, None]
        s = s.view(nkv, g, b, n).masked_fill(~seen, -math.inf)
        p = torch.softmax(s, -1).view(nkv, g * b, n)
        out[r:r + b] = torch.matmul(p, v).view(nkv, g, b, hd).permute(2, 0, 1, 3).reshape(b, nq, hd)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "swap":
        return None
    if kind == "gemm":
        s = _prepare_gemm(case, seed)
        y = torch.matmul(s["x"].double(), s["w"].double().t().contiguous())
        return y + s["y"].double() if case["acc"] else y
    if kind == "step":
        return _exact_step(case, seed)
    _, _, hd, _, _ = MODELS[case["model"]]
    seqs = _sequences(case)
    m = sum(n for _, n in seqs)
    q, k, v, gate = _new(case, seed, m)
    pos = torch.tensor([c + i for c, n in seqs for i in range(n)], device="cuda")
    q64, k64 = q.double(), k.double()
    if case["rope"]:
        cos, sin = (torch.from_numpy(t).cuda().double()[pos] for t in _tables(case["model"], max(map(sum, seqs))))
        qn, kn = _norms(case, seed)
        q64, k64 = _rotate64(q, cos, sin, qn), _rotate64(k, cos, sin, kn).to(k.dtype)
    k64, v64 = _encode(k64, case["kv"]), _encode(v, case["kv"])
    out, r = [], 0
    for s, (c, n) in enumerate(seqs):
        kc, vc = (torch.cat([a.double(), b[r:r + n].transpose(0, 1)], 1) for a, b in
                  zip(_cached(case, seed, s, c), (k64, v64)))
        out.append(_attend64(q64[r:r + n], kc, vc, c, case["window"], case["softcap"]))
        r += n
    y = torch.cat(out)
    if gate is not None:
        y = y * torch.sigmoid(gate.double())
    return {"y": y, "pool": None}


def _exact_step(case, seed):
    nq, _, hd, hidden, _ = MODELS[case["model"]]
    lens, b = _step_lens(case), case["batch"]
    h = _randn(_gen(seed, 8), b, hidden).double()
    cos, sin = (torch.from_numpy(t).cuda().double()[lens] for t in _tables(case["model"], max(lens) + 1))
    ys = []
    for layer in range(case["layers"]):
        q, k, v, w = _step_inputs(case, seed, layer)
        q64 = _rotate64(q, cos, sin, None)
        k64, v64 = _encode(_rotate64(k, cos, sin, None).half(), case["kv"]), _encode(v, case["kv"])
        y = []
        for s, n in enumerate(lens):
            kc, vc = (torch.cat([a.double(), x[s:s + 1].transpose(0, 1)], 1) for a, x in
                      zip(_step_cached(case, seed, layer, s, n), (k64, v64)))
            y.append(_attend64(q64[s:s + 1], kc, vc, n, 0, 0.0))
        y = torch.cat(y).view(b, nq * hd)
        ys.append(y)
        h = h + torch.matmul(y, w.double().t().contiguous())
    return {"h": h, "y": torch.stack(ys), "pool": None}


# ------------------------------------------------------- work and tolerance


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        r, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": n * k * 2 + r * k * BYTES[case["x"]] + r * n * 4 * (2 if case["acc"] else 1),
                "flops": 2 * r * n * k}
    nq, nkv, hd, hidden, _ = MODELS[case["model"]]
    if kind == "swap":
        # each word out of the pool, into a buffer, out of it and into the pool
        return {"bytes": sum(_swap_lens(case)) * case["layers"] * nkv * hd * 2 * 2 * 4, "flops": 0}
    if kind == "step":
        lens, b = _step_lens(case), case["batch"]
        kv = sum(n + 1 for n in lens) * nkv * hd * 2 * 2
        io = b * (nq * hd * (2 + 2) + nkv * hd * 2 * (2 + 2)) + b * nq * hd * 2
        return {"bytes": case["layers"] * (kv + io + hidden * nq * hd * 2) + 2 * b * hidden * 4,
                "flops": case["layers"] * (4 * sum(n + 1 for n in lens) * nq * hd + 2 * b * hidden * nq * hd)}
    keys = pairs = 0
    seqs = _sequences(case)
    window = case["window"]
    for s, (c, n) in enumerate(seqs):
        first = max(0, c + 1 - window) if window else 0
        if not case["fork"] or s < case["batch"]:
            keys += c + n - first  # a fork reads its source's pages
        pairs += sum(min(c + i + 1, window or c + i + 1) for i in range(n))
    m = sum(n for _, n in seqs)
    x, y = BYTES[case["x"]], BYTES[case["y"]]
    io = m * (nq * hd * (x * (2 if case["gate"] else 1) + y) + nkv * hd * 2 * (x + 2))
    return {"bytes": keys * nkv * hd * 2 * 2 + io, "flops": 4 * pairs * nq * hd}


def tolerance(case):
    """About four times the error against 64 bits that the present kernels
    show over the declared ranges: the rounding of the output's type, or of
    the sums (an operand wider than the matrix cores' 16 bits is multiplied
    in two parts, ~16 bits together in bf16, ~22 in f16)."""
    kind = case["kind"]
    if kind == "swap":
        return "exact"
    if kind == "gemm":
        return {"rel": 2e-6} if case["x"] == case["w"] else {"rel": 1e-5}
    if kind == "step":  # bf16 layer outputs, summed over the layers
        return {"rel": 7e-3, "max": 0.05}
    if case["y"] == "f16":
        return {"rel": 8e-4, "max": 4e-3}
    return {"rel": 2e-5 if case["kv"] == "bf16" else 1e-5}
