"""What a user of this engine has it do, as cases that can be timed and compared.

A case is one step (or one short exchange) through ``Engine.step``, the function that every way of generating in this
package goes through, on a model with random weights of a named size:

* ``decode``: every live request brings one token, at contexts spread over a range;
* ``read``: prompts are read whole, only their last token's logits wanted, and the requests end;
* ``mixed``: requests that decode beside a portion of a prompt, as the scheduler cuts them;
* ``serve``: requests come, are read and decode some tokens together, and go (the way of a model whose mixers keep
  state, which cannot go back a token).

``listed`` names the cases that are always measured, ``draw`` gives others of the same ranges.  Lengths are spread evenly
over a case's range by its numbers alone, so that the work of a case does not change with the seed; token ids and weights
come from the seed.  ``exact`` computes a case's logits in 64 bits with plain tensor operations.
"""

import math

import torch

from mlx_lm_amd.engine import Engine, StepEntry
from mlx_lm_amd.utils import model_from_tensors

F64 = torch.float64

# GPT-2's published sizes (the last one: layers of the largest size, few of them, with positions for long documents)
GPT2 = {
    "small": dict(n_layer=12, n_embd=768, n_head=12, n_positions=1024),
    "large": dict(n_layer=36, n_embd=1280, n_head=20, n_positions=1024),
    "xl": dict(n_layer=48, n_embd=1600, n_head=25, n_positions=1024),
    "xl12-8k": dict(n_layer=12, n_embd=1600, n_head=25, n_positions=8192),
}
# a design of three mixers by turns: differential attention, gated linear attention, latent attention
ZATINEX = {
    "zatinex-1024": dict(width=1024, heads=16, dim=64, ff=2688, layers=12),
    "zatinex-2048": dict(width=2048, heads=16, dim=128, ff=5440, layers=8),
}
VOCAB = {"gpt2": 50257, "zatinex": 32000}


def _family(case):
    return "gpt2" if case["model"] in GPT2 else "zatinex"


def _positions(case):
    return GPT2[case["model"]]["n_positions"] if _family(case) == "gpt2" else 2048


def _config(case):
    if _family(case) == "gpt2":
        s = GPT2[case["model"]]
        return dict(s, model_type="gpt2", n_inner=4 * s["n_embd"], vocab_size=VOCAB["gpt2"], n_ctx=s["n_positions"],
                    layer_norm_epsilon=1e-5, activation_function="gelu_new")
    s = ZATINEX[case["model"]]
    H, d, D = s["heads"], s["dim"], s["width"]
    turn = {"factor": 8.0, "original": 1024, "fast": 16.0, "slow": 2.0}
    layers = []
    for i in range(s["layers"]):
        if i % 3 == 0:
            entry = {"type": "attention", "mixer": {"heads": H // 2, "kv_heads": H // 2, "dim": d, "vdim": 2 * d, "conv": 4, "diff": 0.3,
                                                    "scale": d ** -0.5, "rot": {"dims": d, "base": 10000.0, "scaling": turn}}}
        elif i % 3 == 1:
            entry = {"type": "gla", "mixer": {"heads": H, "dim": d, "vdim": d, "tau": 8.0, "decay_rank": 16}}
        else:
            m = {"heads": H, "dim": d, "rot_dim": d // 2, "vdim": d, "q_rank": D // 2, "kv_rank": 192,
                 "scale": (d + d // 2) ** -0.5, "rot": {"dims": d // 2, "base": 10000.0}}
            if (i // 3) % 2 == 1:
                m["kv_from"] = 2
            entry = {"type": "latent_attention", "mixer": m}
        layers.append(dict(entry, mlp={"kind": "dense", "ff": s["ff"]}))
    return {"architecture": "Zatinex", "vocab": VOCAB["zatinex"], "width": D, "max_positions": 2048, "norm": {"eps": 1e-5}, "layers": layers}


# ---------------------------------------------------------------------------
# the cases


def listed():
    return [
        # one person's chat with a small model: a token a step, the smallest call there is
        dict(name="small-b1", model="small", dtype="bfloat16", kind="decode", batch=1, lo=93, hi=93),
        # one person's chat with a large model, and a few and many of them served together, at contexts of all lengths
        dict(name="xl-b1", model="xl", dtype="bfloat16", kind="decode", batch=1, lo=700, hi=700),
        dict(name="xl-b8", model="xl", dtype="bfloat16", kind="decode", batch=8, lo=512, hi=1001),
        dict(name="xl-b64", model="xl", dtype="bfloat16", kind="decode", batch=64, lo=300, hi=1001),
        # two full prompts in one step (the benchmark's prefill), and one short question of no round length
        dict(name="xl-prompts-2x1024", model="xl", dtype="bfloat16", kind="read", batch=2, lo=1024, hi=1024),
        dict(name="xl-prompt-333", model="xl", dtype="bfloat16", kind="read", batch=1, lo=333, hi=333),
        # continuous batching: requests that decode beside a new prompt's portion
        dict(name="xl-mixed-24+512", model="xl", dtype="bfloat16", kind="mixed", batch=24, lo=200, hi=900, portion=512),
        # long documents: one read whole, and answers about eight of them
        dict(name="long-prompt-8000", model="xl12-8k", dtype="bfloat16", kind="read", batch=1, lo=8000, hi=8000),
        dict(name="long-b8", model="xl12-8k", dtype="bfloat16", kind="decode", batch=8, lo=4000, hi=8001),
        # the 32-bit path, for comparisons and scoring: prompts of several lengths, then a token each
        dict(name="large-f32-prompts", model="large", dtype="float32", kind="read", batch=3, lo=200, hi=500),
        dict(name="large-f32-b8", model="large", dtype="float32", kind="decode", batch=8, lo=300, hi=900),
        # a design with other mixers: requests come, are read together, answer some tokens and go
        dict(name="zatinex-serve", model="zatinex-1024", dtype="bfloat16", kind="serve", batch=8, lo=40, hi=300, new=8),
    ]


def _cost(case):
    """Seconds, roughly, on a card that reads 4 TB/s and computes 500 (32 bits: 80) TFLOP/s: to bound what is drawn."""
    w = work(case)
    steps = 1 + case.get("new", 0)
    return w["bytes"] / 4e12 + w["flops"] / (5e14 if case["dtype"] == "bfloat16" else 8e13) + steps * 3e-4


def draw(rng):
    def spread(lo, hi):  # evenly over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    most = max(_cost(c) for c in listed())
    while True:
        dtype = "float32" if rng.random() < 0.2 else "bfloat16"
        model = rng.choice(["small", "large", "xl", "xl12-8k", "zatinex-1024", "zatinex-2048"])
        case = dict(model=model, dtype=dtype)
        P = _positions(case)
        if model in ZATINEX:
            case.update(kind="serve", batch=spread(1, 32), new=rng.randint(1, 12))
            a, b = spread(5, 900), spread(5, 900)
        else:
            case["kind"] = rng.choice(["decode", "decode", "read", "mixed"])
            case["batch"] = spread(1, 64) if case["kind"] == "decode" else spread(1, 8) if case["kind"] == "read" else spread(2, 48)
            a, b = spread(16, P - 2), spread(16, P - 2)
            if case["kind"] == "mixed":
                case["portion"] = spread(16, 1000)
        case.update(lo=min(a, b), hi=max(a, b))
        tokens = sum(_lengths(case))
        if _cost(case) <= most and tokens <= 65536 and (case["kind"] not in ("read", "serve") or tokens <= 8192):
            return case


def _lengths(case):
    """The requests' lengths: spread evenly from ``lo`` to ``hi``, in an order of no pattern."""
    n, lo, hi = case["batch"], case["lo"], case["hi"]
    if n == 1:
        return [(lo + hi) // 2]
    even = [lo + (hi - lo) * i // (n - 1) for i in range(n)]
    step = next(k for k in (7, 5, 3, 11, 13, 17, 1) if math.gcd(k, n) == 1)
    return [even[(i * step) % n] for i in range(n)]


# ---------------------------------------------------------------------------
# weights and tokens, from the seed


def _weights(case, seed):
    """Tensors under a checkpoint's names, on the GPU: matrices in the case's type, vectors in 32 bits."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    wide = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    t = {}

    def put(name, shape, std, mean=0.0):
        x = torch.randn(shape, generator=g, device="cuda").mul_(std).add_(mean)
        t[name] = x.to(wide) if len(shape) > 1 else x

    c = _config(case)
    if _family(case) == "gpt2":
        D, L = c["n_embd"], c["n_layer"]
        put("wte.weight", (c["vocab_size"], D), 0.02)
        put("wpe.weight", (c["n_positions"], D), 0.02)
        for i in range(L):
            p = f"h.{i}."
            for n in ("ln_1", "ln_2"):
                put(p + n + ".weight", (D,), 0.1, 1.0)
                put(p + n + ".bias", (D,), 0.02)
            for n, a, b, std in (("attn.c_attn", D, 3 * D, 0.02), ("attn.c_proj", D, D, 0.02 / math.sqrt(2 * L)),
                                 ("mlp.c_fc", D, 4 * D, 0.02), ("mlp.c_proj", 4 * D, D, 0.02 / math.sqrt(2 * L))):
                put(p + n + ".weight", (a, b), std)
                put(p + n + ".bias", (b,), 0.02)
        put("ln_f.weight", (D,), 0.1, 1.0)
        put("ln_f.bias", (D,), 0.02)
        return t
    D = c["width"]

    def square(name, n, k):
        put(name, (n, k), k ** -0.5)

    put("embed", (c["vocab"], D), 1.0)
    for i, layer in enumerate(c["layers"]):
        p, m, q = f"l{i}.", layer["mixer"], f"l{i}.mix."
        put(p + "norm1", (D,), 0.1, 1.0)
        H, d = m["heads"], m["dim"]
        if layer["type"] == "attention":
            for name, n in (("q", 2 * H * d), ("k", 2 * H * d), ("v", H * m["vdim"])):
                square(q + name, n, D)
                put(q + name + ".b", (n,), 0.1)
                put(q + name + ".conv", (n, m["conv"]), 0.5)
            for name in ("q.norm", "k.norm"):
                put(q + name, (d,), 0.1, 1.0)
            for name in ("lq1", "lk1", "lq2", "lk2"):
                put(q + name, (d,), 0.1)
            square(q + "o", D, H * m["vdim"])
        elif layer["type"] == "gla":
            for name in ("q", "k", "v", "g"):
                square(q + name, H * d, D)
            square(q + "o", D, H * d)
            put(q + "norm", (d,), 0.1, 1.0)
            square(q + "a1", m["decay_rank"], D)
            square(q + "a2", H * d, m["decay_rank"])
            put(q + "a2.b", (H * d,), 1.0, 2.0)
        else:
            dr, dv, Q, R = m["rot_dim"], m["vdim"], m["q_rank"], m["kv_rank"]
            square(q + "dq", Q, D)
            put(q + "dq.norm", (Q,), 0.1, 1.0)
            square(q + "uq", H * (d + dr), Q)
            if "kv_from" not in m:
                square(q + "dkv", R + dr, D)
                put(q + "dkv.norm", (R,), 0.1, 1.0)
            square(q + "uk", H * d, R)
            square(q + "uv", H * dv, R)
            square(q + "g", H, D)
            square(q + "o", D, H * dv)
        put(p + "norm2", (D,), 0.1, 1.0)
        F = layer["mlp"]["ff"]
        square(p + "mlp.gate", F, D)
        square(p + "mlp.up", F, D)
        square(p + "mlp.down", D, F)
    put("final.norm", (D,), 0.1, 1.0)
    square("head", c["vocab"], D)
    return t


def _tokens(case, seed):
    """The requests' token ids, the portion's last in a ``mixed`` case; what a request brings in the pass is at its end."""
    extra = {"decode": 1, "mixed": 1, "read": 0, "serve": case.get("new", 0)}[case["kind"]]
    lengths = [n + extra for n in _lengths(case)] + ([case["portion"]] if case["kind"] == "mixed" else [])
    g = torch.Generator().manual_seed(int(seed) + 1)
    return [torch.randint(0, VOCAB[_family(case)], (n,), generator=g).tolist() for n in lengths]


# ---------------------------------------------------------------------------
# what a program holds before a pass, and the pass


def prepare(case, seed):
    """The loaded model, its engine, and, where the pass decodes, requests whose contexts have been read."""
    model = model_from_tensors(_config(case), _weights(case, seed), dtype=case["dtype"], device="cuda:0")
    tokens = _tokens(case, seed)
    total = sum(len(t) + 32 for t in tokens)
    engine = Engine(model, dtype=case["dtype"], page_size=16, max_tokens=total, max_requests=64, record_prompt_steps=True)
    state = dict(kind=case["kind"], engine=engine, model=model)
    kind, B = case["kind"], case["batch"]
    if kind in ("decode", "mixed"):
        step, held = [], 0
        for i in range(B):
            engine.add_request(i)
            known = tokens[i][:-1]
            if step and held + len(known) > 8192:
                engine.step(step)
                step, held = [], 0
            step.append(StepEntry(i, known))
            held += len(known)
        engine.step(step)
        state["decoding"] = [StepEntry(i, tokens[i][-1:], [0]) for i in range(B)]
        state["portion"] = StepEntry("portion", tokens[B], [len(tokens[B]) - 1]) if kind == "mixed" else None
    elif kind == "read":
        state["prompts"] = [StepEntry(i, t, [len(t) - 1]) for i, t in enumerate(tokens)]
    else:
        n = case["new"]
        state["prompts"] = [StepEntry(i, t[: len(t) - n], [len(t) - n - 1]) for i, t in enumerate(tokens)]
        state["answers"] = [[StepEntry(i, [t[len(t) - n + k]], [0]) for i, t in enumerate(tokens)] for k in range(n)]
    return state


def run(state):
    """One pass: float32 logits at the wanted places (``serve``: of every step)."""
    engine, kind = state["engine"], state["kind"]
    if kind in ("decode", "mixed"):
        entries = state["decoding"]
        if kind == "mixed":
            engine.add_request("portion")
            entries = entries + [state["portion"]]
        logits = engine.step(entries)
        for e in state["decoding"]:  # a request can be asked for another token at the same place
            engine.trim(e.request_id, 1)
        if kind == "mixed":
            engine.end_request("portion")
        return logits
    for e in state["prompts"]:
        engine.add_request(e.request_id)
    logits = engine.step(state["prompts"])
    if kind == "serve":
        logits = [logits.clone()]  # (a step's logits lie in a buffer that the next one writes)
        for step in state["answers"]:
            logits.append(engine.step(step).clone())
    for e in state["prompts"]:
        engine.end_request(e.request_id)
    return logits


# ---------------------------------------------------------------------------
# what a pass cannot do without


def work(case):
    """Weights read once a step, the token rows that are asked for, keys and values (or states) read and written once,
    logits written; products and causal attention counted in full, two operations a multiply and add."""
    c, e = _config(case), 2 if case["dtype"] == "bfloat16" else 4
    lengths = _lengths(case)
    kind, B = case["kind"], case["batch"]
    # steps as lists of (tokens brought, tokens known before) a request
    if kind == "decode":
        steps = [[(1, n) for n in lengths]]
    elif kind == "mixed":
        steps = [[(1, n) for n in lengths] + [(case["portion"], 0)]]
    elif kind == "read":
        steps = [[(n, 0) for n in lengths]]
    else:
        steps = [[(n, 0) for n in lengths]] + [[(1, n + k) for n in lengths] for k in range(case["new"])]
    total_bytes = total_flops = 0.0
    for step in steps:
        tokens = sum(n for n, _ in step)
        pairs = sum(n * k + n * (n + 1) // 2 for n, k in step)  # (query, key) pairs under the causal mask
        held = sum(n + k for n, k in step)  # keys read, the new ones among them
        rows = len(step)
        if _family(case) == "gpt2":
            D, L, V = c["n_embd"], c["n_layer"], c["vocab_size"]
            matrices = L * 12 * D * D
            total_bytes += (matrices + V * D) * e + L * 13 * D * 4 + 2 * tokens * D * e + rows * V * 4 + tokens * 4
            total_bytes += L * 2 * D * held * e
            total_flops += 2.0 * matrices * tokens + L * 4.0 * D * pairs + 2.0 * V * D * rows
            continue
        D, V = c["width"], c["vocab"]
        total_bytes += V * D * e + tokens * D * e + rows * V * 4 + tokens * 4
        total_flops += 2.0 * V * D * rows
        for layer in c["layers"]:
            m = layer["mixer"]
            H, d, dv = m["heads"], m["dim"], m["vdim"]
            matrices = 3 * D * layer["mlp"]["ff"]
            if layer["type"] == "attention":
                matrices += D * (4 * H * d + 2 * H * dv)
                total_bytes += H * (2 * d + dv) * held * e
                total_flops += 2.0 * H * (2 * d + 2 * dv) * pairs
            elif layer["type"] == "gla":
                r = m["decay_rank"]
                matrices += D * 5 * H * d + r * (D + H * d)
                total_bytes += 2.0 * B * H * d * dv * 4 * (1 if step[0][1] else 0.5)
                total_flops += 4.0 * H * d * dv * tokens
            else:
                dr, Q, R = m["rot_dim"], m["q_rank"], m["kv_rank"]
                own = "kv_from" not in m
                matrices += Q * D + H * (d + dr) * Q + (R + dr) * D * own + H * (d + dv) * R + H * D + D * H * dv
                total_bytes += (R + dr) * held * e
                total_flops += 2.0 * H * (d + dr + dv) * pairs
            total_bytes += matrices * e
            total_flops += 2.0 * matrices * tokens
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    """About four times the distance from ``exact`` that was measured: GPT-2 0.0039 in bfloat16 and 1.9e-6 in 32 bits,
    the other design 0.015 in bfloat16 (its attention takes one map off another) and taken as 1e-5 in 32 bits."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4} if _family(case) == "gpt2" else {"rel": 4e-5, "max": 4e-4}
    return {"rel": 0.015, "max": 0.1} if _family(case) == "gpt2" else {"rel": 0.03, "max": 0.3}


# ---------------------------------------------------------------------------
# the same logits in 64 bits


def exact(case, seed):
    flops = work(case)["flops"]
    tokens = _tokens(case, seed)
    if _family(case) == "gpt2":
        # (a decoded token's logits need its whole context run)
        c = _config(case)
        flops = 2.0 * 12 * c["n_layer"] * c["n_embd"] ** 2 * sum(map(len, tokens))
    if flops > 4e14:
        return None
    w = _weights(case, seed)
    with torch.no_grad():
        if _family(case) == "gpt2":
            return torch.cat([_gpt2_last(_config(case), w, t) for t in _groups(tokens)])
        n = case["new"]
        rows = torch.stack([_zatinex_tail(_config(case), w, t, n + 1) for t in tokens])
        return [rows[:, k].contiguous() for k in range(n + 1)]


def _groups(tokens):
    """Neighbours of one length, run together."""
    out = []
    for t in tokens:
        if out and len(out[-1][0]) == len(t) and len(out[-1]) * len(t) < 8192:
            out[-1].append(t)
        else:
            out.append([t])
    return out


def _layer_norm(x, w, name, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w[name + ".weight"].double() + w[name + ".bias"].double()


def _attend(q, k, v, scale, rows=512):
    """Causal softmax attention: ``q``, ``k`` ``[heads, T, d]``, ``v`` ``[heads, T, dv]``, some queries at a time."""
    H, T, out = q.shape[0], q.shape[1], []
    rows = max(1, min(rows, (1 << 28) // (H * T)))
    kt = k.transpose(1, 2).contiguous()
    for a in range(0, T, rows):
        b = min(T, a + rows)
        s = torch.bmm(q[:, a:b].contiguous(), kt) * scale
        late = torch.arange(T, device=q.device)[None, :] > torch.arange(a, b, device=q.device)[:, None]
        out.append(torch.bmm(torch.softmax(s.masked_fill(late, float("-inf")), -1), v))
    return torch.cat(out, 1)


def _gpt2_last(c, w, prompts):
    """Logits ``[prompts, vocab]`` of the last token of prompts of one length."""
    D, H, eps = c["n_embd"], c["n_head"], c["layer_norm_epsilon"]
    B, T, d = len(prompts), len(prompts[0]), c["n_embd"] // c["n_head"]
    ids = torch.tensor(prompts, device="cuda")
    x = (w["wte.weight"][ids].double() + w["wpe.weight"][:T].double()).reshape(B * T, D)

    def linear(x, name):
        return x @ w[name + ".weight"].double() + w[name + ".bias"].double()

    for i in range(c["n_layer"]):
        p = f"h.{i}."
        qkv = linear(_layer_norm(x, w, p + "ln_1", eps), p + "attn.c_attn").view(B, T, 3, H, d)
        q, k, v = (qkv[:, :, j].transpose(1, 2).reshape(B * H, T, d) for j in range(3))
        o = _attend(q, k, v, d ** -0.5).view(B, H, T, d).transpose(1, 2).reshape(B * T, D)
        x = x + linear(o, p + "attn.c_proj")
        u = linear(_layer_norm(x, w, p + "ln_2", eps), p + "mlp.c_fc")
        u = 0.5 * u * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (u + 0.044715 * u ** 3)))
        x = x + linear(u, p + "mlp.c_proj")
    x = x.view(B, T, D)[:, -1]
    return _layer_norm(x, w, "ln_f", eps) @ w["wte.weight"].double().t().contiguous()


def _rms(x, weight, eps):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight.double()


def _frequencies(rot):
    """A rotation's frequencies, and the factor of its cosines and sines: with ``scaling`` the slow ones are divided."""
    n, base = rot["dims"], rot["base"]
    f = [base ** (-2.0 * i / n) for i in range(n // 2)]
    s = rot.get("scaling")
    if not s:
        return f, 1.0

    def place(turns):
        return n * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(base))

    lo, hi = max(math.floor(place(s["fast"])), 0), min(math.ceil(place(s["slow"])), n - 1)
    ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(n // 2)]
    return [x * (1 - r) + x / s["factor"] * r for x, r in zip(f, ramp)], 0.1 * math.log(s["factor"]) + 1.0


def _turn(x, rot):
    """``x`` ``[T, ..., n]``: neighbours ``2i`` and ``2i + 1`` of the first ``dims`` columns turn with the position."""
    f, mult = _frequencies(rot)
    n = 2 * len(f)
    f = torch.tensor(f, dtype=F64, device=x.device)
    angle = (torch.arange(x.shape[0], device=x.device, dtype=F64)[:, None] * f).view(x.shape[0], *[1] * (x.dim() - 2), n // 2)
    c, s = torch.cos(angle) * mult, torch.sin(angle) * mult
    u, v = x[..., 0:n:2], x[..., 1:n:2]
    return torch.cat([torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2), x[..., n:]], -1)


def _zatinex_tail(c, w, tokens, n_last):
    """Logits ``[n_last, vocab]`` of one request's last tokens."""
    eps, T = c["norm"]["eps"], len(tokens)
    x = w["embed"][torch.tensor(tokens, device="cuda")].double()

    def linear(x, name):
        return x @ w[name].double().t().contiguous()

    def heads_first(x):
        return x.transpose(0, 1).contiguous()

    latents = {}
    for i, layer in enumerate(c["layers"]):
        p, m, q_ = f"l{i}.", layer["mixer"], f"l{i}.mix."
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        h = _rms(x, w[p + "norm1"], eps)
        if layer["type"] == "attention":
            got = []
            for name in ("q", "k", "v"):
                u, taps = linear(h, q_ + name) + w[q_ + name + ".b"].double(), w[q_ + name + ".conv"].double()
                y = torch.zeros_like(u)
                for j in range(m["conv"]):
                    back = m["conv"] - 1 - j
                    if back < T:
                        y[back:] += taps[:, j] * u[: T - back]
                got.append(y)
            q, k = (_turn(_rms(y.view(T, H, 2, d), w[q_ + name + ".norm"], eps), m["rot"]) for y, name in zip(got, ("q", "k")))
            v = heads_first(got[2].view(T, H, dv))
            a, b = (_attend(heads_first(q[:, :, j]), heads_first(k[:, :, j]), v, m["scale"]) for j in (0, 1))
            lam = (torch.exp((w[q_ + "lq1"].double() * w[q_ + "lk1"].double()).sum())
                   - torch.exp((w[q_ + "lq2"].double() * w[q_ + "lk2"].double()).sum()) + m["diff"])
            o = heads_first(_rms(a - lam * b, None, eps) * (1.0 - m["diff"])).view(T, H * dv)
        elif layer["type"] == "gla":
            q, k, v = ((linear(h, q_ + name)).view(T, H, -1) for name in ("q", "k", "v"))
            z = linear(linear(h, q_ + "a1"), q_ + "a2") + w[q_ + "a2.b"].double()
            alpha = torch.sigmoid(z).pow(1.0 / m["tau"]).view(T, H, d, 1)
            S, o = torch.zeros(H, d, dv, dtype=F64, device=x.device), torch.empty(T, H, dv, dtype=F64, device=x.device)
            added = k[..., None] * v[:, :, None, :]
            for t in range(T):
                S = torch.addcmul(added[t], alpha[t], S)
                o[t] = (S * q[t][..., None]).sum(1)
            o = _rms(o * d ** -0.5, w[q_ + "norm"], eps).view(T, H * dv)
            gate = linear(h, q_ + "g")
            o = o * gate * torch.sigmoid(gate)
        else:
            r = m["kv_rank"]
            q = linear(_rms(linear(h, q_ + "dq"), w[q_ + "dq.norm"], eps), q_ + "uq").view(T, H, -1)
            if "kv_from" in m:
                lat, turned = latents[m["kv_from"]]
            else:
                both = linear(h, q_ + "dkv")
                lat, turned = latents[i] = _rms(both[:, :r], w[q_ + "dkv.norm"], eps), _turn(both[:, r:], m["rot"])
            k = torch.cat([linear(lat, q_ + "uk").view(T, H, d), turned[:, None].expand(T, H, -1)], -1)
            q = torch.cat([q[..., :d], _turn(q[..., d:], m["rot"])], -1)
            o = _attend(heads_first(q), heads_first(k), heads_first(linear(lat, q_ + "uv").view(T, H, dv)), m["scale"])
            o = (heads_first(o) * torch.sigmoid(linear(h, q_ + "g"))[..., None]).reshape(T, H * dv)
        x = x + linear(o, q_ + "o")
        h = _rms(x, w[p + "norm2"], eps)
        gate = linear(h, p + "mlp.gate")
        x = x + linear(gate * torch.sigmoid(gate) * linear(h, p + "mlp.up"), p + "mlp.down")
    return linear(_rms(x[-n_last:], w["final.norm"], eps), "head")

