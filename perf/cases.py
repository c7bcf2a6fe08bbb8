"""Timed cases of the decoder framework: what a program that transcribes with it
has it do, through the public entry points of `qasr_attn`.

A case is a dict of plain values.  `kind` says which entry points it takes:

  decode   qk-norm + MRoPE + KV append + attention of one decode step
           (`decode_step`), `layers` layers, each on its own cache
  prefill  the same stages of one prefill chunk (`prefill_layer`)
  gemm     one prefill projection (`gemm_f16`)
  step     one token step of a text decoder (`TextDecoder.step_tokens`)
  prompt   prefill of one or several prompts by a text decoder
           (`TextDecoder.prefill` / `prefill_batch`)

The shapes are the 0.6B and 1.7B Qwen3 text decoders of bench.py and the tests
(16 q / 8 kv heads of 128, hidden 1024 / 2048, MLP 3072 / 6144, vocabulary
151,936); weights, caches and activations are seeded random values scaled as
bench.py scales them.  The attention layers are captured in a HIP graph, as
bench.py runs them (one layer's launches are shorter than a Python call); the
decoder and GEMM calls are plain calls.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "qwen3-asr-wgpu_amd"))

NQH, NKVH, HD = 16, 8, 128
QDIM, KDIM = NQH * HD, NKVH * HD
TOT = QDIM + 2 * KDIM
VOCAB = 151936
EPS = 1e-6
THETA = 1e6
MODELS = {"0.6B": (1024, 3072), "1.7B": (2048, 6144)}
PROJECTIONS = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")


def listed():
    return [
        # The smallest call: one live transcription, 512 keys, all 28 layers.
        {"name": "decode 1 slot", "kind": "decode", "layers": 28, "slots": 1, "lo": 511, "hi": 511},
        # The headline workload: 16 slots with ragged contexts.
        {"name": "decode 16 slots ragged", "kind": "decode", "layers": 28, "slots": 16, "lo": 400,
         "hi": 2400},
        # One long recording's context.
        {"name": "decode 1 slot long", "kind": "decode", "layers": 28, "slots": 1, "lo": 8192,
         "hi": 8192},
        # The attention of one 420-row prompt (30 s of audio).
        {"name": "prefill 420", "kind": "prefill", "layers": 28, "rows": 420, "start": 0},
        # The last chunk of a long prompt prefilled in 512-row chunks.
        {"name": "prefill 512 at 7680", "kind": "prefill", "layers": 8, "rows": 512, "start": 7680},
        # down_proj of one prompt, without the residual: few tiles, a long sum.
        {"name": "gemm 420x2048x6144", "kind": "gemm", "m": 420, "n": 2048, "k": 6144},
        # gate|up of 16 prompts together.
        {"name": "gemm 4269x12288x2048", "kind": "gemm", "m": 4269, "n": 12288, "k": 2048},
        # One live transcription's token step, int8 weights, the small model.
        {"name": "step 0.6B int8 1 slot", "kind": "step", "model": "0.6B", "int8": True,
         "layers": 28, "slots": 1, "lo": 511, "hi": 511},
        # A batch job's token step.
        {"name": "step 1.7B 16 slots", "kind": "step", "model": "1.7B", "int8": False,
         "layers": 28, "slots": 16, "lo": 400, "hi": 2400},
        # A short continuation of a stream, the cached prefix kept; int8 weights.
        {"name": "prompt 0.6B int8 131 at 300", "kind": "prompt", "model": "0.6B", "int8": True,
         "layers": 8, "prompts": 1, "lo": 131, "hi": 131, "start": 300},
        # One prompt: the time to the first token.
        {"name": "prompt 1.7B 420", "kind": "prompt", "model": "1.7B", "int8": False, "layers": 8,
         "prompts": 1, "lo": 420, "hi": 420, "start": 0},
        # A batch job's admission: 16 prompts of 150-450 rows in one call.
        {"name": "prompt 1.7B 16 batched", "kind": "prompt", "model": "1.7B", "int8": False,
         "layers": 4, "prompts": 16, "lo": 150, "hi": 450, "start": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "gemm", "step", "prompt", "prompt"])
    if kind == "decode":
        slots = _log_int(rng, 1, 16)
        lo = _log_int(rng, 32, 2400)
        hi = min(_log_int(rng, lo, 8192), 2400 if slots > 4 else 8192)
        return {"kind": kind, "layers": rng.randint(4, 28), "slots": slots, "lo": lo,
                "hi": max(lo, hi)}
    if kind == "prefill":
        rows = _log_int(rng, 5, 1024)
        start = rng.choice([0, _log_int(rng, 50, 7680)])
        return {"kind": kind, "layers": rng.randint(4, 8), "rows": rows, "start": start}
    if kind == "gemm":
        n, k = rng.choice([(4096, 1024), (1024, 2048), (6144, 1024), (1024, 3072),
                           (4096, 2048), (2048, 2048), (12288, 2048), (2048, 6144)])
        return {"kind": kind, "m": _log_int(rng, 17, 4269), "n": n, "k": k}
    model = rng.choice(["0.6B", "1.7B"])
    int8 = rng.random() < 0.4
    if kind == "step":
        lo = _log_int(rng, 100, 1600)
        return {"kind": kind, "model": model, "int8": int8, "layers": rng.randint(4, 28),
                "slots": _log_int(rng, 1, 16), "lo": lo, "hi": rng.randint(lo, 1800)}
    if rng.random() < 0.5:
        rows = _log_int(rng, 9, 1024)
        return {"kind": kind, "model": model, "int8": int8, "layers": rng.randint(2, 8),
                "prompts": 1, "lo": rows, "hi": rows,
                "start": rng.choice([0, rng.randint(50, 900)])}
    lo = _log_int(rng, 9, 200)
    return {"kind": kind, "model": model, "int8": int8, "layers": rng.randint(2, 4),
            "prompts": rng.randint(2, 16), "lo": lo, "hi": rng.randint(lo, 300), "start": 0}


# ---- inputs ------------------------------------------------------------------

def _lengths(lo, hi, n, salt):
    """n lengths over [lo, hi], the same for every seed of a case (the work of
    a case is fixed), by a SplitMix64 walk."""
    if lo >= hi:
        return [lo] * n
    state, out = (0x51A50000 + salt) & (2 ** 64 - 1), []
    for _ in range(n):
        state = (state + 0x9E3779B97F4A7C15) & (2 ** 64 - 1)
        z = state
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & (2 ** 64 - 1)
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & (2 ** 64 - 1)
        out.append(lo + (z ^ (z >> 31)) % (hi - lo + 1))
    return out


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, std=1.0, mean=0.0):
    return (torch.randn(shape, device="cuda", generator=g) * std + mean).half()


def _cap(need):
    return max(1024, (need + 255) // 256 * 256)


def _attn_inputs(case, seed):
    """Raw qkv rows, gains and cached rows of an attention case."""
    g = _gen(seed)
    layers = case["layers"]
    if case["kind"] == "decode":
        cached = _lengths(case["lo"], case["hi"], case["slots"], 3)
        rows = case["slots"]
    else:
        cached, rows = [case["start"]], case["rows"]
    return {"cached": cached, "rows": rows,
            "qkv": _normal(g, (layers, rows, TOT)),
            "gains": _normal(g, (layers, 2, HD), 0.1, 1.0),
            "cache": [_normal(g, (layers, 2, NKVH, n, HD)) for n in cached]}


def _weights(case, g):
    """Decoder weights keyed like a checkpoint's tensors; int8 linears with a
    scale per output row where the case asks for them."""
    hs, inter = MODELS[case["model"]]
    shapes = {"q_proj": (QDIM, hs), "k_proj": (KDIM, hs), "v_proj": (KDIM, hs),
              "o_proj": (hs, QDIM), "gate_proj": (inter, hs), "up_proj": (inter, hs),
              "down_proj": (hs, inter)}
    W = {"embed": _normal(g, (VOCAB, hs), 0.1), "norm": _normal(g, (hs,), 0.1, 1.0)}
    for l in range(case["layers"]):
        for name in ("input_layernorm", "post_attention_layernorm"):
            W[(l, name)] = _normal(g, (hs,), 0.1, 1.0)
        for name in ("q_norm", "k_norm"):
            W[(l, name)] = _normal(g, (HD,), 0.1, 1.0)
        for name in PROJECTIONS:
            w = torch.randn(shapes[name], device="cuda", generator=g) * shapes[name][1] ** -0.5
            if case["int8"]:
                s = w.abs().amax(dim=1).clamp_min(1e-8) / 127.0
                W[(l, name)] = torch.round(w / s[:, None]).clamp(-128, 127).to(torch.int8)
                W[(l, name + "_scale")] = s
            else:
                W[(l, name)] = w.half()
    return W


def _model_inputs(case, seed):
    g = _gen(seed)
    out = {"W": _weights(case, g)}
    hs = MODELS[case["model"]][0]
    if case["kind"] == "step":
        out["cached"] = _lengths(case["lo"], case["hi"], case["slots"], 3)
        out["tokens"] = torch.randint(0, VOCAB, (case["slots"],), dtype=torch.int32, device="cuda",
                                      generator=g)
    else:
        out["rows"] = _lengths(case["lo"], case["hi"], case["prompts"], 23)
        out["cached"] = [case["start"]] * case["prompts"]
        out["hidden"] = [_normal(g, (n, hs)) for n in out["rows"]]
    out["cache"] = [_normal(g, (case["layers"], 2, NKVH, n, HD)) for n in out["cached"]]
    return out


def _gemm_inputs(case, seed):
    g = _gen(seed)
    return (_normal(g, (case["m"], case["k"])),
            _normal(g, (case["n"], case["k"]), case["k"] ** -0.5))


# ---- the framework's calls ---------------------------------------------------

def prepare(case, seed):
    import qasr_attn as q

    kind = case["kind"]
    if kind == "gemm":
        a, b = _gemm_inputs(case, seed)
        return {"kind": kind, "q": q, "ctx": q.Context(), "a": a, "b": b,
                "c": torch.empty((case["m"], case["n"]), dtype=torch.float16, device="cuda")}
    if kind in ("decode", "prefill"):
        return _prepare_attn(case, seed, q)
    x = _model_inputs(case, seed)
    n = len(x["cached"])
    news = [1] * n if kind == "step" else x["rows"]
    dec = q.TextDecoder(x.pop("W"), NQH, NKVH, HD, case["layers"], EPS, 16384, slots=n,
                        max_rows=max(16, sum(news)),
                        cap=_cap(max(c + m for c, m in zip(x["cached"], news))))
    pool = dec.kv.tensor()
    for i, rows in enumerate(x.pop("cache")):
        pool[i, :, :, :, :rows.shape[3]].copy_(rows)
    st = {"kind": kind, "dec": dec, "pos": x["cached"],
          "logits": torch.empty((n, VOCAB), dtype=torch.float32, device="cuda"),
          "kv": _rows_written(dec, pool, x["cached"], news)}
    if kind == "step":
        st.update(slots=list(range(n)), tokens=x["tokens"], next=torch.empty_like(x["tokens"]))
    else:
        st.update(hidden=x["hidden"], start=case["start"])
    return st


def _rows_written(owner, pool, starts, counts):
    """Views of the K/V rows a pass appends.  The pool's memory is the
    library's and goes with its owner, so each view holds on to it."""
    views = [pool[i, :, :, :, c:c + m] for i, (c, m) in enumerate(zip(starts, counts))]
    for v in views:
        v.owner = owner
    return views


def _prepare_attn(case, seed, q):
    x = _attn_inputs(case, seed)
    layers, n, rows = case["layers"], len(x["cached"]), x["rows"]
    new = 1 if case["kind"] == "decode" else rows
    ctx = q.Context(NQH, NKVH, HD, layers, EPS, 16384, 0)
    ctx.set_rope_tables(*q.mrope_text_tables(16384))
    kv = q.KVPool(ctx, n, _cap(max(x["cached"]) + new))
    pool = kv.tensor()
    for i, c in enumerate(x.pop("cache")):
        pool[i, :, :, :, :c.shape[3]].copy_(c)
    qkv, gains = x["qkv"], x["gains"]
    out = torch.empty((layers, rows, QDIM), dtype=torch.float16, device="cuda")
    work = torch.empty((rows, QDIM), dtype=torch.float16, device="cuda")

    def layers_once():
        for l in range(layers):
            if case["kind"] == "decode":
                q.decode_step(ctx, kv, l, x["cached"], qkv[l], gains[l, 0], gains[l, 1], out[l])
            else:
                q.prefill_layer(ctx, kv, l, 0, case["start"], rows, qkv[l], gains[l, 0],
                                gains[l, 1], work, out[l])

    layers_once()  # argument checks and workspace growth, before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layers_once()
    return {"kind": case["kind"], "graph": graph, "out": out, "keep": (ctx, kv, qkv, gains, work),
            "kv": _rows_written(kv, pool, x["cached"], [new] * n)}


def run(state):
    kind = state["kind"]
    if kind == "gemm":
        return state["q"].gemm_f16(state["ctx"], state["a"], state["b"], state["c"])
    if kind in ("decode", "prefill"):
        state["graph"].replay()
        return [state["out"], state["kv"]]
    dec, logits = state["dec"], state["logits"]
    if kind == "step":
        dec.step_tokens(state["slots"], state["pos"], state["tokens"], state["next"], logits)
    elif len(state["hidden"]) == 1:
        dec.prefill(state["hidden"][0], state["start"], logits=logits[0])
    else:
        dec.prefill_batch(list(enumerate(state["hidden"])), logits=logits)
    return [logits, state["kv"]]


# ---- what a pass cannot do without -------------------------------------------

def _attn_work(cached, new):
    """Bytes and FLOPs of one layer's attention: qkv rows in, K/V rows read and
    appended, outputs; causal-exact products (2 x 2 x 128 per key and q head)."""
    b = f = 0
    for c, m in zip(cached, new):
        b += 2 * (m * TOT + 2 * KDIM * (c + m) + m * QDIM)
        f += 4 * HD * NQH * (m * c + m * (m + 1) // 2)
    return b, f


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + n * k + m * n), "flops": 2 * m * n * k}
    layers = case["layers"]
    if kind == "decode":
        b, f = _attn_work(_lengths(case["lo"], case["hi"], case["slots"], 3), [1] * case["slots"])
        return {"bytes": layers * b, "flops": layers * f}
    if kind == "prefill":
        b, f = _attn_work([case["start"]], [case["rows"]])
        return {"bytes": layers * b, "flops": layers * f}
    hs, inter = MODELS[case["model"]]
    if kind == "step":
        cached = _lengths(case["lo"], case["hi"], case["slots"], 3)
        new = [1] * case["slots"]
    else:
        new = _lengths(case["lo"], case["hi"], case["prompts"], 23)
        cached = [case["start"]] * case["prompts"]
    rows, n = sum(new), len(new)
    proj = TOT * hs + QDIM * hs + 3 * inter * hs
    kv = sum(2 * 2 * KDIM * (c + m) for c, m in zip(cached, new))
    _, f = _attn_work(cached, new)
    return {"bytes": layers * (proj * (1 if case["int8"] else 2) + kv) + 2 * VOCAB * hs
            + 2 * rows * hs + 4 * n * VOCAB,
            "flops": layers * (2 * proj * rows + f) + 2 * n * VOCAB * hs}


def tolerance(case):
    """About four times the largest error against 64 bits that the listed and
    some drawn cases showed at f16 storage with f32 sums: gemm 2.1e-4 (one f16
    rounding), attention 3.6e-4; text decoders 4.8e-3 over 28 layers and
    1.4e-3 over 8, whose roundings add up layer by layer."""
    kind = case["kind"]
    if kind == "gemm":
        return {"rel": 8e-4}
    if kind in ("decode", "prefill"):
        return {"rel": 1.4e-3}
    return {"rel": 2e-2 if case["layers"] > 8 else 5.6e-3}


# ---- the same results in 64 bits ---------------------------------------------

def _rope(x, gain, pos):
    """q/k RMSNorm with `gain` and rotate-half RoPE: x [rows][heads][128]; the
    cos / sin tables are f16 by definition."""
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * gain
    inv = THETA ** (-2.0 * torch.arange(HD // 2, dtype=torch.float64, device="cuda") / HD)
    ang = pos.double()[:, None] * inv
    c, s = ang.cos().float().half().double()[:, None], ang.sin().float().half().double()[:, None]
    a, b = y[..., :HD // 2], y[..., HD // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(qkv, qg, kg, cache, start):
    """One layer's attention of rows at start..: (outputs, new K/V rows)."""
    m = qkv.shape[0]
    pos = torch.arange(start, start + m, device="cuda")
    h = qkv.view(m, NQH + 2 * NKVH, HD)
    q = _rope(h[:, :NQH], qg, pos).transpose(0, 1)
    new = torch.stack([_rope(h[:, NQH:NQH + NKVH], kg, pos), h[:, NQH + NKVH:]]).transpose(1, 2)
    k, v = torch.cat([cache[:, :, :start].double(), new], 2)
    out = torch.empty((m, NQH, HD), dtype=torch.float64, device="cuda")
    keys = torch.arange(start + m, device="cuda")
    for i in range(NQH):
        s = q[i] @ k[i // 2].t() / math.sqrt(HD)
        s.masked_fill_(keys[None] > pos[:, None], -math.inf)
        out[:, i] = torch.softmax(s, -1) @ v[i // 2]
    return out.reshape(m, QDIM), new


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        a, b = _gemm_inputs(case, seed)
        return a.double() @ b.double().t()
    if kind in ("decode", "prefill"):
        x = _attn_inputs(case, seed)
        per = 1 if kind == "decode" else x["rows"]
        out, kv = [], [[] for _ in x["cached"]]
        for l in range(case["layers"]):
            rows = []
            qg, kg = x["gains"][l].double()
            for i, c in enumerate(x["cached"]):
                o, new = _attend(x["qkv"][l, i * per:(i + 1) * per].double(), qg, kg,
                                 x["cache"][i][l], c)
                rows.append(o)
                kv[i].append(new)
            out.append(torch.cat(rows))
        return [torch.stack(out), [torch.stack(k) for k in kv]]
    x = _model_inputs(case, seed)
    W = x["W"]

    def linear(h, l, name):
        w = W[(l, name)]
        if case["int8"]:  # the weight is f16(q * scale) by definition
            w = (w.float() * W[(l, name + "_scale")][:, None]).half()
        return h @ w.double().t()

    def norm(h, w):
        return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * w.double()

    if kind == "step":
        h, new = W["embed"][x["tokens"].long()].double(), [1] * len(x["cached"])
    else:
        h, new = torch.cat(x["hidden"]).double(), x["rows"]
    kv = [[] for _ in new]
    for l in range(case["layers"]):
        n = norm(h, W[(l, "input_layernorm")])
        qkv = torch.cat([linear(n, l, p) for p in ("q_proj", "k_proj", "v_proj")], 1)
        qg, kg = W[(l, "q_norm")].double(), W[(l, "k_norm")].double()
        rows, r0 = [], 0
        for i, m in enumerate(new):
            o, fresh = _attend(qkv[r0:r0 + m], qg, kg, x["cache"][i][l], x["cached"][i])
            rows.append(o)
            kv[i].append(fresh)
            r0 += m
        h = h + linear(torch.cat(rows), l, "o_proj")
        n = norm(h, W[(l, "post_attention_layernorm")])
        h = h + linear(torch.nn.functional.silu(linear(n, l, "gate_proj"))
                       * linear(n, l, "up_proj"), l, "down_proj")
    last = torch.tensor(new, device="cuda").cumsum(0) - 1
    logits = norm(h[last], W["norm"]) @ W["embed"].double().t()
    return [logits, [torch.stack(k) for k in kv]]
