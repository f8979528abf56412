"""Performance cases of the device: what a program does through tensomite_hip's
public entry points, from one small product to a whole generation.

A case is a dict of plain values; its "work" names the path:

  product    dst = x · wᵀ (+ bias), HIPDevice.block_matmul: one linear layer
             of a decode step (1 row), of batched decode (2 to 31 rows) or of
             a prompt (32 rows and more)
  plan       the one-row products of a whole token recorded once and run as
             one launch, HIPDevice.plan
  attention  queries against the f32 KV cache, HIPDevice.attention: a
             prompt's (causal, every position its own end) or a batched
             decode step's (one query a sequence, ragged lengths)
  mlp        RMSNorm, gate_up, SwiGLU, down and the residual, op by op, as a
             host that schedules the graph itself issues them
  attn_block RMSNorm, qkv, RoPE with the cache write, attention, o and the
             residual, op by op
  generate   the device-resident decoder, HIPLlama: every row's prompt
             (its last logits), greedy tokens, and the logits after them

The device promises the host path's bits for all of these, whatever kernel
runs, so every result is compared exactly.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "tensomite.cr_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "tensomite.cr_amd"))

import tensomite_hip as th  # noqa: E402

BLOCK = th.BLOCK_BYTES
KIND = th.KINDS

# The Llama shapes of the repository's configurations: SmolLM2-135M and the
# 1.7B shape.
MODELS = {
    "135m": dict(layers=30, width=576, heads=9, kv_heads=3, head_width=64, hidden=1536, vocab=49152),
    "1p7b": dict(layers=24, width=2048, heads=32, kv_heads=32, head_width=64, hidden=8192, vocab=49152),
}
CONTEXT, EPS, THETA = 2048, 1e-5, 10000.0


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # GPT-2 small's c_attn at decode: the smallest call, a launch and little else.
        {"name": "c_attn_row", "work": "product", "kind": "Q8_0", "rows": 1, "n": 2304, "k": 768, "bias": True},
        # The tied head of the 1.7B shape at decode: the largest single one-row product.
        {"name": "head_row", "work": "product", "kind": "Q4_0", "rows": 1, "n": 49152, "k": 2048, "bias": False},
        # Batched decode: four sequences through an MLP's up projection.
        {"name": "up_4_rows", "work": "product", "kind": "Q4_1", "rows": 4, "n": 8192, "k": 2048, "bias": False},
        # Batched decode: sixteen sequences through the down projection (long rows).
        {"name": "down_16_rows", "work": "product", "kind": "Q4_1", "rows": 16, "n": 2048, "k": 8192, "bias": False},
        # A 512-token prompt through an MLP projection.
        {"name": "prefill_512_rows", "work": "product", "kind": "Q8_0", "rows": 512, "n": 8192, "k": 2048,
         "bias": False},
        # SmolLM2-135M: a token's 121 products in one launch.
        {"name": "token_plan", "work": "plan", "kind": "Q4_0", "model": "135m", "layers": 30, "head": True},
        # A 512-token prompt's attention in one layer of the 1.7B shape.
        {"name": "attention_prompt", "work": "attention", "heads": 32, "kv_heads": 32, "width": 64, "prompt": True,
         "past": 0, "tokens": 512, "capacity": 2048},
        # Eight sequences' decode attention, ragged lengths up to the context.
        {"name": "attention_decode", "work": "attention", "heads": 32, "kv_heads": 32, "width": 64, "prompt": False,
         "past": 2000, "tokens": 8, "capacity": 2048},
        # An MLP block of the 1.7B shape over a short prompt, op by op.
        {"name": "mlp_100_rows", "work": "mlp", "kind": "Q4_0", "model": "1p7b", "rows": 100},
        # An attention block of SmolLM2-135M (grouped heads, rows of 18
        # blocks) over a ragged prompt, op by op.
        {"name": "attn_block_77_rows", "work": "attn_block", "kind": "Q8_0", "model": "135m", "rows": 77,
         "capacity": 512},
        # One user: a 128-token prompt, then 64 greedy tokens, 1.7B shape.
        {"name": "generate_1", "work": "generate", "kind": "Q4_0", "model": "1p7b", "rows": 1, "prompt": 128,
         "steps": 64},
        # Eight users: ragged prompts of up to 300 tokens, then 32 greedy tokens each.
        {"name": "generate_8", "work": "generate", "kind": "Q4_0", "model": "1p7b", "rows": 8, "prompt": 300,
         "steps": 32},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    work = rng.choice(["product"] * 5 + ["plan", "attention", "attention", "mlp", "attn_block", "generate"])
    kind = rng.choice(["Q8_0", "Q4_0", "Q4_1"])
    if work == "product":
        rows = rng.choice([1, _log_int(rng, 2, 8), _log_int(rng, 9, 31), _log_int(rng, 32, 512)])
        k = 64 * _log_int(rng, 8, 128)
        n = _log_int(rng, 192, 49152 if rows <= 8 else 8192)
        return {"work": work, "kind": kind, "rows": rows, "n": n - n % rng.choice([1, 64, 64]), "k": k,
                "bias": rng.random() < 0.3}
    if work == "plan":
        return {"work": work, "kind": kind, "model": "135m", "layers": rng.randint(1, 30), "head": rng.random() < 0.5}
    if work == "attention":
        kv = rng.choice([3, 4, 8, 32])
        prompt = rng.random() < 0.5
        case = {"work": work, "heads": kv * rng.choice([1, 3]) if kv < 32 else 32, "kv_heads": kv,
                "width": rng.choice([64, 64, 128]), "prompt": prompt}
        if prompt:
            case.update(past=rng.choice([0, _log_int(rng, 1, 512)]), tokens=_log_int(rng, 16, 512))
        else:
            case.update(past=_log_int(rng, 32, 2000), tokens=rng.randint(1, 8))
        return dict(case, capacity=CONTEXT)
    if work == "mlp":
        return {"work": work, "kind": kind, "model": rng.choice(["135m", "1p7b"]), "rows": _log_int(rng, 1, 256)}
    if work == "attn_block":
        return {"work": work, "kind": kind, "model": rng.choice(["135m", "1p7b"]), "rows": _log_int(rng, 1, 256),
                "capacity": rng.choice([512, CONTEXT])}
    model = rng.choice(["135m", "1p7b"])
    return {"work": work, "kind": kind, "model": model, "rows": rng.choice([1, 1, 2, 4, 8]),
            "prompt": _log_int(rng, 4, 256), "steps": _log_int(rng, 4, 32)}


# ------------------------------------------------- inputs, as a program has them

class Borrowed(th.Buffer):
    """A torch tensor's memory as a device buffer: torch keeps owning it."""

    def __init__(self, device, tensor):
        super().__init__(device, tensor.data_ptr(), tensor.numel() * tensor.element_size())
        self.tensor = tensor

    def release(self):
        pass

    def __del__(self):
        pass


_device = None


def _dev():
    global _device
    if _device is None:
        _device = th.HIPDevice(0)
    return _device


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, *shape, std=1.0):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32) * std


def _quantise(values, kind):
    """[n, k] f32 weights as ggml block bytes [n, k / 32 · block bytes]."""
    n, k = values.shape
    v = values.view(n, k // 32, 32)
    if kind == "Q8_0":
        d = v.abs().amax(-1, keepdim=True) / 127.0
        q = torch.where(d > 0, v / d, torch.zeros_like(v)).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        parts = [_half_bytes(d), q]
    else:
        if kind == "Q4_0":
            at = v.abs().argmax(-1, keepdim=True)
            d = v.gather(-1, at) / -8.0
            low = []
            q = torch.where(d != 0, v / d, torch.zeros_like(v)) + 8.5
        else:
            m = v.amin(-1, keepdim=True)
            d = (v.amax(-1, keepdim=True) - m) / 15.0
            low = [_half_bytes(m)]
            q = torch.where(d > 0, (v - m) / d, torch.zeros_like(v)) + 0.5
        q = q.floor().clamp(0, 15).to(torch.uint8)
        parts = [_half_bytes(d), *low, q[..., :16] | (q[..., 16:] << 4)]
    return torch.cat(parts, -1).reshape(n, -1).contiguous()


def _half_bytes(v):
    return v.to(torch.float16).contiguous().view(torch.uint8)


def _weights(gen, n, k, kind):
    return _quantise(_normal(gen, n, k, std=0.02), kind)


def _norm(gen, n):
    return 1.0 + _normal(gen, n, std=0.05)


def _lengths(case, seed):
    """Positions a decode query sees, per sequence: ragged up to `past` + 1."""
    rng = np.random.default_rng(seed)
    out = rng.integers(max(1, case["past"] // 4), case["past"] + 2, case["tokens"])
    out[0] = case["past"] + 1
    return out


def _rope_tables(capacity, width):
    freq = 1.0 / torch.pow(torch.tensor(THETA), torch.arange(0, width, 2, dtype=torch.float32) / width)
    angle = torch.arange(capacity, dtype=torch.float32)[:, None] * torch.cat([freq, freq])[None]
    return angle.cos().cuda(), angle.sin().cuda()


def _prompts(case, seed):
    """Each row's prompt ids: row 0 has `prompt` of them, the others at least a quarter."""
    rng = np.random.default_rng(seed)
    c = MODELS[case["model"]]
    sizes = [case["prompt"]] + [int(rng.integers(max(1, case["prompt"] // 4), case["prompt"] + 1))
                                for _ in range(case["rows"] - 1)]
    return [rng.integers(0, c["vocab"], size).astype(np.int32) for size in sizes]


def _products(case):
    c = MODELS[case["model"]]
    kv = c["kv_heads"] * c["head_width"]
    qn = c["heads"] * c["head_width"]
    layer = [(qn + 2 * kv, c["width"]), (c["width"], qn), (2 * c["hidden"], c["width"]), (c["width"], c["hidden"])]
    return layer * case["layers"] + ([(c["vocab"], c["width"])] if case["head"] else [])


def _tensors(case, seed):
    """The case's inputs as torch tensors on the GPU (weights as block bytes)."""
    gen, work = _gen(seed), case["work"]
    if work == "product":
        return {"w": _weights(gen, case["n"], case["k"], case["kind"]), "x": _normal(gen, case["rows"], case["k"]),
                "bias": _normal(gen, case["n"], std=0.1) if case["bias"] else None}
    if work == "plan":
        return {"items": [(_weights(gen, n, k, case["kind"]), _normal(gen, k)) for n, k in _products(case)]}
    if work == "attention":
        tokens, heads, kv, hw, cap = (case[key] for key in ("tokens", "heads", "kv_heads", "width", "capacity"))
        rows = 1 if case["prompt"] else tokens
        if case["prompt"]:
            table = [(0, case["past"] + t, case["past"] + tokens) for t in range(tokens)]
        else:
            table = [(t, int(n) - 1, int(n)) for t, n in enumerate(_lengths(case, seed))]
        return {"q": _normal(gen, tokens, heads, hw), "keys": _normal(gen, rows, kv, cap, hw),
                "values": _normal(gen, rows, kv, cap, hw), "table": torch.tensor(table, dtype=torch.int32).cuda()}
    c = MODELS[case["model"]]
    W, H, hw, heads, kv = c["width"], c["hidden"], c["head_width"], c["heads"], c["kv_heads"]
    if work == "mlp":
        return {"x": _normal(gen, case["rows"], W), "norm": _norm(gen, W),
                "gate_up": _weights(gen, 2 * H, W, case["kind"]), "down": _weights(gen, W, H, case["kind"])}
    if work == "attn_block":
        cos, sin = _rope_tables(case["capacity"], hw)
        rows = case["rows"]
        return {"x": _normal(gen, rows, W), "norm": _norm(gen, W),
                "qkv": _weights(gen, (heads + 2 * kv) * hw, W, case["kind"]),
                "o": _weights(gen, W, heads * hw, case["kind"]), "cos": cos, "sin": sin,
                "slots": torch.arange(rows, dtype=torch.int32).cuda(),
                "table": torch.tensor([(0, t, rows) for t in range(rows)], dtype=torch.int32).cuda()}
    layers = range(c["layers"])
    return {"embed": _weights(gen, c["vocab"], W, case["kind"]), "norm": _norm(gen, W),
            "attn_norm": [_norm(gen, W) for _ in layers], "ffn_norm": [_norm(gen, W) for _ in layers],
            "qkv": [_weights(gen, (heads + 2 * kv) * hw, W, case["kind"]) for _ in layers],
            "o": [_weights(gen, W, heads * hw, case["kind"]) for _ in layers],
            "gate_up": [_weights(gen, 2 * H, W, case["kind"]) for _ in layers],
            "down": [_weights(gen, W, H, case["kind"]) for _ in layers]}


def prepare(case, seed):
    dev, work = _dev(), case["work"]
    dev.bind()
    t = _tensors(case, seed)
    buf = lambda a: None if a is None else Borrowed(dev, a)  # noqa: E731
    new = lambda *shape: torch.zeros(*shape, dtype=torch.float32, device="cuda")  # noqa: E731
    state = {"case": dict(case), "dev": dev}
    if work == "product":
        state["out"] = new(case["rows"], case["n"])
        state["args"] = (case["kind"], buf(t["w"]), buf(t["x"]), case["rows"], case["n"], case["k"])
        state["bias"] = buf(t["bias"])
        state["dst"] = buf(state["out"])
    elif work == "plan":
        shapes = _products(case)
        state["out"] = new(sum(n for n, _ in shapes))  # the products' outputs one after another
        dst = state["out"].split([n for n, _ in shapes])
        state["plan"] = dev.plan(case["kind"], [(buf(w), 0, buf(x), buf(y), None, n, k)
                                                for (w, x), y, (n, k) in zip(t["items"], dst, shapes)])
    elif work == "attention":
        state["out"] = new(case["tokens"], case["heads"], case["width"])
        state.update({key: buf(t[key]) for key in ("q", "keys", "values", "table")}, dst=buf(state["out"]))
    elif work == "mlp":
        c, rows = MODELS[case["model"]], case["rows"]
        state["out"] = new(rows, c["width"])
        state.update({key: buf(a) for key, a in t.items()}, h=buf(new(rows, c["width"])),
                     gu=buf(new(rows, 2 * c["hidden"])), act=buf(new(rows, c["hidden"])),
                     y=buf(new(rows, c["width"])), dst=buf(state["out"]))
    elif work == "attn_block":
        c, rows = MODELS[case["model"]], case["rows"]
        cache = (1, c["kv_heads"], case["capacity"], c["head_width"])
        state["out"] = {"y": new(rows, c["width"]), "keys": new(*cache), "values": new(*cache)}
        qn, nqkv = c["heads"] * c["head_width"], (c["heads"] + 2 * c["kv_heads"]) * c["head_width"]
        state.update({key: buf(a) for key, a in t.items()}, h=buf(new(rows, c["width"])), qkv_out=buf(new(rows, nqkv)),
                     q=buf(new(rows, qn)), att=buf(new(rows, qn)), y=buf(new(rows, c["width"])),
                     dst=buf(state["out"]["y"]), keys=buf(state["out"]["keys"]), values=buf(state["out"]["values"]))
    else:
        config = dict(MODELS[case["model"]], context=CONTEXT, eps=EPS, theta=THETA, kind=case["kind"])
        host = {key: [a.cpu().numpy() for a in v] if isinstance(v, list) else v.cpu().numpy() for key, v in t.items()}
        state["model"] = th.HIPLlama(dev, config, host, rows=case["rows"], capacity=CONTEXT,
                                     max_tokens=max(128, min(512, case["prompt"])))
        state["prompts"] = _prompts(case, seed)
    torch.cuda.synchronize()
    return state


# ------------------------------------------------------------------- one pass

def run(state):
    case, dev = state["case"], state["dev"]
    work = case["work"]
    if work == "product":
        dev.block_matmul(*state["args"], dst=state["dst"], bias=state["bias"])
        return state["out"]
    if work == "plan":
        state["plan"].run()
        return state["out"]
    if work == "attention":
        rows = 1 if case["prompt"] else case["tokens"]
        dev.attention(state["q"], case["tokens"], case["heads"], state["keys"], state["values"], rows,
                      case["kv_heads"], case["capacity"], case["width"], state["table"],
                      1.0 / math.sqrt(case["width"]), dst=state["dst"])
        return state["out"]
    if work == "generate":
        model, steps = state["model"], case["steps"]
        model.reset()
        prompt = [model.forward(ids, row=r, last_only=True) for r, ids in enumerate(state["prompts"])]
        tokens = model.generate(steps)
        last = [model.forward(tokens[r, -1:], row=r, last_only=True) for r in range(case["rows"])]
        return {"prompt": np.concatenate(prompt), "tokens": tokens, "logits": np.concatenate(last)}
    c, rows, kind = MODELS[case["model"]], case["rows"], case["kind"]
    W, H, hw, heads, kv = c["width"], c["hidden"], c["head_width"], c["heads"], c["kv_heads"]
    s = state
    dev.rmsnorm(s["x"], s["norm"], rows, W, EPS, dst=s["h"])
    if work == "mlp":
        dev.block_matmul(kind, s["gate_up"], s["h"], rows, 2 * H, W, dst=s["gu"])
        dev.swiglu(s["gu"], s["gu"], 2 * H, rows, H, dst=s["act"], value_offset=H)
        dev.block_matmul(kind, s["down"], s["act"], rows, W, H, dst=s["y"])
    else:
        qn, nqkv, cap = heads * hw, (heads + 2 * kv) * hw, case["capacity"]
        dev.block_matmul(kind, s["qkv"], s["h"], rows, nqkv, W, dst=s["qkv_out"])
        dev.rope_write(s["qkv_out"], nqkv, rows, heads, kv, hw, s["cos"], s["sin"], cap, s["slots"], 1, cap, s["q"],
                       s["keys"], s["values"])
        dev.attention(s["q"], rows, heads, s["keys"], s["values"], 1, kv, cap, hw, s["table"], 1.0 / math.sqrt(hw),
                      dst=s["att"])
        dev.block_matmul(kind, s["o"], s["att"], rows, W, qn, dst=s["y"])
    dev.add(s["x"], s["y"], rows * W, dst=s["dst"])
    return s["out"]


# ---------------------------------------------------------------- what it costs

def _block_bytes(n, k, kind):
    return n * (k // 32) * BLOCK[KIND[kind]]


def _mean_prompt(case):
    return case["prompt"] * (1.0 + (case["rows"] - 1) * 0.625) / case["rows"]


def work(case):
    what = case["work"]
    if what == "product":
        r, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": _block_bytes(n, k, case["kind"]) + 4 * r * (n + k) + (4 * n if case["bias"] else 0),
                "flops": 2 * r * n * k}
    if what == "plan":
        shapes = _products(case)
        return {"bytes": sum(_block_bytes(n, k, case["kind"]) + 4 * (n + k) for n, k in shapes),
                "flops": sum(2 * n * k for n, k in shapes)}
    if what == "attention":
        tokens, heads, kv, hw = case["tokens"], case["heads"], case["kv_heads"], case["width"]
        if case["prompt"]:
            seen = tokens * case["past"] + tokens * (tokens + 1) // 2
            held = case["past"] + tokens
        else:
            seen = held = int(case["past"] * (1.0 + 0.625 * (tokens - 1))) + tokens
        return {"bytes": 4 * (2 * tokens * heads * hw + 2 * held * kv * hw), "flops": 4 * seen * heads * hw}
    c = MODELS[case["model"]]
    W, H, hw, heads, kv, L = c["width"], c["hidden"], c["head_width"], c["heads"], c["kv_heads"], c["layers"]
    qn, nqkv = heads * hw, (heads + 2 * kv) * hw
    rows, kind = case["rows"], case["kind"]
    if what == "mlp":
        return {"bytes": _block_bytes(3 * H, W, kind) + 4 * (2 * rows * W + W), "flops": 6 * rows * H * W}
    if what == "attn_block":
        return {"bytes": _block_bytes(nqkv, W, kind) + _block_bytes(W, qn, kind) + 4 * (2 * rows * W + W)
                + 8 * rows * kv * hw, "flops": 2 * rows * (nqkv * W + W * qn) + 2 * rows * (rows + 1) * heads * hw}
    # every prompt reads the weights once, every step after it once for all
    # rows, the logits after the last token once a row
    layer = nqkv * W + W * qn + 3 * H * W
    weights = _block_bytes(L * layer // 32, 32, kind) + _block_bytes(c["vocab"], W, kind)
    prompt, steps = _mean_prompt(case), case["steps"]
    positions = prompt + steps
    cache = 8 * L * kv * hw * rows * (prompt + steps * (prompt + steps / 2) + positions)
    flops = 2 * rows * (layer * L * (prompt + steps) + c["vocab"] * W * (steps + 1))
    flops += 4 * L * qn * rows * (prompt * prompt / 2 + steps * (prompt + steps / 2))
    return {"bytes": weights * (2 * rows + steps - 1) + cache, "flops": flops}


def tolerance(case):
    # The device's contract: the host path's bits, in any mode but the
    # measurement ones, for every shape.
    return "exact"


# ------------------------------------------------- the same in 64 bits, in torch

def _dequantised(w, k, kind):
    """Block bytes as (values without the minimum [n, k] f64, minima [n, k / 32] f64 or None)."""
    n, bb = w.shape[0], BLOCK[KIND[kind]]
    b = w.view(n, k // 32, bb)
    half = lambda at: b[..., at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if kind == "Q8_0":
        q = b[..., 2:].contiguous().view(torch.int8).double()
    else:
        q = b[..., bb - 16:]
        q = torch.cat([q & 15, q >> 4], -1).double()
        if kind == "Q4_0":
            q = q - 8.0
    return (q * half(0)).view(n, k), half(2)[..., 0] if kind == "Q4_1" else None


def _linear(x, w, k, kind):
    """x · wᵀ with x quantised to 8 bits a block as the product's definition has it (f64 sums)."""
    rows = x.shape[0]
    v = x.float().view(rows, k // 32, 32)
    d = v.abs().amax(-1, keepdim=True) / 127.0
    y = v * torch.where(d == 0, d, 1.0 / d)
    y = torch.sign(y) * torch.floor(y.abs() + 0.5)
    values, minima = _dequantised(w, k, kind)
    out = (y.double() * d.half().double()).view(rows, k) @ values.t().contiguous()
    if minima is not None:
        sums = (y.sum(-1) * d[..., 0]).half().double()
        out = out + sums @ minima.t().contiguous()
    return out


def _rmsnorm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _attend(q, keys, values, first):
    """q [tokens, heads, width], keys and values [kv, positions, width]; query t sees positions up to first + t."""
    tokens, heads, hw = q.shape
    group = heads // keys.shape[0]
    out = torch.empty_like(q)
    seen = torch.arange(keys.shape[1], device=q.device)[None] <= first + torch.arange(tokens, device=q.device)[:, None]
    for h in range(heads):
        s = q[:, h].contiguous() @ keys[h // group].t().contiguous() / math.sqrt(hw)
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ values[h // group]
    return out


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], -1)
    return x * cos[:, None].double() + turned * sin[:, None].double()


def _attention_block(c, kind, x, norm, qkv, o, cos, sin):
    """One block over a whole prompt: (x + attention, keys, values [kv, tokens, width])."""
    W, hw, heads, kv = c["width"], c["head_width"], c["heads"], c["kv_heads"]
    p = _linear(_rmsnorm(x, norm), qkv, W, kind).view(x.shape[0], heads + 2 * kv, hw)
    q, k = _rotate(p[:, :heads], cos, sin), _rotate(p[:, heads:heads + kv], cos, sin)
    k, v = k.transpose(0, 1).contiguous(), p[:, heads + kv:].transpose(0, 1).contiguous()
    a = _attend(q, k, v, 0).reshape(x.shape[0], heads * hw)
    return x + _linear(a, o, heads * hw, kind), k, v


def _mlp_block(c, kind, x, norm, gate_up, down):
    W, H = c["width"], c["hidden"]
    g = _linear(_rmsnorm(x, norm), gate_up, W, kind)
    return x + _linear(g[:, :H] * torch.sigmoid(g[:, :H]) * g[:, H:], down, H, kind)


def exact(case, seed):
    t, what = _tensors(case, seed), case["work"]
    if what == "product":
        y = _linear(t["x"], t["w"], case["k"], case["kind"])
        return y if t["bias"] is None else y + t["bias"].double()
    if what == "plan":
        return torch.cat([_linear(x[None], w, x.numel(), case["kind"])[0] for w, x in t["items"]])
    if what == "attention":
        q, keys, values = t["q"].double(), t["keys"].double(), t["values"].double()
        if case["prompt"]:
            held = case["past"] + case["tokens"]
            return _attend(q, keys[0, :, :held], values[0, :, :held], case["past"])
        return torch.cat([_attend(q[i:i + 1], keys[i, :, :n], values[i, :, :n], n - 1)
                          for i, n in enumerate(int(n) for n in _lengths(case, seed))])
    c, kind = MODELS[case["model"]], case["kind"]
    if what == "mlp":
        return _mlp_block(c, kind, t["x"].double(), t["norm"], t["gate_up"], t["down"])
    if what == "attn_block":
        rows = case["rows"]
        cos, sin = t["cos"][:rows], t["sin"][:rows]
        y, k, v = _attention_block(c, kind, t["x"].double(), t["norm"], t["qkv"], t["o"], cos, sin)
        pad = lambda a: torch.nn.functional.pad(a, (0, 0, 0, case["capacity"] - rows))[None]  # noqa: E731
        return {"y": y, "keys": pad(k), "values": pad(v)}
    # the prompts' logits; what follows depends on the tokens chosen
    logits = []
    cos, sin = _rope_tables(case["prompt"], c["head_width"])
    for ids in _prompts(case, seed):
        at = torch.from_numpy(ids).long().cuda()
        values, minima = _dequantised(t["embed"][at], c["width"], kind)
        x = values if minima is None else values + minima.repeat_interleave(32, -1)
        for layer in range(c["layers"]):
            x, _, _ = _attention_block(c, kind, x, t["attn_norm"][layer], t["qkv"][layer], t["o"][layer],
                                       cos[:len(ids)], sin[:len(ids)])
            x = _mlp_block(c, kind, x, t["ffn_norm"][layer], t["gate_up"][layer], t["down"][layer])
        logits.append(_linear(_rmsnorm(x[-1:], t["norm"]), t["embed"], c["width"], kind))
    return {"prompt": torch.cat(logits), "tokens": None, "logits": None}
