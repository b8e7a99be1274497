"""Performance cases: what a program that runs a quantized llama-family model
on this package has it do, through the package's public entry points.

Two paths are covered.

* "product": ``matmul_batch_device`` on device-resident activations, one call
  per pass, for each weight format (Q4_K, Q6_K, I2_S, F16 widened at load),
  from the one token of a decode step over small batches to prompts of 2048
  tokens, ragged counts included. Several matrices sharing one activation
  (Q/K/V, gate and up) go in one call, as the decoder calls them.
* "decoder": ``Decoder`` over a few layers of the package's TinyLlama-shaped
  configuration (``synth.TINYLLAMA``), or of the same width with wider heads:
  prompts of 2 to 2048 tokens fed whole or in chunks, then decode steps, each
  returning its logits; and greedy generation followed by one more forward.

The package's contract is that every product and every logit has the bits of
the CPU path (quantized activations, integer dots, float sums in the CPU's
order), so the tolerance is "exact" throughout. ``exact`` gives the same
quantities in 64 bits: products of the dequantized weights and the quantized
activations, and the decoder's forward with every float step in double.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import rusticide_amd as R
from rusticide_amd import synth

TYPES = {"Q4_K": R.Q4_K, "Q6_K": R.Q6_K, "I2_S": R.I2_S, "F16": R.F16}
WEIGHT_BYTES = {"Q4_K": 144 / 256, "Q6_K": 210 / 256, "I2_S": 0.25, "F16": 4.0}  # F16 rows are held as f32
TERNARY_SCALE = 0.02

_context = None


def context() -> R.Context:
    """One context per process, as a program keeps it."""
    global _context
    if _context is None:
        _context = R.Context(0)
    return _context


# ---------------------------------------------------------------------- cases


def product(name, kind, rows, cols, tokens):
    return {"name": name, "path": "product", "type": kind, "rows": rows, "cols": cols, "tokens": tokens}


def decoder(name, layers, head_dim, kv_heads, prompt, chunk, steps, generate=False):
    return {"name": name, "path": "decoder", "layers": layers, "head_dim": head_dim, "kv_heads": kv_heads,
            "prompt": prompt, "chunk": chunk, "steps": steps, "generate": generate}


def listed():
    return [
        # a decode step's Q/K/V projections: the smallest call
        product("qkv_token", "Q4_K", "2048+256+256", 2048, 1),
        # a decode step's output matrix, the largest matrix read per token
        product("output_token", "Q6_K", "32000", 2048, 1),
        # a ternary model's down projection in a decode step
        product("ternary_token", "I2_S", "2560", 6912, 1),
        # an unquantized output matrix (tied F16 embeddings) in a decode step
        product("dense_token", "F16", "32000", 2048, 1),
        # gate and up for a small batch of sequences decoded together
        product("gate_up_5", "Q4_K", "5632+5632", 2048, 5),
        # the down projection of a ragged prompt
        product("down_509", "Q6_K", "2048", 5632, 509),
        # gate and up of a long prompt, the largest product
        product("gate_up_2048", "Q4_K", "5632+5632", 2048, 2048),
        # a ternary model's up projection over a prompt
        product("ternary_1000", "I2_S", "6912", 2560, 1000),
        # a short chat turn through generate_greedy: prefill in its chunks of
        # 64, then the device-resident decode loop
        decoder("generate_short", 3, 64, 4, 100, 0, 40, generate=True),
        # a long prompt in one batch
        decoder("prompt_2000", 2, 64, 4, 2000, 2000, 0),
        # decoding behind a long context, the prompt fed in chunks
        decoder("decode_long", 2, 64, 4, 1777, 512, 40),
        # heads of 128 values, as most larger llama models have
        decoder("heads_128", 2, 128, 4, 700, 700, 24),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.6:
        kind = rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q6_K", "I2_S", "F16"])
        block = {"I2_S": 128, "F16": 1}.get(kind, 256)
        cols = max(block, _log_uniform(rng, 1024, 8192) // block * block)
        tokens = 1 if rng.random() < 0.3 else _log_uniform(rng, 2, 2048)
        if kind == "F16":
            # unquantized matrices are small or read by few tokens
            tokens = 1 if tokens > 8 else tokens
        # no more weights x tokens than the largest listed product
        most = min(32000.0, 2.0 * 5632 * 2048 * 2048 / (cols * tokens), 65e6 / cols)
        rows = max(64, min(int(most), _log_uniform(rng, 256, 32000)))
        if rng.random() < 0.4:
            part = max(32, rows // rng.choice([3, 4, 8]))
            rows = "%d+%d+%d" % (rows, part, part) if rows + 2 * part <= most else str(rows)
        return {"path": "product", "type": kind, "rows": str(rows), "cols": cols, "tokens": tokens}
    head_dim = rng.choice([64, 64, 64, 128])
    kv_heads = rng.choice([4, 8]) if head_dim == 64 else rng.choice([4, 16])
    generate = rng.random() < 0.3
    prompt = _log_uniform(rng, 2, 512 if generate or head_dim == 128 else 2048)
    chunk = 0 if generate else rng.choice([prompt, 64, 512, 200])
    return {"path": "decoder", "layers": rng.choice([1, 2]), "head_dim": head_dim, "kv_heads": kv_heads,
            "prompt": prompt, "chunk": min(chunk, prompt), "steps": rng.randint(0 if not generate else 1, 40),
            "generate": generate}


def _row_counts(case):
    return [int(r) for r in case["rows"].split("+")]


def _config(case):
    c = dict(synth.TINYLLAMA)
    c["block_count"] = case["layers"]
    c["head_dim"] = case["head_dim"]
    c["head_count"] = c["embedding_length"] // case["head_dim"]
    c["head_count_kv"] = case["kv_heads"]
    c["context_length"] = 3200 if case["prompt"] + case["steps"] >= 2047 else 2048
    return c


# ------------------------------------------------------------------- one pass


def _product_data(case, seed):
    """Host bytes of each matrix and the f32 activations [tokens, cols]."""
    rng = np.random.Generator(np.random.PCG64([seed, 17]))
    mats = []
    for i, rows in enumerate(_row_counts(case)):
        s = int(rng.integers(0, 2 ** 31))
        cols = case["cols"]
        if case["type"] == "Q4_K":
            data = synth.q4k_centered(rows, cols, s)
        elif case["type"] == "Q6_K":
            data = synth.q6k_centered(rows, cols, s)
        elif case["type"] == "I2_S":
            # byte-wise: two bits a weight, codes 0..2 (weight + 1)
            g = np.random.Generator(np.random.PCG64(s))
            c = g.integers(0, 3, size=(4, rows * cols // 4), dtype=np.uint8)
            packed = (c[0] << 6) | (c[1] << 4) | (c[2] << 2) | c[3]
            trailer = np.zeros(32, np.uint8)
            trailer[:4] = np.array([TERNARY_SCALE], np.float32).view(np.uint8)
            data = np.concatenate([packed, trailer])
        else:
            g = np.random.Generator(np.random.PCG64(s))
            data = (g.standard_normal(rows * cols, dtype=np.float32) * 0.02).astype(np.float16).view(np.uint8)
        mats.append(data)
    x = rng.standard_normal((case["tokens"], case["cols"]), dtype=np.float32)
    return mats, x


def _decoder_data(case, seed):
    model = synth.decoder_model(_config(case), seed)
    rng = np.random.Generator(np.random.PCG64([seed, 29]))
    ids = rng.integers(0, model["config"]["vocab_size"], case["prompt"] + max(1, case["steps"])).astype(np.uint32)
    return model, ids


def prepare(case, seed):
    ctx = context()
    if case["path"] == "product":
        mats, x = _product_data(case, seed)
        rows, cols = _row_counts(case), case["cols"]
        loaded = [R.Matrix.load(ctx, TYPES[case["type"]], m, r, cols) for m, r in zip(mats, rows)]
        outs = [torch.zeros(r * case["tokens"], dtype=torch.float32, device="cuda") for r in rows]
        xd = torch.from_numpy(x).cuda()
        torch.cuda.synchronize()
        return {"case": dict(case), "ctx": ctx, "x": xd, "jobs": list(zip(loaded, outs))}
    model, ids = _decoder_data(case, seed)
    return {"case": dict(case), "ctx": ctx, "decoder": R.Decoder(ctx, model), "ids": ids}


def run(state):
    case = state["case"]
    if case["path"] == "product":
        R.matmul_batch_device(state["ctx"], state["x"], case["tokens"], state["jobs"])
        return [out for _, out in state["jobs"]]
    d, ids, n = state["decoder"], state["ids"], case["prompt"]
    if case["generate"]:
        tokens = d.generate_greedy(ids[:n], case["steps"])
        return {"tokens": tokens, "logits": d.forward(int(ids[n]), d.position)}
    d.reset()
    logits = []
    for start in range(0, n, case["chunk"]):
        logits.append(d.forward_batch(ids[start: min(n, start + case["chunk"])], start))
    logits = logits[-1:]  # the prompt's last logits, as a program keeps them
    for i in range(case["steps"]):
        logits.append(d.forward(int(ids[n + i]), n + i))
    return logits


# -------------------------------------------------- what a pass cannot do without


def work(case):
    if case["path"] == "product":
        rows, cols, tokens = sum(_row_counts(case)), case["cols"], case["tokens"]
        return {"bytes": rows * cols * WEIGHT_BYTES[case["type"]] + 4.0 * tokens * (cols + rows),
                "flops": 2.0 * rows * cols * tokens}
    c = _config(case)
    w, f, vocab = c["embedding_length"], c["feed_forward_length"], c["vocab_size"]
    kv = c["head_count_kv"] * c["head_dim"]
    weights = c["block_count"] * (2 * w * w + 2 * w * kv + 3 * w * f)
    down = c["block_count"] * w * f
    read = (weights - down) * 144 / 256 + down * (144 / 256 * (c["block_count"] // 2)
                                                  + 210 / 256 * ((c["block_count"] + 1) // 2)) / c["block_count"]
    head = vocab * w
    n, steps = case["prompt"], case["steps"] + (1 if case["generate"] else 0)
    chunk = 64 if case["generate"] else case["chunk"]
    chunks = -(-n // chunk)
    pairs = n * (n + 1) / 2 + sum(n + i + 1 for i in range(steps))  # (token, cached row) pairs
    kv_rows = sum(min(n, (i + 1) * chunk) for i in range(chunks)) + sum(n + i + 1 for i in range(steps))
    layers = c["block_count"]
    return {
        "bytes": (chunks + steps) * read + (chunks + steps) * (head * 210 / 256 + 4 * vocab) + layers * kv_rows * 8.0 * kv,
        "flops": 2.0 * weights * (n + steps) + 2.0 * head * (chunks + steps) + layers * pairs * 4.0 * w,
    }


def tolerance(case):
    return "exact"


# --------------------------------------------------------------- in 64 bits


def _f16(b):
    return torch.from_numpy(np.ascontiguousarray(b).view(np.float16).astype(np.float64)).cuda()


def _dequantize(kind, data, rows, cols):
    """[rows, cols] in double, on the GPU."""
    if kind == "F16":
        return torch.from_numpy(data.view(np.float16).reshape(rows, cols)).cuda().double()
    if kind == "I2_S":
        b = torch.from_numpy(data[: rows * cols // 4].reshape(rows, cols // 128, 1, 32)).cuda()
        shifts = torch.tensor([6, 4, 2, 0], dtype=torch.uint8, device="cuda").reshape(1, 1, 4, 1)
        scale = float(np.float32(TERNARY_SCALE))
        return (((b >> shifts) & 3).double() - 1.0).reshape(rows, cols) * scale
    n = rows * cols // 256
    if kind == "Q4_K":
        host = data.reshape(n, 144)
        d, dmin = _f16(host[:, 0:2]).reshape(n, 1, 1), _f16(host[:, 2:4]).reshape(n, 1, 1)
        s = torch.from_numpy(np.ascontiguousarray(host[:, 4:16])).cuda().int()
        lo, hi, last = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([lo & 63, (last & 15) | ((lo >> 6) << 4)], 1).double().reshape(n, 8, 1)
        mn = torch.cat([hi & 63, (last >> 4) | ((hi >> 6) << 4)], 1).double().reshape(n, 8, 1)
        q = torch.from_numpy(np.ascontiguousarray(host[:, 16:])).cuda().reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32).double()
        return (d * sc * q - dmin * mn).reshape(rows, cols)
    host = data.reshape(n, 210)
    ql = torch.from_numpy(np.ascontiguousarray(host[:, :128])).cuda().int().reshape(n, 2, 2, 32)
    qh = torch.from_numpy(np.ascontiguousarray(host[:, 128:192])).cuda().int().reshape(n, 2, 1, 32)
    sc = torch.from_numpy(np.ascontiguousarray(host[:, 192:208]).view(np.int8)).cuda().double().reshape(n, 2, 4, 2, 1)
    d = _f16(host[:, 208:210]).reshape(n, 1, 1, 1, 1)
    low = torch.cat([ql & 15, ql >> 4], 2)
    shifts = torch.tensor([0, 2, 4, 6], dtype=torch.int32, device="cuda").reshape(1, 1, 4, 1)
    q = (low | (((qh >> shifts) & 3) << 4)).double() - 32.0
    return (d * sc * q.reshape(n, 2, 4, 2, 16)).reshape(rows, cols)


def _quantized(x, kind):
    """The activation the integer products see: quants times their scale, the
    quantization itself in the dtype of x (f32 as the formats define it)."""
    if kind == "F16":
        return x.double()
    t, cols = x.shape
    if kind == "I2_S":  # one divisor a row, 127 / max |x| with the maximum from 1e-5
        top = x.abs().amax(1, keepdim=True).double().clamp_min(1e-5)
        div = (127.0 / top).to(x.dtype)
        return torch.round(x * div).clamp(-128, 127).double() / div.double()
    b = x.reshape(t, cols // 256, 256)
    at = b.abs().argmax(2, keepdim=True)  # ties of opposite sign differ only in the quants' sign
    top = torch.gather(b, 2, at)
    inv = torch.where(top == 0, torch.zeros_like(top), torch.full_like(top, -127.0) / top)
    step = torch.where(top == 0, torch.zeros_like(top), torch.ones_like(top) / inv)
    return (torch.round(b * inv).clamp(-127, 127).double() * step.double()).reshape(t, cols)


def _exact_decoder(case, seed):
    model, ids = _decoder_data(case, seed)
    c = model["config"]
    hd, heads, kvh = c["head_dim"], c["head_count"], c["head_count_kv"]
    group, eps = heads // kvh, float(np.float32(c["rms_norm_eps"]))
    names = {v: k for k, v in TYPES.items()}
    n = case["prompt"] + case["steps"]
    ids = torch.from_numpy(ids[:n].astype(np.int64))

    def mm(x, m):
        kind = names[m[0]]
        return _quantized(x, kind) @ _dequantize(kind, m[1], m[2], m[3]).T

    def norm(x, weight):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * torch.from_numpy(weight).cuda().double()

    pos = np.arange(n, dtype=np.float32)[:, None]
    expo = -np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd)
    angle = torch.from_numpy(pos * np.power(np.float32(c["rope_freq_base"]), expo)[None, :]).cuda().double()
    cos, sin = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]

    def rope(x, count):
        x = x.reshape(n, count, hd // 2, 2)
        a, b = x[..., 0], x[..., 1]
        return torch.stack([a * cos - b * sin, b * cos + a * sin], -1).reshape(n, count, hd)

    t, data, rows, cols = model["token_embd"]
    h = _dequantize(names[t], data, rows, cols)[ids.cuda()]
    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
    for b in model["blocks"]:
        x = norm(h, b["attn_norm"])
        q, k = rope(mm(x, b["attn_q"]), heads), rope(mm(x, b["attn_k"]), kvh)
        v = mm(x, b["attn_v"]).reshape(n, kvh, hd)
        mixed = torch.empty(n, heads, hd, dtype=torch.float64, device="cuda")
        for j in range(heads):
            s = (q[:, j] @ k[:, j // group].T / math.sqrt(hd)).masked_fill(mask, -math.inf)
            mixed[:, j] = torch.softmax(s, 1) @ v[:, j // group]
        h = h + mm(mixed.reshape(n, heads * hd), b["attn_output"])
        x = norm(h, b["ffn_norm"])
        gate = mm(x, b["ffn_gate"])
        h = h + mm(gate / (1.0 + torch.exp(-gate)) * mm(x, b["ffn_up"]), b["ffn_down"])
    x = norm(h[case["prompt"] - 1:], model["output_norm"])
    return list(mm(x, model["output"]).cpu().numpy())


def exact(case, seed):
    if case["path"] == "product":
        mats, x = _product_data(case, seed)
        a = _quantized(torch.from_numpy(x), case["type"]).cuda()
        return [(_dequantize(case["type"], m, r, case["cols"]) @ a.T).reshape(-1)
                for m, r in zip(mats, _row_counts(case))]
    if case["generate"]:
        return None  # the picks depend on the last bits of near ties
    return _exact_decoder(case, seed)
