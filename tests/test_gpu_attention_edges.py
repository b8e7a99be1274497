"""What the attention kernels' bits rest on, where ordinary prompts do not reach
it: the f32 matrix cores as chains of fused adds over special operands, the
strips' ordered sum and division over hostile values, peaked and overflowing
scores, single steps up to and past the rows the split step holds, and small
batches behind long contexts.
"""

import ctypes

import numpy as np
import pytest

import oracle as O
import rusticide_amd as R
from rusticide_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = R.Context(0)
    yield c
    c.close()


def same_bits_or_nan(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return bool(np.all((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))))


# ------------------------------------------------------------- matrix cores


def special_operands(kind, shape, rng):
    bits = rng.integers(0, 1 << 32, shape, dtype=np.uint64).astype(np.uint32)
    if kind == "normal":
        return rng.standard_normal(shape).astype(np.float32)
    if kind == "any bits":
        return bits.view(np.float32)
    if kind == "subnormal products":  # products on both sides of 2^-126, some below 2^-149
        return (rng.standard_normal(shape) * 2.0 ** rng.integers(-80, -55, shape)).astype(np.float32)
    if kind == "subnormal operands":
        sub = (bits & 0x807FFFFF).view(np.float32)
        return np.where(rng.random(shape) < 0.5, sub, (2.0 ** rng.integers(0, 20, shape)).astype(np.float32))
    if kind == "overflow":
        return (rng.standard_normal(shape) * 2.0 ** rng.integers(50, 66, shape)).astype(np.float32)
    if kind == "signed zeros":
        return rng.choice(np.float32([0.0, -0.0, 1.0, -1.0, 1e-30, -1e-30]), shape)
    if kind == "cancelling":  # each product close to the negative of a sum before it
        return (rng.choice([-1.0, 1.0], shape) * (1.0 + rng.integers(0, 8, shape) * 2.0 ** -23)).astype(np.float32)
    v = rng.standard_normal(shape).astype(np.float32)
    return np.where(rng.random(shape) < 0.02, rng.choice(np.float32([np.inf, -np.inf, np.nan]), shape), v)


@pytest.mark.parametrize("kind", ["normal", "any bits", "subnormal products", "subnormal operands", "overflow",
                                  "signed zeros", "cancelling", "infinities and NaN"])
def test_the_matrix_cores_add_products_as_a_chain_of_fused_adds(ctx, kind):
    rng = np.random.default_rng(len(kind))
    for k in (4, 8, 64, 1000, 2048):
        a, b = special_operands(kind, (16, k), rng), special_operands(kind, (k, 16), rng)
        got = np.full((16, 16), np.nan, np.float32)
        ab = np.ascontiguousarray(np.concatenate([a.reshape(-1), b.reshape(-1)]))
        ctx.check(R.lib().rh_mfma_chain_device(ctx.handle, ctypes.c_void_p(ab.ctypes.data),
                                               ctypes.c_size_t(k), ctypes.c_void_p(got.ctypes.data)))
        rows = np.ascontiguousarray(a.T).reshape(-1)  # [k][16]
        for j in range(16):
            want = O.mix_rows(np.ascontiguousarray(b[:, j]), rows, 16, 0, np.zeros(16, np.float32))
            assert same_bits_or_nan(got[:, j], want), (kind, k, j)


# ------------------------------------------------- the strips' sum and division


def half_sums(ctx, first, second):
    groups = (max(first.size, second.size) + 15) // 16
    v = np.zeros((2, 16 * groups), np.float32)
    v[0, :first.size], v[1, :second.size] = first, second
    sums, rounds = np.zeros(2, np.float32), np.zeros(2, np.uint32)
    ctx.check(R.lib().rh_ordered_sum_half_device(
        ctx.handle, ctypes.c_void_p(v.ctypes.data), ctypes.c_size_t(groups), ctypes.c_size_t(first.size),
        ctypes.c_size_t(second.size), ctypes.c_void_p(sums.ctypes.data), ctypes.c_void_p(rounds.ctypes.data)))
    return sums, rounds


def sum_cases():
    rng = np.random.default_rng(23)
    cases = [rng.exponential(1.0, n).astype(np.float32)
             for n in (1, 2, 15, 16, 17, 31, 33, 496, 512, 513, 1000, 1024, 1025, 2000, 2481, 2495, 2496)]
    for _ in range(24):
        n = int(rng.integers(1, 2497))
        cases.append(np.exp(-rng.exponential(30.0, n)).astype(np.float32))  # exps of spread scores
        cases.append((rng.random(n) * np.exp(rng.uniform(-60, 30, n))).astype(np.float32))
        peaked = np.zeros(n, np.float32)
        peaked[rng.integers(0, n, 3)] = 1.0
        cases.append(peaked)
    n = 2048
    cases.append(np.zeros(n, np.float32))
    cases.append(np.float32(2.0 ** -24) * rng.integers(0, 4, n).astype(np.float32) + np.float32(1.0))
    cases.append(rng.integers(1, 1 << 23, n, dtype=np.uint32).view(np.float32))  # subnormals
    cases.append(np.full(n, 3e37, np.float32))  # to infinity
    cases.append(np.full(2496, np.float32(1.0) / np.float32(3.0)))
    with_nan = rng.exponential(1.0, n).astype(np.float32)
    with_nan[1500] = np.nan
    cases.append(with_nan)
    # every value half an ulp of the running sum it meets: each add rounds
    cases.append(np.concatenate([np.float32([1.0]), np.full(2400, 2.0 ** -24, np.float32) * np.float32(1.5)]))
    # tiny first runs, each next run dwarfing all before
    cases.append((2.0 ** (np.arange(2400) // 80 * 3.0 - 60) * rng.random(2400)).astype(np.float32))
    return cases


def fold(values):
    with np.errstate(all="ignore"):
        return np.add.accumulate(np.concatenate([np.zeros(1, np.float32), values]), dtype=np.float32)[-1]


def test_the_strips_ordered_sum_is_the_sequential_fold(ctx):
    cases = sum_cases()
    most = 0
    for i, first in enumerate(cases):
        # the two rows of a wave differ in length and in the rounds they take
        for second in (cases[(i + 1) % len(cases)], cases[(7 * i + 3) % len(cases)]):
            sums, rounds = half_sums(ctx, first, second)
            for got, values in zip(sums, (first, second)):
                assert same_bits_or_nan([got], [fold(values)]), (i, values.size, got, fold(values), rounds)
            most = max(most, int(rounds.max()))
    assert most == 7, most  # 7: the closing sequential chain ran too


@pytest.mark.parametrize("d", [1.0, 1.5, 3.0, 1.0 + 2.0 ** -23, 2.0 - 2.0 ** -23, 7.3, 255.99998, 2496.0,
                               float(np.sqrt(np.float32(128.0)))])
def test_division_by_one_divisor_is_the_ieee_quotient(ctx, d):
    d = np.float32(d)
    rng = np.random.default_rng(31)
    mant = rng.integers(0, 1 << 23, 200000, dtype=np.uint32)
    expo = np.concatenate([rng.integers(0, 255, 100000), rng.integers(0, 16, 100000)]).astype(np.uint32)
    sign = rng.integers(0, 2, 200000, dtype=np.uint32)
    x = [((sign << 31) | (expo << 23) | mant).view(np.float32)]
    # quotients at and beside the ends of the subnormal range and its midpoints
    for q in (2.0 ** -126, 2.0 ** -126 - 2.0 ** -150, 2.0 ** -127, 2.0 ** -149, 2.0 ** -150, 3 * 2.0 ** -150):
        c = np.float32(q * float(d)).view(np.uint32).astype(np.int64) + np.arange(-64, 65)
        c = c[c >= 0].astype(np.uint32).view(np.float32)
        x += [c, -c]
    x.append(np.float32([0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, 3.4028235e38]))
    x = np.concatenate(x)
    x = np.ascontiguousarray(np.concatenate([x, np.ones(-x.size % 4, np.float32)]))
    y = np.empty_like(x)
    ctx.check(R.lib().rh_div_by_device(ctx.handle, ctypes.c_void_p(x.ctypes.data), ctypes.c_size_t(x.size),
                                       ctypes.c_float(d), ctypes.c_void_p(y.ctypes.data)))
    with np.errstate(all="ignore"):
        want = x / d
    assert np.sum((want != 0) & (np.abs(want) < 2.0 ** -126)) > 1000  # subnormal quotients are among them
    assert same_bits_or_nan(y, want)


# ------------------------------------------------------------------ decoders


def config(heads, kv_heads, head_dim, context, blocks=1):
    return dict(embedding_length=heads * head_dim, block_count=blocks, feed_forward_length=512, head_count=heads,
                head_count_kv=kv_heads, head_dim=head_dim, context_length=context, vocab_size=128,
                rope_freq_base=10000.0, rms_norm_eps=1e-5)


def check(ctx, model, chunks, seed):
    c = model["config"]
    gpu, cpu = R.Decoder(ctx, model), O.Decoder(model, threads=8)
    ids = np.random.default_rng(seed).integers(0, c["vocab_size"], sum(chunks)).astype(np.uint32)
    start, logits = 0, []
    for n in chunks:
        g = np.asarray(gpu.forward_batch(ids[start:start + n], start), np.float32)
        w = np.asarray(cpu.forward_batch(ids[start:start + n], start), np.float32)
        assert same_bits_or_nan(g, w), f"{n} tokens at {start}: max |diff| {np.max(np.abs(g.astype(np.float64) - w))}"
        start += n
        logits.append(w)
    gpu.close()
    cpu.close()
    return ids, logits


# single steps over the split step's second and third pass over the rows
# (2048, 4096), the late value pieces, and its last row, 4488, to the kernels
# that follow it
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(4, 1, 64), (2, 1, 128)])
def test_steps_to_the_split_steps_last_row(ctx, heads, kv_heads, head_dim):
    model = synth.decoder_model(config(heads, kv_heads, head_dim, 4500), head_dim)
    chunks = [2044] + [1] * 8 + [248, 1, 1, 1, 1792] + [1] * 4 + [387] + [1] * 6
    check(ctx, model, chunks, 5)
    assert sum(chunks) == 4492


# few tokens behind a context long enough for strips: eight, four, sixteen and
# one heads a kv head, heads of 128, and tiles of more workgroups than an XCD has CUs
@pytest.mark.parametrize("heads,kv_heads,head_dim,chunks", [
    (8, 1, 64, [230, 2, 3, 8, 5]), (8, 2, 64, [640, 2, 7, 8, 3]), (16, 1, 64, [820, 2, 5, 8]),
    (4, 4, 64, [900, 2, 5, 8, 13]), (4, 1, 128, [150, 2, 3, 8]), (4, 4, 128, [150, 2, 3, 8]),
    (36, 12, 64, [30, 17, 12])])
def test_few_tokens_behind_a_long_context(ctx, heads, kv_heads, head_dim, chunks):
    check(ctx, synth.decoder_model(config(heads, kv_heads, head_dim, 1000, 2), heads), chunks, 9)


def f16_scaled(matrix, factor, offsets):
    """The matrix with the f16 scales at `offsets` of each 144-byte block times factor."""
    t, data, rows, cols = matrix
    blocks = np.array(data, np.uint8).reshape(-1, 144)
    for o in offsets:
        d = np.ascontiguousarray(blocks[:, o:o + 2]).view(np.float16).astype(np.float32) * np.float32(factor)
        blocks[:, o:o + 2] = d.astype(np.float16).view(np.uint8).reshape(-1, 2)
    return t, blocks.reshape(-1), rows, cols


def scores(model, ids):
    """The first block's scores [head][token][row], in double from unquantized
    activations: what the float path forms, to a few parts in a hundred."""
    c, b = model["config"], model["blocks"][0]
    hd, n = c["head_dim"], len(ids)

    def rows(m):
        t, data, r, _ = m
        return np.stack([O.dequantize_row(t, row) for row in np.asarray(data).reshape(r, -1)]).astype(np.float64)

    cos, sin = (a.reshape(n, 1, hd // 2).astype(np.float64) for a in O.rope_table(n, hd, c["rope_freq_base"]))

    def rope(x):
        x = x.reshape(n, -1, hd // 2, 2)
        lo, hi = x[..., 0], x[..., 1]
        return np.stack([lo * cos - hi * sin, hi * cos + lo * sin], -1).reshape(n, -1, hd)

    h = rows(model["token_embd"])[ids]
    x = h / np.sqrt((h * h).mean(1, keepdims=True) + c["rms_norm_eps"]) * b["attn_norm"]
    q, k = rope(x @ rows(b["attn_q"]).T), rope(x @ rows(b["attn_k"]).T)
    group = c["head_count"] // c["head_count_kv"]
    return np.stack([q[:, j] @ k[:, j // group].T for j in range(c["head_count"])]) / np.sqrt(hd)


# scores that spread past the exponential's cutoff (exp 0 below -103.97) over
# its subnormal results (below -87.3), as peaked attention has them: batches
# and single steps of each kernel
@pytest.mark.parametrize("heads,kv_heads,head_dim,chunks", [
    (8, 2, 64, [300, 64, 1, 1, 9, 1]), (4, 4, 64, [200, 1, 90, 1, 1]), (4, 1, 128, [180, 1, 40, 1, 2, 1]),
    (8, 1, 64, [40, 1, 230, 8, 1])])
def test_peaked_scores(ctx, heads, kv_heads, head_dim, chunks):
    model = synth.decoder_model(config(heads, kv_heads, head_dim, 400, 2), heads)
    for b in model["blocks"]:
        b["attn_norm"] = (b["attn_norm"] * np.float32(15.0)).astype(np.float32)
        b["attn_v"] = f16_scaled(b["attn_v"], 1 / 15.0, (0, 2))
    ids, _ = check(ctx, model, chunks, 13)
    s = scores(model, ids)[:, -1]
    below = s.max(1, keepdims=True) - s
    assert np.any(below > 104) and np.any((below > 88) & (below < 103)) and np.sum(below < 80) > len(s)


# scores that overflow: minus infinity, a weight of 0 in a row that goes on,
# and plus infinity, a row of NaN
@pytest.mark.parametrize("heads,kv_heads,head_dim,scale", [(4, 1, 64, 1e19), (4, 4, 64, 1e19), (2, 1, 128, 0.9e19)])
def test_overflowing_scores(ctx, heads, kv_heads, head_dim, scale):
    model = synth.decoder_model(config(heads, kv_heads, head_dim, 400), heads)
    b = model["blocks"][0]
    b["attn_norm"] = (b["attn_norm"] * np.float32(scale)).astype(np.float32)
    # brought back down, so that what follows attention stays finite
    b["attn_v"] = f16_scaled(b["attn_v"], 2.0 ** -9, (0, 2))
    b["attn_output"] = f16_scaled(b["attn_output"], 2.0 ** -9, (0, 2))
    chunks = [260, 1, 1, 1, 30, 1, 9, 1, 1, 1]
    ids, _ = check(ctx, model, chunks, 17)
    dots = scores(model, ids) * np.sqrt(head_dim)  # overflow comes before the division
    up = down = 0
    for end in np.cumsum(chunks):
        last = dots[:, end - 1, :end]
        up += np.sum((last > 3.6e38).any(1))
        down += np.sum((last < -3.6e38).any(1) & ~(last > 3.2e38).any(1))
    assert up > 0 and down > 0, (up, down)
