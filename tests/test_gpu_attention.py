"""The prompt attention on the matrix cores against the CPU path, bit for bit.

Every prompt is followed by a second block, so each token's attention output
reaches the logits compared: through the second block's keys and values, and
the last token's through its own row.
"""

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


def config(heads, kv_heads, head_dim, context):
    return dict(embedding_length=heads * head_dim, block_count=2, feed_forward_length=512, head_count=heads,
                head_count_kv=kv_heads, head_dim=head_dim, context_length=context, vocab_size=128,
                rope_freq_base=10000.0, rms_norm_eps=1e-5)


def check(ctx, c, chunks, seed):
    model = synth.decoder_model(c, seed)
    gpu, cpu = R.Decoder(ctx, model), O.Decoder(model, threads=8)
    ids = np.random.default_rng(seed).integers(0, c["vocab_size"], sum(chunks)).astype(np.uint32)
    start = 0
    for n in chunks:
        g = np.asarray(gpu.forward_batch(ids[start:start + n], start), np.float32)
        w = np.asarray(cpu.forward_batch(ids[start:start + n], start), np.float32)
        assert np.array_equal(g.view(np.uint32), w.view(np.uint32)), \
            f"{n} tokens at {start}: max |diff| {np.max(np.abs(g.astype(np.float64) - w))}"
        start += n
    gpu.close()
    cpu.close()


# query heads a kv head: 8, 4, 2, 1 (strips of that many heads) and 3 (one
# head a strip); chunk ends on and around multiples of 16 rows
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(8, 1, 64), (8, 2, 64), (4, 2, 64), (4, 4, 64), (12, 4, 64),
                                                     (4, 1, 128), (2, 2, 128), (6, 2, 128)])
def test_prompt_chunks(ctx, heads, kv_heads, head_dim):
    c = config(heads, kv_heads, head_dim, 400)
    check(ctx, c, [2, 13, 1, 16, 31, 9, 64, 113, 150], heads + head_dim)


# the longest strips a workgroup's LDS holds, launches cut by strip length,
# and a chunk past them
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(8, 1, 64), (4, 1, 128)])
def test_long_prompt(ctx, heads, kv_heads, head_dim):
    check(ctx, config(heads, kv_heads, head_dim, 2600), [2400, 90, 37, 40], 5)


# single tokens behind a prompt, at and around whole tiles of 128 and 256 rows
@pytest.mark.parametrize("heads,kv_heads,head_dim", [(8, 1, 64), (12, 4, 64), (4, 1, 128), (8, 8, 128)])
@pytest.mark.parametrize("prompt", [126, 222, 254, 510, 1000])
def test_steps_behind_a_prompt(ctx, heads, kv_heads, head_dim, prompt):
    check(ctx, config(heads, kv_heads, head_dim, 1100), [prompt, 1, 1, 1, 1], prompt)
