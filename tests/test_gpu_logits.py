"""A forward's logits through page-locked memory: any length the caller asks
for, a vocabulary that is no multiple of four, batches and single tokens, and
nothing written past the length.
"""

import numpy as np
import pytest

import oracle as O
import rusticide_amd as R
from rusticide_amd import synth

pytestmark = pytest.mark.gpu

CONFIG = dict(embedding_length=256, block_count=1, feed_forward_length=512, head_count=4, head_count_kv=2, head_dim=64,
              context_length=32, vocab_size=1031, rope_freq_base=10000.0, rms_norm_eps=1e-5)


@pytest.mark.parametrize("length", [0, 1, 3, 4, 1023, 1025, 1030, 1031, 1040])
def test_logits_lengths(length):
    ctx = R.Context(0)
    model = synth.decoder_model(CONFIG, 3)
    gpu, cpu = R.Decoder(ctx, model), O.Decoder(model, threads=4)
    ids = np.array([5, 1030, 17, 9], np.uint32)
    start = 0
    for n in (2, 1, 1):
        want = np.asarray(cpu.forward_batch(ids[start:start + n], start), np.float32)
        got = np.full(1100, -7.25, np.float32)
        chunk = np.ascontiguousarray(ids[start:start + n])
        ctx.check(R._dec_lib().rh_decoder_forward_batch(gpu.handle, chunk.ctypes.data, n, start, got.ctypes.data, length))
        m = min(length, CONFIG["vocab_size"])
        assert np.array_equal(got[:m].view(np.uint32), want[:m].view(np.uint32))
        assert np.all(got[m:] == np.float32(-7.25))
        start += n
    gpu.close()
    cpu.close()
    ctx.close()
