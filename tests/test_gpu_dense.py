"""Dense f32 rows, four lanes a row, against the CPU path's eight-lane dot,
bit for bit: rows around a workgroup's 16 and 64, widths around the chunks in
flight, ragged widths, rows at a 4-byte stride, several tokens and matrices.
"""

import numpy as np
import pytest

import oracle as O
import rusticide_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,tokens", [
    ((1,), 8, 1), ((15,), 126, 1), ((17, 64), 128, 1), ((63,), 136, 3), ((65, 1, 16), 248, 1), ((130,), 256, 2),
    ((16385,), 264, 1), ((16448, 40), 390, 1), ((40,), 2048, 8), ((33,), 2054, 4), ((20,), 129, 1), ((9,), 16390, 1),
    ((9,), 8192, 4)])
def test_dense_rows(rows, cols, tokens):
    ctx = R.Context(0)
    rng = np.random.default_rng(cols + tokens)
    x = rng.standard_normal(cols * tokens).astype(np.float32)
    ws = [rng.standard_normal(r * cols).astype(np.float32) for r in rows]
    mats = [R.Matrix.load(ctx, R.F32, w, r, cols) for w, r in zip(ws, rows)]
    outs = [np.full(r * tokens, np.nan, np.float32) for r in rows]
    R.matmul_batch(ctx, x, tokens, list(zip(mats, outs)))
    for w, r, out in zip(ws, rows, outs):
        want = np.full(r * tokens, np.nan, np.float32)
        O.matmul_batch(x, tokens, [(O.Weights.dense(w, cols), want)])
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
    for m in mats:
        m.free()
    ctx.close()
