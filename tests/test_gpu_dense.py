"""Dense f32 rows, by the tiled kernel and by the one for short rows, wide
activations and rows at a 4-byte stride, against the CPU path's eight-lane
dot, bit for bit: rows around a workgroup's 16 and 64, widths around the
chunks in flight, ragged widths, several tokens and matrices.
"""

import ctypes

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
    check(rows, cols, tokens)


# the tiled kernel at its edges: rows around a wave's 16 and a workgroup's 64
# (grids of one and of four waves a workgroup), rows that end inside a tile of
# 256 values or a chunk of eight, the widest activation, several matrices
@pytest.mark.parametrize("rows,cols,tokens", [
    ((1,), 1024, 1), ((15,), 1028, 1), ((17, 64), 1032, 1), ((65, 1, 16), 1276, 1), ((16385,), 384, 1),
    ((16448, 40), 396, 1), ((130,), 768, 1), ((63,), 88, 3), ((33,), 2052, 4), ((20,), 2048, 8), ((9,), 16384, 1),
    ((5, 3), 8188, 2)])
def test_tiled_dense_rows(rows, cols, tokens):
    L = R.lib()
    L.rh_dense_route_host.argtypes = [ctypes.c_size_t] * 3
    assert cols % 4 == 0 and L.rh_dense_route_host(sum(rows), cols, tokens)
    check(rows, cols, tokens)


def check(rows, cols, tokens):
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
