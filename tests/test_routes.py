"""Which kernel a call takes, and where a launch's workgroups go: the host-side
rules, checked without a GPU. (That every route gives the CPU path's bits is
the GPU tests' part.)
"""

import ctypes

import pytest

import rusticide_amd as R


def strip_places(tiles, hx):
    L = R.lib()
    L.rh_strip_place_host.restype = ctypes.c_uint32
    tile, heads = ctypes.c_uint32(), ctypes.c_uint32()
    grid, places = 1, []
    b = 0
    while b < grid:
        grid = L.rh_strip_place_host(b, tiles, hx, ctypes.byref(tile), ctypes.byref(heads))
        places.append((tile.value, heads.value))
        b += 1
    return places


@pytest.mark.parametrize("hx", [1, 2, 3, 8, 31, 32, 40])
@pytest.mark.parametrize("tiles", [1, 2, 3, 7, 8, 9, 16, 63])
def test_strips_cover_every_tile_and_never_crowd_one_xcd(tiles, hx):
    places = strip_places(tiles, hx)
    work = [(b, p) for b, p in enumerate(places) if p[0] < tiles]
    assert sorted(p for _, p in work) == [(t, h) for t in range(tiles) for h in range(hx)]
    # workgroup b runs on XCD b % 8
    load = [0] * 8
    for b, _ in work:
        load[b % 8] += 1
    assert max(load) - min(load) <= (1 if tiles < 8 and hx >= 32 else hx), load


# us a layer of the strips less the kernels they replaced, beside each shape:
# (head_dim, heads, kv_heads, rows, tokens, grouped, quantized, token-major)
SLOWER = [
    (64, 32, 8, 246, 8, 1, 1, 0),     # +2.1
    (64, 32, 8, 524, 4, 1, 1, 0),     # +1.6
    (64, 32, 8, 269, 9, 1, 1, 1),     # +2.1
    (64, 32, 16, 2, 2, 0, 1, 0),      # +4.6
    (64, 32, 16, 1010, 8, 0, 1, 0),   # +2.5
    (64, 32, 32, 400, 2, 0, 1, 0),    # +4.5
    (64, 32, 32, 1230, 8, 0, 1, 0),   # +2.6
    (64, 40, 8, 604, 2, 0, 1, 0),     # +3.8
    (64, 8, 4, 408, 8, 0, 0, 0),      # +2.1
    (64, 32, 32, 140, 16, 0, 0, 0),   # +3.3
    (64, 32, 16, 48, 24, 0, 0, 0),    # +4.9
    (128, 16, 4, 2, 2, 0, 1, 0),      # +3.5
    (128, 16, 16, 128, 8, 0, 1, 0),   # +0.8
    (128, 8, 1, 32, 16, 0, 0, 0),     # +5.2
]
FASTER = [
    (64, 32, 4, 320, 2, 1, 1, 0),     # -5.9
    (64, 32, 8, 1010, 2, 1, 1, 0),    # -8.6
    (64, 32, 8, 404, 24, 1, 1, 1),    # -6.2
    (64, 32, 16, 1710, 2, 0, 1, 0),   # -1.6
    (64, 32, 2, 1210, 4, 0, 1, 0),    # -2.3
    (64, 32, 16, 9, 9, 0, 1, 1),      # -0.3
    (64, 32, 32, 250, 32, 0, 0, 0),   # -3.7
    (64, 32, 4, 2000, 2000, 1, 1, 1),
    (128, 16, 4, 320, 2, 0, 1, 0),    # -4.5
    (128, 16, 16, 20, 12, 0, 1, 1),   # -3.5
    (128, 16, 4, 700, 700, 0, 1, 1),
]


@pytest.mark.parametrize("shape", SLOWER + FASTER)
def test_batches_take_strips_where_those_measured_faster(shape):
    L = R.lib()
    L.rh_strip_route_host.argtypes = [ctypes.c_size_t] * 5 + [ctypes.c_int] * 3
    assert L.rh_strip_route_host(*shape) == (shape in FASTER)


def test_strips_take_no_shape_beyond_their_lds_or_one_token():
    L = R.lib()
    L.rh_strip_route_host.argtypes = [ctypes.c_size_t] * 5 + [ctypes.c_int] * 3
    for head_dim, heads, kv_heads in ((64, 32, 4), (64, 32, 8), (64, 32, 32), (128, 16, 4)):
        grouped = int(head_dim == 64 and heads // kv_heads in (4, 8))
        assert L.rh_strip_route_host(head_dim, heads, kv_heads, 2496, 64, grouped, 1, 1)
        assert not L.rh_strip_route_host(head_dim, heads, kv_heads, 2497, 64, grouped, 1, 1)
        assert not L.rh_strip_route_host(head_dim, heads, kv_heads, 1000, 1, grouped, 1, 0)
    assert not L.rh_strip_route_host(96, 8, 2, 1000, 64, 0, 1, 1)


@pytest.mark.parametrize("head_dim,rows,split", [
    (64, 225, 0), (64, 256, 0), (64, 257, 1), (64, 4480, 1), (64, 4500, 0),  # +1.4 us a layer at 235 rows, -0.1 at 260
    (128, 1, 1), (128, 4480, 1), (128, 4500, 0), (32, 1000, 0), (96, 1000, 0)])
def test_one_token_takes_the_split_step_where_it_measured_faster(head_dim, rows, split):
    L = R.lib()
    L.rh_step_route_host.argtypes = [ctypes.c_size_t] * 2
    assert L.rh_step_route_host(head_dim, rows) == split


@pytest.mark.parametrize("head_dim,heads,context", [(64, 32, 200), (64, 32, 256), (64, 32, 257), (64, 32, 2048),
                                                    (64, 32, 4488), (64, 32, 32576), (128, 16, 40), (128, 16, 32576),
                                                    (2, 4096, 32576), (96, 8, 2048)])
def test_step_scratch_holds_the_rows_the_split_step_takes_and_no_more(head_dim, heads, context):
    L = R.lib()
    L.rh_step_route_host.argtypes = [ctypes.c_size_t] * 2
    L.rh_step_scratch_host.argtypes, L.rh_step_scratch_host.restype = [ctypes.c_size_t] * 3, ctypes.c_size_t
    rows = max((r for r in range(1, min(context, 6000) + 1) if L.rh_step_route_host(head_dim, r)), default=0)
    assert L.rh_step_scratch_host(head_dim, heads, context) == heads * ((rows + 63) // 64 * 64)


# us, the tiled kernel and gemv_dense_kernel
@pytest.mark.parametrize("rows,cols,tokens,tiled", [
    (64, 8, 1, 0),         # 2.8, 2.1
    (32000, 8, 1, 0),      # 4.4, 2.6
    (32000, 64, 1, 0),     # 4.5, 3.3
    (20000, 64, 2, 0),     # 5.0, 4.0
    (32000, 32, 5, 0),     # 6.1, 6.0
    (20000, 256, 1, 0),    # 7.5, 5.1
    (12000, 384, 1, 0),    # 6.6, 5.7
    (5632, 512, 1, 0),     # 6.9, 6.5
    (5632, 128, 2, 1),     # 4.2, 4.8
    (2048, 768, 1, 1),     # 8.2, 8.7
    (32000, 384, 1, 1),    # 11.0, 12.7
    (12000, 512, 1, 1),    # 7.9, 9.3
    (32000, 2048, 1, 1), (64, 1024, 1, 1), (64, 16384, 1, 1), (64, 16385, 1, 0), (64, 2048, 8, 1), (64, 2052, 8, 0)])
def test_dense_rows_take_the_tiled_kernel_where_it_measured_faster(rows, cols, tokens, tiled):
    L = R.lib()
    L.rh_dense_route_host.argtypes = [ctypes.c_size_t] * 3
    assert L.rh_dense_route_host(rows, cols, tokens) == tiled
