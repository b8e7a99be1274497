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
