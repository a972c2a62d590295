"""The FP8 GEMM's tile choice (no GPU): the shapes of gemm_tiles.py take the tiles they are listed under, so the GPU
tests that use them cover every tile; arguments are checked."""
import ctypes
import os
import re

import pytest

import _tglib as L
import gemm_tiles as G


def test_header_and_signatures_agree():
    text = open(os.path.join(os.path.dirname(L.HEADER_PATH), "tg_fp8_tiles.h")).read()
    names = set(re.findall(r"\b(tg_[a-z0-9_]+)\s*\(", re.sub(r"/\*.*?\*/", "", text, flags=re.S)))
    assert names == set(L.TILE_SIGNATURES)


@pytest.mark.parametrize("tile", sorted(G.GEMM))
def test_listed_shapes_take_their_tile(tile):
    for M, N, K, km in G.GEMM[tile]:
        assert G.tile_of(M, N, K, km) == tile, (M, N, K, km)


def test_listed_linears_take_their_tiles():
    seen = set()
    for (M, K, N), (dx, dw) in G.LINEAR_F32.items():
        assert G.tile_of(M, K, G.up128(N), True, f32=True) == dx, (M, K, N)
        assert G.tile_of(K, N, G.up128(M), True, f32=True) == dw, (M, K, N)
        seen |= {dx, dw}
    # the 128 x 128 tile is for kept weights only
    assert seen == set(G.GEMM) - {(128, 128)}


def test_kept_weights_do_not_take_two_rounds_of_64_rows_where_one_of_128_does():
    """Some 10 k columns and a few hundred rows: 64-row tiles read the weight's blocks twice as often."""
    for M, N, K in ((300, 14336, 4096), (448, 10240, 3072), (350, 12288, 2048), (448, 10240, 1024), (512, 9216, 2304),
                    (350, 9216, 2304), (512, 6912, 2304), (256, 14336, 4096), (400, 8192, 4096)):
        assert G.tile_of(M, N, K, False)[0] == 128, (M, N, K)


def test_bad_calls():
    r, c = ctypes.c_int(), ctypes.c_int()
    p, q = ctypes.byref(r), ctypes.byref(c)
    call = L.lib().tg_gemm_fp8_tile
    for args in ((-1, 8, 128, 0, 0, 256, p, q), (8, 8, 100, 0, 0, 256, p, q), (8, 8, 128, 0, 2, 256, p, q),
                 (8, 8, 128, 0, 0, 0, p, q), (8, 8, 128, 0, 0, 256, None, q), (8, 8, 128, 0, 0, 256, p, None)):
        assert call(*args) == L.TG_EINVAL
    # past 32-bit offsets, and nothing to multiply: no tile
    for M, N, K in ((1 << 24, 128, 128), (0, 8, 128), (8, 0, 128)):
        assert G.tile_of(M, N, K, False) == (0, 0)
