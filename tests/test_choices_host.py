"""Host checks of the rules by which a launch picks its variant: the library's
own host-only queries, at sizes where both sides were measured on 256 CUs."""
from __future__ import annotations

import pytest

from comfyui_turing_utils_kernel import _lib

CUS = 256


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


# (rows, columns, group): the rows that share a table, 0 for none, and what was slower
GELU_ROWS = [
    (4096, 16896, 128, {8}),          # 99 us; 1 to 7 rows 117-154
    (4096, 20480, 128, {8}),          # 116; 134-177
    (1560, 20480, 256, {0, 7}),       # 70, 74; one row 87, eight 83
    (4096, 20480, 256, {0}),          # 157; four rows 176, eight 172
    (10000, 5120, 128, {5}),          # 66; eight 78
    (6144, 8192, 256, {4, 6}),        # 63, 70; eight 84
    (6145, 8192, 256, {4, 5, 6}),     # as 6144: no step between them
    (6145, 13824, 128, {8}),          # 100; seven 108
    (2050, 13824, 128, {2, 3}),       # 41; eight 59
    (512, 13824, 128, {1}),           # 16; eight 58
    (7800, 8960, 128, {4, 8}),        # 93; one row 119
    (32760, 13824, 128, {8}),
]


@pytest.mark.parametrize("rows,k,group,good", GELU_ROWS)
def test_gelu_rows(lib, rows, k, group, good):
    assert lib.tu_convrot_table_rows(rows, k, group, 1, CUS) in good


def test_gelu_rows_range(lib):
    """Short rows, rows too wide for a table, other activations and bad
    arguments have none; the choice never leaves 0 .. 8."""
    for rows in (1, 300, 8190, 16000, 32760):
        for k in (512, 1536, 3072):
            assert lib.tu_convrot_table_rows(rows, k, 128, 1, CUS) == 0
        assert lib.tu_convrot_table_rows(rows, 65536, 128, 1, CUS) == 0
    for act in (0, 2, 3):
        assert lib.tu_convrot_table_rows(4096, 8960, 128, act, CUS) == 0
    for rows, k, group, cus in ((0, 8960, 128, CUS), (5, 0, 128, CUS), (5, 8960, 64, CUS), (5, 8960, 128, 0), (5, 65537, 128, CUS)):
        assert lib.tu_convrot_table_rows(rows, k, group, 1, cus) == 0
    for cus in (1, 64, 256, 304):
        for rows in (1, 2, 255, 257, 4097, 100003, 2 ** 31 - 1):
            for k in (3200, 4096, 4224, 8192, 16896, 20480, 32768):
                assert 0 <= lib.tu_convrot_table_rows(rows, k, 128, 1, cus) <= 8


@pytest.mark.parametrize("rows,k,good", [
    (2050, 14336, {3}),           # 46 us; without a table 54
    (16380, 13824, {4, 5, 8}),    # 285; 336
    (1, 14336, {1}),              # 13.0; 14.4
    (4096, 8960, {0}), (513, 8448, {0}), (2050, 20480, {0}), (1000, 32768, {0}), (4096, 5120, {0}),  # slower with one
])
def test_swiglu_rows(lib, rows, k, good):
    """Only rows of four waves share a SwiGLU table."""
    for group in (128, 256):
        if k % group == 0:
            assert lib.tu_convrot_table_rows(rows, k, group, 2, CUS) in good


# (m, n, k): the tiles within 3 % of the best one, and what was slower
GEMM_TILES = [
    (2050, 8960, 1536, {(256, 192)}),                # 40.9 us; 128 x 256 47.2
    (16380, 1536, 1536, {(256, 192)}),               # 44.6; 256 x 256 and 128 x 256 50
    (1024, 5120, 256, {(128, 192)}),                 # 7.5; 256 x 192 9.2
    (4096, 10240, 5120, {(256, 256)}),               # 183; 128 x 256 202
    (7800, 5120, 5120, {(256, 256)}),                # 184; 128 x 256 198
    (7800, 5120, 13824, {(256, 256)}),               # 469; 128 x 256 503
    (16380, 5376, 14336, {(256, 256)}),              # 1032; 256 x 192 1078
    (1560, 5120, 13824, {(256, 192)}),               # 127; 128 x 192 138
    (2050, 5376, 14336, {(256, 192)}),               # 139; 128 x 192 161
    (32760, 13824, 5120, {(256, 256)}),              # 1845; 256 x 192 2058
    (1024, 8960, 1536, {(256, 192)}),                # 20.8; 256 x 256 23.2, 128 x 192 26.0
    (512, 10240, 5120, {(128, 192)}),                # 29.9; 128 x 256 34.4
    (512, 5120, 5120, {(128, 128)}),                 # 22.6; 128 x 192 27.6
    (1024, 1536, 1536, {(128, 64)}),                 # 8.2; 64 x 64 9.4
    (1, 8960, 1536, {(64, 64)}),                     # 6.1; 128 x 64 7.3
]


@pytest.mark.parametrize("m,n,k,good", GEMM_TILES)
def test_gemm_tile(lib, m, n, k, good):
    t = lib.tu_int8_gemm_tile(m, n, k, CUS)
    assert (t >> 16, t & 0xFFFF) in good


def test_gemm_tile_range(lib):
    """A grid of the tile taken holds fewer than 2^32 threads wherever one of
    256 x 256 tiles does, and bad arguments are answered with 0."""
    for m in (1, 2 ** 20, 2 ** 29 - 64, 2 ** 29, 2 ** 30, 2 ** 30 + 1, 2 ** 31 - 256):
        for n, k in ((8, 16), (64, 16), (64, 4096), (128, 256), (256, 512)):
            t = lib.tu_int8_gemm_tile(m, n, k, CUS)
            bm, bn = t >> 16, t & 0xFFFF
            assert -(-m // bm) * -(-n // bn) * 512 < 2 ** 32, (m, n, k)
    for bad in ((0, 8, 16, 256), (8, 0, 16, 256), (8, 8, 0, 256), (8, 8, 16, 0)):
        assert lib.tu_int8_gemm_tile(*bad) == 0
