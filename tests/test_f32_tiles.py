"""Which rows of a matrix the 32-bit products of few rows read: the kernel's own map, walked on the host."""
import ctypes

import pytest

PLAIN, GATED, ROPE = 0, 1, 2


@pytest.fixture(scope="module")
def row_of():
    from tokenizer_amd.kernels import build
    path = build.find_library() or build.build_library(verbose=False)
    return ctypes.CDLL(path).ta_gemm_f32_tile_row


@pytest.mark.parametrize("heads", [3, 6, 18])
@pytest.mark.parametrize("d", [16, 32, 64, 96, 256])
@pytest.mark.parametrize("rows", [8, 4, 2])
def test_rows_of_a_pair_of_halves(row_of, heads, d, rows):
    n, seen = heads * d, set()
    for block in range(heads * (d // 2 // rows)):
        head, first = divmod(block * rows, d // 2)
        for i in range(16):
            got = row_of(ROPE, block, n, rows, d, i)
            assert 0 <= got < n                                # (also where row i of the tile is not there: some forms load it)
            if i % 8 < rows:
                assert got == head * d + first + i % 8 + (d // 2 if i >= 8 else 0)
                seen.add(got)
    assert seen == set(range(n))


@pytest.mark.parametrize("n", [2, 8, 30, 100, 1152])
def test_rows_of_a_gated_matrix(row_of, n):
    half, seen = n // 2, set()
    for block in range(-(-half // 8)):
        for i in range(16):
            got = row_of(GATED, block, n, 8, 0, i)
            assert 0 <= got < n and got == min(block * 8 + i % 8, half - 1) + (half if i >= 8 else 0)
            seen.add(got)
    assert seen == set(range(n))


@pytest.mark.parametrize("n", [1, 4, 17, 100, 1150])
@pytest.mark.parametrize("rows", [4, 7, 16])
def test_rows_of_a_plain_matrix(row_of, n, rows):
    seen = set()
    for block in range(-(-n // rows)):
        for i in range(16):
            got = row_of(PLAIN, block, n, rows, 0, i)
            assert 0 <= got < n and (i >= rows or got == min(block * rows + i, n - 1))
            seen.add(got)
    assert seen == set(range(n))


@pytest.mark.parametrize("kind, block, n, rows, d, i", [(ROPE, 0, 576, 0, 96, 0), (ROPE, 0, 576, 8, 0, 0), (PLAIN, 0, 0, 16, 0, 0),
                                                        (GATED, -1, 8, 8, 0, 0), (PLAIN, 0, 8, 16, 0, 16)])
def test_what_is_no_tile(row_of, kind, block, n, rows, d, i):
    assert row_of(kind, block, n, rows, d, i) == -1
