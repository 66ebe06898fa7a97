"""Which tile shape a prefill GEMM call takes (host only): the cases of the GPU
test take the shapes that they are listed under, every shape has one that goes
round all its buffers, and the rows past 32-bit offsets have a shape of their
own."""
import ctypes

import pytest

from modgrad_amd import _lib
from tests.test_gpu_gemm_tiles import CASES


def pick(n, bpr, m, cus=256):
    shape = (ctypes.c_int * 3)()
    at = [ctypes.byref(shape, 4 * i) for i in range(3)]
    return _lib.load().mgq_gemm_tile(n, bpr, m, cus, *at), tuple(shape)


@pytest.mark.parametrize("tile", CASES)
def test_cases_take_their_tile(tile):
    for n, bpr, m in CASES[tile]:
        assert pick(n, bpr, m)[1] == tile, (n, bpr, m)
    # at most 4 half blocks of tokens are buffered and 2 blocks of W held
    n, bpr, m = CASES[tile][-1]
    shares = tile[2]
    assert bpr // shares >= 3 and -(-bpr // shares) >= 4 and (shares == 1 or bpr % shares)


def test_every_tile_has_cases():
    index = {pick(*CASES[tile][0])[0] for tile in CASES}
    assert index == set(range(len(CASES)))


def test_long_rows_take_64_bit_offsets():
    # 16 tokens x 2^27 f16 values are 2^32 bytes
    assert pick(3, 524288, 2) == (len(CASES), (32, 32, 4))
    assert pick(3, 524287, 2) == (0, (32, 16, 4))


def test_invalid_arguments():
    assert pick(0, 1, 1)[0] == -1
    assert pick(1, 0, 1)[0] == -1
    assert pick(1, 1, 0)[0] == -1
    assert pick(1, 1, 1, 0)[0] == -1
    assert _lib.load().mgq_gemm_tile(1, 1, 1, 256, None, None, None) == -1
