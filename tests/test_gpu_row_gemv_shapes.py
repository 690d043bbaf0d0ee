"""The FP8 decode GEMV on both sides of the lines between its workgroup shapes: up to 4 chunks of K and more (a workgroup
of four tiles, the last one with fewer), the widest K whose 4 or 8 parts quantize the call's 1 to 4 tokens and one chunk
more, and 12 | 13 chunks of many tiles. On representable inputs the FP32 sums equal the oracle's bit for bit, with and
without codes asked for."""

import pytest

from tests.test_gpu_row_gemv_split import check_exact

pytestmark = pytest.mark.gpu

SHORT = [(rows, 128 * chunks, tokens) for rows in (64, 4160, 16448) for chunks in (1, 3, 4, 5) for tokens in (1, 4, 5, 32)]
FEW = [(192, 128 * chunks, tokens) for tokens, chunks in ((1, 55), (1, 56), (1, 128), (1, 129), (2, 27), (2, 28), (2, 33), (2, 64),
                                                         (2, 65), (3, 20), (3, 21), (3, 40), (3, 41), (4, 16), (4, 17),
                                                         (4, 32), (4, 33))]
BETWEEN = [(4160, 128 * chunks, tokens) for tokens, chunks in ((1, 64), (1, 65), (2, 33), (3, 20), (3, 21), (3, 41), (4, 16),
                                                              (4, 17), (4, 33))]
MANY = [(16448, 128 * chunks, tokens) for tokens, chunks in ((2, 13), (3, 12), (3, 13), (3, 21), (4, 12), (4, 16), (4, 17),
                                                        (4, 31), (4, 32))]


@pytest.mark.parametrize("block", [32, 128])
@pytest.mark.parametrize("rows,width,tokens", SHORT + FEW + BETWEEN + MANY)
def test_both_sides_of_each_line(gpu_ctx, block, rows, width, tokens):
    check_exact(gpu_ctx, block, rows, width, tokens)
