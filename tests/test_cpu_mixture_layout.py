"""Which layout the rows of a mixture's prompt step get (blocks of 64 rows an expert, or whole tiles of 256): the estimate against steps measured on both sides."""
import ctypes

import pytest

from candle_vllm_amd._lib import lib

Q4, Q6 = 12, 14


# hidden, columns of an expert, experts, rows (tokens x experts a token), type of the down product, whole tiles; measured us of both products, blocks / tiles
@pytest.mark.parametrize("hid,inter,experts,pairs,down,tiles", [
    (4096, 14336, 8, 8192, Q4, 1),                                    # 3759 / 3473
    (4096, 14336, 8, 4200, Q6, 1),                                    # 2668 / 2155
    (4096, 14336, 8, 3500, Q4, 0),                                    # the down product goes in ranges of K
    (4096, 7168, 8, 3696, Q4, 1),                                     # 1117 / 809
    (4096, 1792, 8, 4200, Q4, 0),                                     # 337 / 395
    (4096, 1792, 8, 6000, Q4, 1),                                     # 480 / 438
    (4096, 1792, 8, 4200, Q6, 1),                                     # 439 / 392
    (2048, 1536, 16, 8192, Q4, 0),                                    # 297 / 352
    (2048, 1536, 16, 16384, Q4, 1),                                   # 620 / 532
    (1024, 3584, 4, 4200, Q4, 0),                                     # 207 / 250
    (1024, 3584, 4, 8192, Q6, 1),                                     # 449 / 364
    (14336, 14336, 8, 200000, Q4, 0)])                                # an image beyond 32-bit offsets
def test_layout(hid, inter, experts, pairs, down, tiles):
    fn = lib.mi355_internal_moe_tiles
    fn.argtypes, fn.restype = [ctypes.c_int32] * 5, ctypes.c_int32
    assert fn(pairs, experts, hid, inter, down) == tiles
