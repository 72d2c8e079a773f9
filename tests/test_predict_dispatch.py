"""The kernel that wgbm_predict_heap takes for a call's sizes (CPU: the rule is
host code).  Each pair below was measured both ways on an MI355X; where the
margin is wide the dispatch has to take the faster one."""
import pytest

from warpgbm_amd import _lib
from warpgbm_amd import device as D

HEAP, ROWS, RESIDENT, COLS = range(4)


# rows, features, classes, rounds, depth, kernel: us by that kernel / by the
# column blocks (or by what else the call could take)
MEASURED = [
    # few rows, many shallow trees: row blocks that fill the CUs
    (500, 128, 17, 100, 1, RESIDENT),     # 14 / 118
    (4000, 30, 10, 100, 3, RESIDENT),     # 16 / 74
    (8000, 128, 10, 100, 1, RESIDENT),    # 20 / 73
    (500, 128, 7, 100, 4, ROWS),          # 33 / 60
    (500, 128, 10, 100, 4, ROWS),         # 44 / 76
    (16_000, 128, 7, 100, 4, ROWS),
    # a class's deep trees one after the other cost less than more passes
    (500, 128, 1, 100, 8, COLS),          # 29 / 42
    (4000, 60, 3, 40, 8, COLS),           # 36 / 61
    (500, 128, 16, 100, 8, COLS),         # 262 / 460
    (500, 128, 10, 5, 4, COLS),           # 11 / 25
    # a thread per (row, class): few rows, tables that fit the L2
    (500, 128, 17, 30, 8, HEAP),          # 70 / 119
    (30_000, 128, 17, 30, 8, COLS),       # 114 / 326
    # every CU has column blocks
    (1_000_000, 100, 10, 200, 6, COLS),   # 1910 / 3600
    (250_000, 128, 10, 100, 1, COLS),
    # one workgroup of it a CU: by the work per row, and by whole passes
    (200_000, 300, 1, 100, 5, RESIDENT),  # 64 / 81
    (70_684, 128, 5, 100, 2, RESIDENT),   # 58 / 82
    (250_000, 380, 8, 30, 4, COLS),
    (1_000_000, 1000, 1, 100, 5, RESIDENT),
]


@pytest.mark.parametrize("n,F,K,rounds,depth,path", MEASURED)
def test_predict_heap_takes_the_faster_kernel(n, F, K, rounds, depth, path):
    got = _lib.load().wgbm_predict_heap_path(n, D.codes_stride(F), rounds, K, depth)
    assert got == path


def test_predict_heap_path_refuses_sizes_out_of_range():
    path = _lib.load().wgbm_predict_heap_path
    for n, S, rounds, K, depth in ((-1, 16, 1, 1, 3), (1, 0, 1, 1, 3), (1, 16, 0, 1, 3),
                                   (1, 16, 1, 0, 3), (1, 16, 1, 1, -1), (1, 16, 1, 1, 30)):
        assert path(n, S, rounds, K, depth) == -1


def test_predict_heap_path_covers_every_size():
    """No combination of sizes divides by zero or names an unknown kernel."""
    path = _lib.load().wgbm_predict_heap_path
    for n in (0, 1, 255, 65_280, 65_281, 10_000_000):
        for S in (1, 8, 16, 128, 384, 496, 512, 1024, 65_536, 70_000):
            for rounds in (1, 7, 1000):
                for K in (1, 7, 8, 16, 17, 32, 33, 5000):
                    for depth in (0, 1, 4, 8, 9, 12, 29):
                        assert path(n, S, rounds, K, depth) in (HEAP, ROWS, RESIDENT, COLS)
