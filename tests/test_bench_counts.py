"""The bytes that bench.py counts for a Coulomb launch: operands in tiles of 16 columns, as the library stores them."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


@pytest.mark.parametrize("prec,size", [("fp64", 8), ("mixed", 4), ("bf16x3", 6), ("bf16x2", 4)])
@pytest.mark.parametrize("nF,cols", [(1, 16), (16, 16), (20, 32), (96, 96), (97, 112), (192, 192), (240, 240)])
def test_coulomb_bytes(nF, cols, prec, size):
    import bench
    M, rows = 1000, 640
    counts = [0, 600, M, 50, nF, 10, rows, 0, 0, 0]
    assert bench.coulomb_bytes(counts, prec) == rows * cols * size + 8 * M * nF + 24 * M
