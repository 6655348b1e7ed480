"""Inputs at the edges of what the entry points take: far queries, queries next
to sources, values that are no numbers, radii below zero, more queries than 32
bits count, calls recorded into a graph."""
import numpy as np
import pytest

import oracle as O
from dwg_amd import gpu

pytestmark = pytest.mark.gpu


def test_knn_far_query_beside_a_cell_boundary(ctx):
    # A point just below a cell's lower boundary that its rounded difference to
    # the grid's corner puts into that cell, and a query so far away that its
    # differences to the point and to the boundary round to neighbouring floats:
    # the cell's box lies farther than the point, which ties with others of
    # higher index for the last place.  n, the extent and two points a cell make
    # the cells 1/64 wide.
    f = np.float32
    rng = np.random.default_rng(3)
    p = np.nextafter(f(0.53125), f(0))
    rows = [(p, 0, 0), (0.535, 0, 0), (0.5, 0, 0), (0.505, 0, 0), (-1, -1, -1), (-0.999, -1, -1)]
    cells = rng.choice(24 * 62 * 62, 16384 - 4, replace=False)
    x, y, z = cells % 24 + 104, cells // 24 % 62 + 65, cells // (24 * 62) + 65
    c = np.stack([x, y, z], 1) / 64 - 1
    far_end = [(1, 0.3, 0.3), (1, 0.301, 0.301)]
    P = np.concatenate([np.array(rows), c + 0.3 / 64, c + 0.7 / 64, far_end]).astype(np.float32)
    Q = np.array([[-524288.0625, 0, 0]], np.float32)
    got, d2 = gpu.KnnIndex(ctx, P, k_hint=1).query(Q, 3, d2=True)
    ref, rd2 = O.knn_brute(P, Q, 3, return_d2=True)
    assert sorted(ref[0]) == [0, 4, 5]
    np.testing.assert_array_equal(got.cpu().numpy(), ref)
    np.testing.assert_array_equal(d2.cpu().numpy(), rd2)
