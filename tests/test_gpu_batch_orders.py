"""Batches below and above the size up to which one launch takes the problems of every order.

A problem's arithmetic is the same in both forms, so its result alone and beside a problem that
takes the batch over that size agree bit for bit. Cells per problem leave remainders in the 64-cell
tiles, and every order has a problem of less than one tile.
"""
import numpy as np
import pytest

from test_gpu_batch import cube, relL2, run_batch, sin_problem, sq

pytestmark = pytest.mark.gpu

# 2 * 370^2 and 6 * 28^3 cells: just over 4096 and 2048 tiles
FILL = {2: lambda ip: sq(ip, 370, 90), 3: lambda ip: cube(ip, 28, 90)}
SIZES = {2: [(5, 1), (4, 2), (5, 3), (5, 4), (9, 2), (8, 3), (13, 4)],
         3: [(2, 1), (2, 2), (2, 3), (2, 4), (3, 2), (4, 4)]}


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("mixed", [False, True])
def test_orders_in_one_launch(ip, dim, mixed):
    mesh = (lambda n, seed: sq(ip, n, seed)) if dim == 2 else (lambda n, seed: cube(ip, n, seed))
    probs = [sin_problem(ip, mesh(n, i), N, rtol=1e-11) for i, (n, N) in enumerate(SIZES[dim])]
    cfg = dict(precision=ip.PRECISION_MIXED if mixed else ip.PRECISION_FP64)
    _, _, small = run_batch(ip, dim, probs, tile=64, **cfg)
    fill = sin_problem(ip, FILL[dim](ip), 1, rtol=1e-11, max_iter=2)
    _, _, large = run_batch(ip, dim, probs + [fill], tile=64, **cfg)
    _, _, wide = run_batch(ip, dim, probs, tile=256, **cfg)
    for s, l, w in zip(small, large, wide):
        assert s[0] == l[0] == w[0] and np.array_equal(s[1], l[1])
        # other tiles add the inner products in another order: both end at 1e-11 of the right-hand
        # side, and the operators' condition numbers here stay below 1e4
        assert relL2(s[1], w[1]) < 1e-7
