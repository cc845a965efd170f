"""Jacobi-CG coarse solves on a coarsest level of order 2 to 4, down to a single level: the element passes with
four waves to a cell, the matrix-core pass (no fused inner product) and odd and even iteration counts.
The solve must end at the oracle's residual."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n,orders", [(2, 9, [2]), (2, 13, [4, 3]), (3, 3, [2]), (3, 4, [3]), (3, 3, [4, 3]),
                                          (3, 2, [4]), (3, 6, [4, 2])])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("iters", [7, 20])
def test_coarsest_order_above_one(ip, oracle, dim, n, orders, mixed, iters):
    print(f"coarsest order {orders} dim={dim} n={n} mixed={mixed}", flush=True)
    mesh = ip.Mesh.square(n, jitter=0.1, seed=8) if dim == 2 else ip.Mesh.cube(n, 0.1, 8)
    s = ip.PoissonSolver(mesh, orders[0])
    o = oracle.Oracle(*mesh.arrays(), orders[0])
    s.set_pmg(orders, coarse_iters=iters)
    s.set_precision(ip.PRECISION_MIXED if mixed else ip.PRECISION_FP64)
    s.set_tol_and_iter(1e-9, 0.0, 2000)
    b = np.random.default_rng(n).standard_normal((s.n_cells, s.Np))
    x = np.zeros_like(b)
    assert s.solve(b, x)
    # 1e-9 of |b| by the solver's own residual, and the rounding of two applies (1e-11 at order 4)
    assert np.linalg.norm(b - o.mult(x)) <= 1.02e-9 * np.linalg.norm(b)
