"""The trace and element passes with four waves to a cell and with one thread to a cell, on both sides of
the mesh sizes where one takes over from the other and at the smallest meshes, against the FP64 oracle:
A u plus a mass term, with and without a coefficient, mixed boundary types. Tolerances as in the parity
tests of the apply (sums of at most 200 terms per entry: 1e-12 FP64, 1e-11 at order 4, where the
oracle's own reference element carries 5e-13; 2e-5 FP32)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (dim, order, hexes or squares per edge): 1 cell pair / 6 cells, remainders of 64 cells, and the
# last mesh below and the first above 2^16, 1.5 x 2^16 and 3 x 2^16 cells
SIZES = [(2, 2, 1), (2, 3, 7), (2, 4, 23), (2, 2, 181), (2, 2, 182), (2, 3, 182), (2, 4, 313), (2, 4, 314),
         (3, 2, 1), (3, 3, 1), (3, 4, 2), (3, 3, 5), (3, 2, 31), (3, 2, 33), (3, 3, 25), (3, 3, 26), (3, 4, 22),
         (3, 4, 23)]


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("dim,N,n", SIZES)
@pytest.mark.parametrize("factor", [False, True])
def test_apply_both_forms(ip, oracle, dim, N, n, factor):
    print(f"split passes dim={dim} N={N} n={n} factor={factor}", flush=True)
    mesh = ip.Mesh.square(n, jitter=0.1, seed=5) if dim == 2 else ip.Mesh.cube(n, 0.1, 5)
    s = ip.PoissonSolver(mesh, N)
    o = oracle.Oracle(*mesh.arrays(), N)
    bt = np.zeros(s.n_bfaces, dtype=np.int32)
    bt[1::4] = 1
    s.set_bc_types(bt)
    o.set_bc_types(bt)
    s.set_solver(ip.SOLVER_JACOBI)
    s.set_element_pass(ip.ELEMENT_PASS_VECTOR)
    rng = np.random.default_rng(n)
    if factor:
        k, mm = 1.0 + rng.random((s.n_cells, s.Np)), 20.0 + 10.0 * rng.random((s.n_cells, s.Np))
        s.set_factor(k)
        o.set_factor(k)
        s.set_mm_factor(mm)
        o.set_mm_factor(mm)
    else:
        s.set_mm_const(40.0)
        o.set_mm_const(40.0)
    x = rng.standard_normal((s.n_cells, s.Np))
    y = o.mult(x)
    assert rel(s.mult(x), y) < (1e-12 if N < 4 else 1e-11)
    assert rel(s.mult_fp32(x), y) < 2e-5
