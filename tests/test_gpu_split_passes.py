"""The trace and element passes with four waves to a cell and with one thread to a cell, on both sides of
the mesh sizes where one takes over from the other and at the smallest meshes, against the FP64 oracle:
A u plus a mass term, with and without a coefficient, mixed boundary types. Tolerances as in the parity
tests of the apply (sums of at most 200 terms per entry: 1e-12 FP64, 1e-11 at order 4, where the
oracle's own reference element carries 5e-13; 2e-5 FP32)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (dim, order, hexes or squares per edge): 1 cell pair / 6 cells, remainders of 64 cells, and meshes on both
# sides of the lines of the element pass (2D 2^16 cells, order 4 3 x 2^16; 3D order 2 12 x 2^16, order 3 1.5
# x 2^16 and FP32 2 x 2^16, order 4 2^16 and FP32 1.5 x 2^16) and of the trace pass (2D order 4 and 3D
# order 2 3 x 2^16, 3D order 3 6 x 2^16)
SIZES = [(2, 2, 1), (2, 3, 7), (2, 4, 23), (2, 2, 181), (2, 2, 182), (2, 3, 182), (2, 4, 313), (2, 4, 314),
         (3, 2, 1), (3, 3, 1), (3, 4, 2), (3, 3, 5), (3, 2, 31), (3, 2, 33), (3, 3, 25), (3, 3, 26), (3, 4, 22),
         (3, 4, 23), (3, 2, 50), (3, 2, 51), (3, 3, 28), (3, 3, 29), (3, 4, 25), (3, 4, 26), (3, 3, 40), (3, 3, 41)]


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


@pytest.mark.parametrize("dim,n", [(2, 250), (3, 28)])
@pytest.mark.parametrize("factor", [False, True])
def test_order1_apply_repeats(ip, oracle, dim, n, factor):
    """Several waves per SIMD: every launch of the order-1 pass gives the same bits, and the oracle's
    values (1e-12: at most 40 terms per entry)."""
    mesh = ip.Mesh.square(n, jitter=0.1, seed=5) if dim == 2 else ip.Mesh.cube(n, 0.1, 5)
    s = ip.PoissonSolver(mesh, 1)
    o = oracle.Oracle(*mesh.arrays(), 1)
    s.set_solver(ip.SOLVER_JACOBI)
    rng = np.random.default_rng(n)
    if factor:
        k = 1.0 + rng.random((s.n_cells, s.Np))
        s.set_factor(k)
        o.set_factor(k)
    x = rng.standard_normal((s.n_cells, s.Np))
    y = s.mult(x)
    assert rel(y, o.mult(x)) < 1e-12
    for _ in range(20):
        assert np.array_equal(s.mult(x), y)


# 3D: 162 cells (direction in the apply) to 215,622 (two pairs per thread); 279,936 and 584,016 cells take
# four pairs per thread and fold both sums, as 2D 361,250 does; 2D 980,000 cells fold r.z and leave p.Ap to
# a kernel in between, 3D 795,906 leave both (two pairs). The two largest carry a mass term, which keeps the
# number of outer iterations small.
@pytest.mark.parametrize("dim,n,iters", [(2, 4, 1), (2, 4, 2), (2, 30, 7), (3, 3, 8), (3, 12, 9), (3, 27, 12),
                                         (3, 33, 12), (2, 425, 21), (3, 36, 12), (3, 46, 13), (2, 700, 8), (3, 51, 9)])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("factor", [False, True])
def test_coarse_cg_forms(ip, oracle, dim, n, iters, mixed, factor):
    """The order-1 Jacobi-CG with the direction formed in the apply (small meshes), as updates of their
    own, with one, two and four pairs per thread, with sums folded into the next kernel and added by a kernel
    in between; odd and even counts. The preconditioned solve must end at the oracle's residual and
    take the same iterations twice."""
    mesh = ip.Mesh.square(n, jitter=0.1, seed=5) if dim == 2 else ip.Mesh.cube(n, 0.1, 5)
    s = ip.PoissonSolver(mesh, 2)
    o = oracle.Oracle(*mesh.arrays(), 2)
    rng = np.random.default_rng(n)
    if factor:
        k = 1.0 + rng.random((s.n_cells, s.Np))
        s.set_factor(k)
        o.set_factor(k)
    if s.n_cells > 750000:
        s.set_mm_const(10.0 * n * n)
        o.set_mm_const(10.0 * n * n)
    s.set_pmg([2, 1], coarse_iters=iters)
    s.set_precision(ip.PRECISION_MIXED if mixed else ip.PRECISION_FP64)
    s.set_tol_and_iter(1e-9, 0.0, 2000)
    b = rng.standard_normal((s.n_cells, s.Np))
    x, y = np.zeros_like(b), np.zeros_like(b)
    assert s.solve(b, x)
    its = s.last_stats["iterations"]
    assert np.linalg.norm(b - o.mult(x)) <= 2e-9 * np.linalg.norm(b)
    assert s.solve(b, y) and s.last_stats["iterations"] == its
    assert np.array_equal(x, y)


@pytest.mark.parametrize("dim,N,n", [(2, 1, 1), (2, 2, 6), (2, 3, 7), (2, 4, 9), (3, 1, 3), (3, 2, 1), (3, 3, 3),
                                     (3, 4, 2)])
def test_over_integrated_apply(ip, oracle, dim, N, n):
    """Remainders of the 64-cell blocks, mixed boundary types, both precisions (tolerances as above; the
    face and volume sums have at most 216 + 64 terms)."""
    mesh = ip.Mesh.square(n, jitter=0.1, seed=6) if dim == 2 else ip.Mesh.cube(n, 0.1, 6)
    s = ip.PoissonSolver(mesh, N)
    o = oracle.Oracle(*mesh.arrays(), N, faces=mesh.faces())
    bt = np.zeros(s.n_bfaces, dtype=np.int32)
    bt[1::3] = 1
    s.set_bc_types(bt)
    o.set_bc_types(bt)
    rule = ip.oi_rule(dim, N)
    rng = np.random.default_rng(n)
    kv = 1.0 + rng.random((s.n_cells, rule[0].shape[0]))
    ks = 1.0 + rng.random((s.n_cells, (dim + 1) * rule[2].shape[0]))
    kn = 1.0 + rng.random((s.n_cells, s.Np))
    s.set_factor(kn)
    o.set_factor(kn)
    s.set_factor_oi(kv)
    s.set_factor_surf_oi(ks)
    s.set_solver(ip.SOLVER_JACOBI)
    x = rng.standard_normal((s.n_cells, s.Np))
    y = o.mult_oi(rule, kv, ks, x)
    assert rel(s.mult(x), y) < (1e-12 if N < 4 else 1e-11)
    assert rel(s.mult_fp32(x), y) < 2e-5
