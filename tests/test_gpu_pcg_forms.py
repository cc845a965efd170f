"""The fused Jacobi and inverse-mass CG iterations: one block and several, sums folded and added by a
kernel in between, iterations launched ahead (small meshes) and one by one, limits that cut a run in the
middle of an eight, restarts, and the vector operator on both sides of the size where its components run
in one launch. The residual of the result is taken under the oracle's operator."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pair(ip, oracle, dim, N, n, mm):
    mesh = ip.Mesh.square(n, jitter=0.1, seed=9) if dim == 2 else ip.Mesh.cube(n, 0.1, 9)
    s = ip.PoissonSolver(mesh, N)
    o = oracle.Oracle(*mesh.arrays(), N)
    if mm:
        s.set_mm_const(mm)
        o.set_mm_const(mm)
    return s, o


@pytest.mark.parametrize("kind", ["jacobi", "scalar", "recp"])
@pytest.mark.parametrize("dim,N,n", [(2, 1, 1), (2, 2, 5), (2, 3, 20), (3, 1, 4), (3, 4, 2), (3, 3, 12), (3, 2, 27),
                                     (3, 3, 27)])
def test_solve_ends_on_the_true_residual(ip, oracle, kind, dim, N, n):
    print(f"pcg {kind} dim={dim} N={N} n={n}", flush=True)
    mm = 1e3 * n * n
    s, o = _pair(ip, oracle, dim, N, n, mm)
    rng = np.random.default_rng(n)
    if kind == "jacobi":
        s.set_solver(ip.SOLVER_JACOBI)
    else:
        s.set_solver(ip.SOLVER_INV_MASS)
        if kind == "scalar":
            s.set_inv_mass_factor(1.0 / mm)
        else:
            s.set_inv_mass_recp_factor(mm * (1.0 + 0.1 * rng.random((s.n_cells, s.Np))))
    s.set_tol_and_iter(1e-9, 0.0, 3000)
    b = rng.standard_normal((s.n_cells, s.Np))
    x = np.zeros_like(b)
    assert s.solve(b, x)
    its = s.last_stats["iterations"]
    # the recursive residual met the tolerance and so did the true one
    assert np.linalg.norm(b - o.mult(x)) <= 1.01e-9 * np.linalg.norm(b)
    assert s.last_stats["fine_applies"] >= its
    y = x.copy()
    assert s.solve(b, y) and s.last_stats["iterations"] == 0 and np.array_equal(x, y)
    # every sum has one order: the same bits again
    y = np.zeros_like(b)
    assert s.solve(b, y) and s.last_stats["iterations"] == its and np.array_equal(x, y)
    # a limit ends the run at its iterate, with the true residual of that iterate reported
    for limit in (1, 5, 8, 13):
        if limit >= its:
            break
        s.set_tol_and_iter(1e-9, 0.0, limit)
        y = np.zeros_like(b)
        assert not s.solve(b, y)
        assert s.last_stats["iterations"] == limit
        r = np.linalg.norm(b - o.mult(y)) / np.linalg.norm(b)
        # both residuals are differences b - A y, relative to |b|: each carries the rounding of its
        # own A y, which the apply's parity bounds by 1e-12 (1e-11 at order 4) of |A y| <= 2 |b| here
        assert abs(s.last_stats["rel_residual"] - r) <= (4e-12 if N < 4 else 4e-11)


def test_breakdown_is_reported(ip):
    """A negative mass factor makes the operator indefinite: p.Ap <= 0 ends the run with its error code."""
    mesh = ip.Mesh.square(6, jitter=0.1, seed=2)
    s = ip.PoissonSolver(mesh, 2)
    s.set_mm_const(-1e9)
    s.set_solver(ip.SOLVER_JACOBI)
    s.set_tol_and_iter(1e-12, 0.0, 100)
    b = np.random.default_rng(0).standard_normal((s.n_cells, s.Np))
    with pytest.raises(ip.InsPoissonError):
        s.solve(b, np.zeros_like(b))


@pytest.mark.parametrize("N,n", [(2, 3), (2, 12), (3, 17), (3, 18), (4, 5), (4, 16)])
@pytest.mark.parametrize("jacobi", [False, True])
def test_vector_solve(ip, oracle, N, n, jacobi):
    print(f"vector pcg N={N} n={n} jacobi={jacobi}", flush=True)
    mesh = ip.Mesh.cube(n, 0.1, 4)
    s = ip.ViscousVecSolver(mesh, N)
    o = oracle.Oracle(*mesh.arrays(), N, faces=mesh.faces())
    t = np.full(s.n_bfaces, 2, dtype=np.int32)
    t[::3] = 0
    t[1::3] = 1
    bct = [t, t, t]
    mm = 1e3 * n * n
    s.set_bc_types(bct)
    s.set_mm_const(mm)
    o.set_mm_const(mm)
    s.set_preconditioner(ip.VEC_PRE_JACOBI if jacobi else ip.VEC_PRE_FACTOR_INV_MASS)
    s.set_inv_mass_factor(1.0 / mm)
    s.set_tol_and_iter(1e-8, 0.0, 2000)
    rng = np.random.default_rng(N)
    u = rng.standard_normal((3, s.n_cells, s.Np))
    want = o.mult_vec(np.stack(bct), u)
    assert np.abs(s.mult(u) - want).max() < (1e-12 if N < 4 else 1e-11) * np.abs(want).max()
    x = np.zeros_like(u)
    assert s.solve(u, x)
    y = np.zeros_like(u)
    assert s.solve(u, y) and np.array_equal(x, y)
    assert np.linalg.norm(u - o.mult_vec(np.stack(bct), x)) <= 1.01e-8 * np.linalg.norm(u)
