"""Device vectors in the solver's own layout: the passes run on the caller's arrays. The results must
equal the host-layout call bit for bit, whatever the inputs' padding holds; the outputs' padding is
cleared; outputs that are (or overlap) inputs give the same results as separate ones."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _device(x, stride, shift=0):
    """cells x rows host array -> device SoA, padding NaN, `shift` doubles into its allocation."""
    a = np.full((x.shape[1], stride), np.nan)
    a[:, :x.shape[0]] = x.T
    buf = torch.full((a.size + shift,), float("nan"), dtype=torch.float64, device="cuda")
    t = buf[shift:].view(a.shape)
    t.copy_(torch.from_numpy(a))
    torch.cuda.synchronize()
    return t


def _same(t, x):
    h = t.cpu().numpy()
    assert np.array_equal(h[:, :x.shape[0]].T, x)
    assert not h[:, x.shape[0]:].any()


def _solver(ip, dim, N):
    # 3^3 x 6 = 162 and 2 x 11^2 = 242 cells: padding inside the last block of 256 and past it
    mesh = ip.Mesh.square(11, jitter=0.1, seed=3) if dim == 2 else ip.Mesh.cube(3, 0.1, 3)
    s = ip.PoissonSolver(mesh, N)
    s.set_solver(ip.SOLVER_JACOBI)
    s.set_factor(1.0 + np.random.default_rng(N).random((s.n_cells, s.Np)))
    s.init()
    return s


@pytest.mark.parametrize("dim,N", [(2, 1), (2, 4), (3, 1), (3, 2), (3, 4)])
@pytest.mark.parametrize("fp32", [False, True])
def test_mult_on_the_callers_vectors(ip, dim, N, fp32):
    s = _solver(ip, dim, N)
    x = np.random.default_rng(7).standard_normal((s.n_cells, s.Np))
    fn = s.mult_fp32 if fp32 else s.mult
    want = fn(x)
    for shift in (0, 1):  # 16-byte aligned and not
        a, b = _device(x, s.stride, shift), _device(np.zeros_like(x), s.stride, shift)
        fn((a.data_ptr(), b.data_ptr()), layout=ip.LAYOUT_DEVICE_SOA)
        _same(b, want)
    fn((a.data_ptr(), a.data_ptr()), layout=ip.LAYOUT_DEVICE_SOA)  # in place
    _same(a, want)


@pytest.mark.parametrize("dim,N", [(2, 1), (2, 3), (3, 1), (3, 3), (3, 4)])
def test_projection_on_the_callers_vectors(ip, dim, N):
    s = _solver(ip, dim, N)
    rng = np.random.default_rng(dim + N)
    p, u = rng.standard_normal((s.n_cells, s.Np)), rng.standard_normal((dim, s.n_cells, s.Np))
    dt = 0.01
    want, grad = s.project_velocity(dt, p, u), s.grad_central(p)

    def call(pd, ud, od):
        ptr = lambda t: [v.data_ptr() for v in t] + [None] * (3 - dim)  # noqa: E731
        if ud is None:
            rc = ip.lib.ins_poisson_grad_central(s._h, pd.data_ptr(), *ptr(od), ip.LAYOUT_DEVICE_SOA)
        else:
            rc = ip.lib.ins_poisson_project_velocity(s._h, dt, pd.data_ptr(), *ptr(ud), *ptr(od),
                                                     ip.LAYOUT_DEVICE_SOA)
        assert rc == ip.OK, ip.lib.ins_poisson_last_error().decode()

    dev = lambda v: _device(v, s.stride)  # noqa: E731
    pd, ud, od = dev(p), [dev(v) for v in u], [dev(v) for v in u]
    call(pd, ud, od)
    for t, w in zip(od, want):
        _same(t, w)
    call(pd, None, od)
    for t, w in zip(od, grad):
        _same(t, w)
    call(pd, ud, ud)  # each component in place
    for t, w in zip(ud, want):
        _same(t, w)
    ud = [dev(v) for v in u]
    call(pd, ud, ud[1:] + ud[:1])  # outputs that are other components' inputs
    for t, w in zip(ud[1:] + ud[:1], want):
        _same(t, w)
    ud = [dev(v) for v in u]
    call(pd, ud, [pd] + od[1:])  # an output over the pressure
    _same(pd, want[0])


@pytest.mark.parametrize("fp32", [False, True])
def test_pinned_host_vectors_go_through_the_copies(ip, fp32):
    """Memory that is not the GPU's own is copied, as every vector once was, with the same results."""
    s = _solver(ip, 3, 2)
    x = np.random.default_rng(7).standard_normal((s.n_cells, s.Np))
    fn = s.mult_fp32 if fp32 else s.mult
    want = fn(x)
    pinned = torch.empty((s.Np, s.stride), dtype=torch.float64, pin_memory=True)
    dev = _device(x, s.stride)
    pinned.copy_(dev)
    torch.cuda.synchronize()
    out = torch.full_like(dev, float("nan"))
    torch.cuda.synchronize()
    fn((pinned.data_ptr(), out.data_ptr()), layout=ip.LAYOUT_DEVICE_SOA)
    _same(out, want)
    fn((dev.data_ptr(), pinned.data_ptr()), layout=ip.LAYOUT_DEVICE_SOA)
    _same(pinned, want)
