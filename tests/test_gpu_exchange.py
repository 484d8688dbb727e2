"""Solves whose kernels exchange sums between blocks, when an exchange does
not go through: the wait is cut to one poll, which finds slots that are still
to be written.  The solve is taken back and done by the kernels per step;
nothing of the lost launches is left in x, the history, the counts or later
solves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def hindered(spk):
    from sparkit_amd import _lib

    def on(yes):
        _lib.call("spk_set_exchange_polls", 1 if yes else 0)
    yield on
    on(False)


def _thrice(hindered, solve):
    """solve() undisturbed, hindered and undisturbed again."""
    a = solve()
    hindered(True)
    b = solve()
    hindered(False)
    c = solve()
    assert np.array_equal(a[1], c[1]) and a[0] == c[0]
    return a, b


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("restart", [1000, 7])
@pytest.mark.parametrize("noalloc", [False, True])
def test_cg(spk, hindered, prec, restart, noalloc):
    A = spk.poisson_2d(300, 200, 0.05)
    dt = np.float64 if prec == "f64" else np.float32
    b = spk.uniform_pm1(3, A.nrows).astype(dt) if prec == "f32" else spk.uniform_pm1(3, A.nrows)
    J, x0 = spk.jacobi(A), np.linspace(-1, 1, A.nrows).astype(dt)
    cfg = spk.CGConfig(0.0, restart, 20, True, spk.F64 if prec == "f64" else spk.F32)
    spk.conjugate_gradient(b, spk.DeviceVector.from_numpy(x0), cfg, A, J)  # FP32 copies
    run = spk.conjugate_gradient_noalloc if noalloc else spk.conjugate_gradient

    def solve():
        x = spk.DeviceVector.from_numpy(x0)
        s = run(b, x, cfg, A, J)
        return (s.computed_iterations, tuple(s.iteration_residuals)), x.numpy()
    (a, xa), (h, xh) = _thrice(hindered, solve)
    assert a[0] == h[0] == 20 and len(h[1]) == 20
    # the dot products' order differs, and for FP32 the roundings of 20 steps
    tol = 1e-12 if prec == "f64" else 20 * 20 * 12 * 2.0 ** -24
    assert np.allclose(a[1], h[1], rtol=0, atol=tol * a[1][0])
    assert np.linalg.norm(xa - xh) <= tol * np.linalg.norm(xa)


def test_reliable_cg(spk, hindered):
    A = spk.poisson_2d(300, 200, 0.05)
    b, J = spk.uniform_pm1(3, A.nrows), spk.jacobi(A)
    cfg = spk.IrConfig(1e-11, 100, 1e-1, 0, 100000, spk.IR_CG_RELIABLE)

    def solve():
        x = spk.DeviceVector.zeros(A.nrows)
        s = spk.ir_solve(b, x, cfg, A, J)
        assert s.converged and spk.true_relres(A, b, x) < 1e-11
        return s.inner_iterations, x.numpy()
    (a, xa), (h, xh) = _thrice(hindered, solve)
    assert abs(a - h) <= 0.1 * a


def test_reliable_cg_budget(spk):
    """A budget of more than one launch's 4,096 steps, undisturbed and lost: it
    is charged with the steps that were kept."""
    from sparkit_amd import _lib
    A = spk.poisson_2d(300, 200, 0.05)
    b, J = spk.uniform_pm1(3, A.nrows), spk.jacobi(A)
    cfg = spk.IrConfig(1e-300, 1, 1e-300, 0, 5000, spk.IR_CG_RELIABLE)  # no update due
    for polls in (0, 1):
        _lib.call("spk_set_exchange_polls", polls)
        try:
            x = spk.DeviceVector.zeros(A.nrows)
            s = spk.ir_solve(b, x, cfg, A, J)
        finally:
            _lib.call("spk_set_exchange_polls", 0)
        assert s.inner_iterations == 5000 and not s.converged
        assert spk.true_relres(A, b, x) < 1e-5  # what FP32 reaches


@pytest.mark.parametrize("precond", ["none", "jacobi", "ilu0", "inner cg"])
def test_gmres(spk, hindered, precond):
    """An inner CG shares the exchange with the outer solver's steps."""
    A = (spk.poisson_2d(300, 200, 0.05) if precond == "inner cg"
         else spk.convdiff_3d(40, 41, 42, 1.0, 5.0, 3.0, 1.0))
    b = spk.uniform_pm1(3, A.nrows)
    M = {"none": lambda: spk.identity, "jacobi": lambda: spk.jacobi(A),
         "ilu0": lambda: spk.ilu0(A),
         "inner cg": lambda: spk.inner_cg(A, spk.jacobi(A), 6, 0.0, spk.F64)}[precond]()
    solver = spk.gmres if precond == "none" else spk.fgmres
    args = (A, M) if solver is spk.fgmres else (A,)
    cfg = spk.GmresConfig(0.0, 10, 25, True)  # three cycles

    def solve():
        x = spk.DeviceVector.from_numpy(np.linspace(-1, 1, A.nrows))
        s = solver(b, x, cfg, *args)
        return (s.computed_iterations, tuple(s.iteration_residuals)), x.numpy()
    (a, xa), (h, xh) = _thrice(hindered, solve)
    assert a[0] == h[0] == 25
    assert np.allclose(a[1], h[1], rtol=0, atol=1e-12 * a[1][0])
    assert np.linalg.norm(xa - xh) <= 1e-10 * np.linalg.norm(xa)
