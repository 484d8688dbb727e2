"""Many CG steps in one launch against the oracle at its edges: one block and
several, every number of rows per thread, the last block nearly empty, rows
of up to five, seven and nine entries (and ten, which the kernels per step
take), short restart intervals, residual histories, no preconditioner."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def O():
    from oracle import oracle
    return oracle


@pytest.fixture(scope="module")
def spk():
    import sparkit_amd
    sparkit_amd.init(0)
    return sparkit_amd


def _spd(O, n, side):
    """Symmetric, diagonally dominant, `side` entries on each side (multiples
    of 1/8: exact in FP32); rows near the ends are shorter."""
    r, c, v = [np.arange(n)], [np.arange(n)], [np.full(n, 2.5 * side + 0.5)]
    for k in range(1, side + 1):
        o = k * k
        if o >= n:
            break
        w = -((np.arange(n - o) % 7) + 1) / 8.0
        i = np.arange(n - o)
        r += [i, i + o]
        c += [i + o, i]
        v += [w, w]
    return O.make_matrix(n, n, np.concatenate(r), np.concatenate(c), np.concatenate(v))


def _check(O, spk, n, side, prec="f64", steps=8, restart=100, left="jacobi"):
    print("cg", n, side, prec, steps, restart, left, flush=True)
    dt = np.float64 if prec == "f64" else np.float32
    A = _spd(O, n, side)
    b = O.uniform_pm1(n, n).astype(dt).astype(np.float64)
    Ad = spk.CsrMatrix.from_oracle(A)
    x = spk.DeviceVector.zeros(n, dt)
    cfg = spk.CGConfig(0.0, restart, steps, True, spk.F64 if prec == "f64" else spk.F32)
    s = spk.conjugate_gradient(spk.DeviceVector.from_numpy(b, dt), x, cfg, Ad,
                               spk.jacobi(Ad) if left else spk.identity)
    xr, sr = O.cg(A, b, tol=0.0, restart_iterations=restart, max_iterations=steps,
                  left=left)
    assert s.computed_iterations == sr.computed_iterations == steps
    # FP64: dot products in another order.  FP32 against the FP64 iteration
    # (the dot products are FP64 on the device): u = 2^-24 rounds each element
    # about side + 8 times a step, and later steps carry the error on
    tol = 1e-12 if prec == "f64" else (side + 8) * steps * steps * 2.0 ** -24
    err = np.linalg.norm(x.numpy().astype(np.float64) - xr) / np.linalg.norm(xr)
    assert err < tol, err
    h, hr = np.array(s.iteration_residuals), np.array(sr.iteration_residuals)
    assert len(h) == steps and np.allclose(h, hr, rtol=0, atol=10 * tol * hr[0])


@pytest.mark.parametrize("n", [2, 5, 447, 448, 449, 1792, 1793, 5000, 448 * 256,
                               448 * 256 + 1, 448 * 2 * 256 + 1, 448 * 3 * 256 + 1,
                               448 * 4 * 256, 448 * 4 * 256 + 1])
def test_sizes(O, spk, n):
    _check(O, spk, n, 2, steps=min(n - 1, 6))


@pytest.mark.parametrize("side", [1, 3, 4, 5])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_row_lengths(O, spk, side, prec):
    for n in (100, 3000, 250000):
        _check(O, spk, n, side, prec)


@pytest.mark.parametrize("restart", [1, 3, 8])
def test_restarts(O, spk, restart):
    for n in (1000, 60000):
        _check(O, spk, n, 2, steps=20, restart=restart)


def test_no_preconditioner(O, spk):
    _check(O, spk, 7000, 3, left=None)
    _check(O, spk, 7000, 3, "f32", left=None)


def test_stops_where_it_converges(O, spk):
    """Converging between two looks of the host; a second solve goes on from
    the first one's x; the same bits every time."""
    A = O.poisson_2d(70, 61, 0.05)
    b = O.uniform_pm1(3, A.nrows)
    Ad = spk.CsrMatrix.from_oracle(A)
    J, bd = spk.jacobi(Ad), spk.DeviceVector.from_numpy(b)
    cfg = spk.CGConfig(1e-9, 10000, 10000, True)
    xr, sr = O.cg(A, b, tol=1e-9, restart_iterations=10000, max_iterations=10000,
                  left="jacobi")
    runs = []
    for _ in range(2):
        x = spk.DeviceVector.zeros(A.nrows)
        s = spk.conjugate_gradient(bd, x, cfg, Ad, J)
        assert s.converged and abs(s.computed_iterations - sr.computed_iterations) <= 1
        assert len(s.iteration_residuals) == s.computed_iterations
        runs.append((s.computed_iterations, x.numpy()))
    assert runs[0][0] == runs[1][0] and np.array_equal(runs[0][1], runs[1][1])
    assert O.true_relres(A, b, runs[0][1]) < 2e-9
    s = spk.conjugate_gradient(bd, x, cfg, Ad, J)
    assert s.converged and s.computed_iterations <= 2


def test_reliable_updates(O, spk):
    """The FP32 recurrence under FP64 reliable updates, Jacobi and none."""
    A = O.poisson_2d(90, 83, 0.02)
    b = O.uniform_pm1(4, A.nrows)
    Ad, bd = spk.CsrMatrix.from_oracle(A), spk.DeviceVector.from_numpy(b)
    for M in (spk.jacobi(Ad), spk.identity):
        for budget in (100000, 37):
            x = spk.DeviceVector.zeros(A.nrows)
            cfg = spk.IrConfig(1e-11, 100, 1e-1, 0, budget, spk.IR_CG_RELIABLE)
            s = spk.ir_solve(bd, x, cfg, Ad, M)
            rel = O.true_relres(A, b, x.numpy())
            assert abs(rel - s.relres) <= 1e-3 * rel + 1e-14
            if budget == 37:
                assert not s.converged and s.inner_iterations == 37
            else:
                assert s.converged and rel < 1e-11
