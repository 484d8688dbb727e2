"""The one-launch modified Gram-Schmidt step of GMRES / FGMRES against the
oracle at its edges: one block and several (a block holds up to 7,168
elements), the last block nearly empty, every register size, and the sizes
beyond the registers (the sequence of kernels).  A few Arnoldi steps without
restart stay well conditioned: the iterates agree to the rounding of the dot
products (FP64) or of the stored vectors (FP32, against the FP64 oracle)."""
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


def _check(O, spk, n, method, slot, prec, steps, restart):
    print(method, n, slot, prec, flush=True)
    A = O.tridiagonal_matrix(n, -1.25, 2.5, -0.875)  # exact in FP32
    dt = np.float64 if prec == "f64" else np.float32
    b = O.uniform_pm1(n, n).astype(dt).astype(np.float64)
    Ad = spk.CsrMatrix.from_oracle(A)
    M = spk.jacobi(Ad) if slot else spk.identity
    bd = spk.DeviceVector.from_numpy(b, dt)
    x = spk.DeviceVector.zeros(n, dt)
    cfg = spk.GmresConfig(0.0, restart, steps, True,
                          spk.F64 if prec == "f64" else spk.F32)
    kw = dict(tol=0.0, restart_dimension=restart, max_iterations=steps)
    if method == "fgmres":
        s = spk.fgmres(bd, x, cfg, Ad, M)
        xr, sr = O.fgmres(A, b, preconditioner="jacobi" if slot else None, **kw)
    else:
        left = M if slot == "left" else spk.identity
        right = M if slot == "right" else spk.identity
        s = spk.gmres(bd, x, cfg, Ad, left, right)
        xr, sr = O.gmres(A, b, left="jacobi" if slot == "left" else None,
                         right="jacobi" if slot == "right" else None, **kw)
    assert s.computed_iterations == sr.computed_iterations == steps
    # FP64: dot products of n terms in another order, n eps at most, over the
    # steps.  FP32 against the FP64 iteration on the same data (the dot
    # products are FP64 on the device): with u = 2^-24 a step rounds each
    # element about 8 times (3 products, 2 sums, the update, the division, the
    # product with y), and every later step carries the error on
    tol = 1e-12 if prec == "f64" else 8 * steps * steps * 2.0 ** -24
    err = np.linalg.norm(x.numpy().astype(np.float64) - xr) / np.linalg.norm(xr)
    assert err < tol, err
    h, hr = np.array(s.iteration_residuals), np.array(sr.iteration_residuals)
    assert np.allclose(h, hr, rtol=10 * tol, atol=0)


@pytest.mark.parametrize("n", [2, 63, 448, 449, 3583, 7168, 7169, 14337,
                               448 * 4 * 256 - 1, 448 * 8 * 256 + 1])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_sizes(O, spk, n, prec):
    _check(O, spk, n, "gmres", None, prec, min(n - 1, 6), 10)


@pytest.mark.parametrize("n", [448 * 16 * 256 + 5, 448 * 28 * 256, 448 * 28 * 256 + 1])
def test_large_sizes(O, spk, n):
    _check(O, spk, n, "gmres", "right", "f64", 3, 5)


@pytest.mark.parametrize("method,slot", [("gmres", "left"), ("gmres", "right"),
                                         ("fgmres", "right"), ("fgmres", None)])
@pytest.mark.parametrize("n", [1000, 20000])
def test_jacobi_slots_and_restarts(O, spk, method, slot, n):
    """The fused Jacobi products, over restarts and a last partial cycle."""
    for prec in ("f64", "f32"):
        _check(O, spk, n, method, slot, prec, 7, 3)


def test_many_columns(O, spk):
    """The largest restart dimension of the one-launch step, and beyond."""
    for restart in (512, 513):
        _check(O, spk, 3000, "gmres", "left", "f64", 40, restart)
