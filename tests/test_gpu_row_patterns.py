"""SpMVs of stores whose rows repeat a few lists of entries (131,072 rows and
9 MiB of entries and more), bit for bit against the oracle: stencils on ragged grids, sizes around
the kernel's blocks, empty and odd rows, the largest number of lists and one
more, the longest rows and longer ones, signed zeros, infinities and NaNs in
the values and in x, FP32, the fused dot product, FP16 values and the other
layouts beside it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 1 << 20
FEW = 1 << 17  # rows below which no lists are looked for


@pytest.fixture(scope="module")
def O():
    from oracle import oracle
    return oracle


@pytest.fixture(scope="module")
def spk():
    import sparkit_amd
    sparkit_amd.init(0)
    return sparkit_amd


class _Csr:
    def __init__(self, nrows, rp, ci, v):
        self.nrows = self.ncols = nrows
        self.row_ptr, self.col_ind, self.vals = rp, ci, v


def _rows(n, lists, which):
    """Row i holds lists[which[i]] = (offsets, values), clipped to the matrix."""
    length = np.array([len(o) for o, _ in lists])[which]
    row = np.repeat(np.arange(n), length)
    offs = np.concatenate([lists[w][0] for w in which]) if n < 5000 else None
    if offs is None:
        width = max(len(o) for o, _ in lists)
        ot = np.zeros((len(lists), width), np.int64)
        vt = np.zeros((len(lists), width))
        for k, (o, v) in enumerate(lists):
            ot[k, :len(o)], vt[k, :len(o)] = o, v
        keep = np.arange(width)[None, :] < length[:, None]
        offs, vals = ot[which][keep], vt[which][keep]
    else:
        vals = np.concatenate([lists[w][1] for w in which])
    col = row + offs
    ok = (col >= 0) & (col < n)
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(row[ok], minlength=n), out=rp[1:])
    return _Csr(n, rp, col[ok], vals[ok])


def _reference(A, x):
    """Storage-order sums of separately rounded products, in x's precision."""
    v = A.vals.astype(x.dtype)
    y = np.zeros(A.nrows, x.dtype)
    length = np.diff(A.row_ptr)
    with np.errstate(all="ignore"):
        for k in range(int(length.max(initial=0))):
            has = length > k
            p = A.row_ptr[:-1][has] + k
            y[has] = y[has] + v[p] * x[A.col_ind[p]]
    return y


def _check(spk, A, x=None, label=""):
    print("patterns", label, A.nrows, len(A.col_ind), flush=True)
    Ad = spk.CsrMatrix.from_oracle(A)
    if x is None:
        x = np.random.default_rng(7).uniform(-1, 1, A.nrows)
    for dt in (np.float64, np.float32):
        xd = spk.DeviceVector.from_numpy(x, dt)
        y, yd = spk.DeviceVector.zeros(A.nrows, dt), spk.DeviceVector.zeros(A.nrows, dt)
        out = spk.DeviceVector.zeros(1)
        ref = _reference(A, x.astype(dt))
        Ad.spmv(xd, y)
        assert np.array_equal(y.numpy(), ref, equal_nan=True)
        Ad.spmv_dot(xd, yd, out)
        assert np.array_equal(yd.numpy(), ref, equal_nan=True)
        real = ~np.isnan(ref)  # signed zeros too
        for z in (y, yd):
            assert np.array_equal(np.signbit(z.numpy()[real]), np.signbit(ref[real]))
        if np.isfinite(ref).all():
            d = float(np.dot(x.astype(dt).astype(np.float64), ref.astype(np.float64)))
            scale = float(np.dot(np.abs(x), np.abs(ref.astype(np.float64))))
            assert abs(out.numpy()[0] - d) <= 1e-12 * scale + 1e-300
    return Ad


STENCIL = [(np.array([-300, -1, 0, 1, 300]), np.array([-1.5, -1.0, 6.0, -0.5, -1.25]))]


@pytest.mark.parametrize("n", [FEW - 1, FEW, FEW + 1, 157285, 157286, 157287, 235930, 235931,
                               1024 * 250 - 1, 1024 * 250, 1024 * 250 + 1,
                               1024 * 4096, 1024 * 4096 + 1, 2048 * 2053 + 1])
def test_sizes(spk, n):
    """157,286 and 235,930 rows: about 9 MiB of FP64 and of FP32 entries."""
    _check(spk, _rows(n, STENCIL, np.zeros(n, int)), label="band")


@pytest.mark.parametrize("dims", [(64, 64, 64), (101, 73, 41), (7, 301, 131)])
def test_stencils(O, spk, dims):
    A = O.convdiff_3d(*dims, 1.0, 0.3, 0.2, 0.1)
    Ad = _check(spk, A, label=str(dims))
    x = O.uniform_pm1(3, A.nrows)
    xd, y = spk.DeviceVector.from_numpy(x), spk.DeviceVector.zeros(A.nrows)
    ref = O.spmv(A, x)
    Ad.spmv(xd, y)
    assert np.array_equal(y.numpy(), ref)
    Ad.set_panels(4)  # the other layouts keep their own stores
    Ad.spmv(xd, y)
    assert np.allclose(y.numpy(), ref, rtol=0, atol=1e-14 * 50)
    Ad.set_panels(1)
    Ad.spmv(xd, y)
    assert np.array_equal(y.numpy(), ref)
    # FP16 values for FP32 products: not the lists' FP32 ones
    Ad.set_half_values(True)
    y32 = spk.DeviceVector.zeros(A.nrows, np.float32)
    Ad.spmv(spk.DeviceVector.from_numpy(x, np.float32), y32)
    B = _Csr(A.nrows, A.row_ptr, A.col_ind,
             A.vals.astype(np.float32).astype(np.float16).astype(np.float64))
    assert np.array_equal(y32.numpy(), _reference(B, x.astype(np.float32)))


@pytest.mark.parametrize("width", [1, 5, 6, 7, 8, 9, 10, 15, 16, 20])
def test_row_lengths(spk, width):
    """Up to 15 entries a row; empty and shorter rows among them."""
    rng = np.random.default_rng(width)
    off = np.sort(rng.choice(np.arange(-400, 400), width, replace=False))
    lists = [(off, rng.uniform(-1, 1, width)), (off[:0], np.zeros(0)),
             (off[:width // 2], rng.uniform(-1, 1, width // 2))]
    which = rng.integers(0, 3, N + 77)
    A = _rows(N + 77, lists, which)
    if width < 16:
        _check(spk, A, label="width %d" % width)
    else:  # several lanes a row: another association of the sum
        Ad = spk.CsrMatrix.from_oracle(A)
        x = rng.uniform(-1, 1, A.nrows)
        y = spk.DeviceVector.zeros(A.nrows)
        Ad.spmv(spk.DeviceVector.from_numpy(x), y)
        assert np.allclose(y.numpy(), _reference(A, x), rtol=0, atol=1e-14 * width)


@pytest.mark.parametrize("count", [254, 255, 256, 400])
def test_number_of_lists(spk, count):
    """Lists that differ in one value; the first and last rows are clipped and
    add lists of their own."""
    lists = [(np.array([0, 1]), np.array([1.0 + k, -0.5])) for k in range(count)]
    which = np.arange(N + 5) % count
    _check(spk, _rows(N + 5, lists, which), label="%d lists" % count)


def test_one_row_differs(spk):
    """A single row with another value, column or length."""
    n = N + 1000
    for odd in ((np.array([-300, -1, 0, 1, 300]), np.array([-1.5, -1.0, 6.0, -0.5, -1.26])),
                (np.array([-300, -1, 0, 1, 301]), STENCIL[0][1]),
                (np.array([-300, -1, 0]), STENCIL[0][1][:3])):
        which = np.zeros(n, int)
        which[n // 2 + 3] = 1
        _check(spk, _rows(n, STENCIL + [odd], which), label="odd row")


def test_special_values(spk):
    """Signed zeros, infinities and NaNs in the values and in x; entries a row
    does not have read nothing into its sum."""
    rng = np.random.default_rng(5)
    n = N + 3
    lists = [(np.array([-2, 0, 1]), np.array([-0.0, 2.0, -0.0])),
             (np.array([0]), np.array([-0.0])),
             (np.array([-1, 0]), np.array([np.inf, 1.0])),
             (np.array([0, 3]), np.array([np.nan, 1.0])),
             (np.array([5]), np.array([1e-300]))]
    which = rng.integers(0, 5, n)
    x = rng.uniform(-1, 1, n)
    x[::101] = np.inf
    x[50::103] = np.nan
    x[7::11] = -0.0
    _check(spk, _rows(n, lists, which), x, "special")


def test_rectangular_and_small(spk):
    """Not square, or fewer rows: the row kernel, same sums."""
    A = _rows(FEW - 500, STENCIL, np.zeros(FEW - 500, int))
    _check(spk, A, label="small")
    R = spk.CsrMatrix.from_host(A.nrows, A.ncols + 9, A.row_ptr, A.col_ind, A.vals)
    x = np.random.default_rng(1).uniform(-1, 1, A.ncols + 9)
    y = spk.DeviceVector.zeros(A.nrows)
    R.spmv(spk.DeviceVector.from_numpy(x), y)
    assert np.array_equal(y.numpy(), _reference(A, x[:A.ncols]))


@pytest.mark.parametrize("solver", ["cg", "bicg", "bicgstab", "cgs", "minres", "qmr"])
@pytest.mark.parametrize("left", [None, "jacobi"])
def test_solvers(O, spk, solver, left):
    """Every solver's products, transposed ones too, and the sums in their
    epilogues, over stores with row patterns; CG at a size whose rows do not
    fit the registers."""
    print("patterned", solver, left, flush=True)
    A = (O.poisson_3d(90, 80, 75) if solver in ("cg", "minres")
         else O.convdiff_3d(61, 63, 67, 1.0, 0.3, 0.2, 0.1))
    b = O.uniform_pm1(9, A.nrows)
    Ad = spk.CsrMatrix.from_oracle(A)
    bd, x = spk.DeviceVector.from_numpy(b), spk.DeviceVector.zeros(A.nrows)
    M = spk.jacobi(Ad) if left else spk.identity
    steps = 8
    if solver == "cg":
        s = spk.conjugate_gradient(bd, x, spk.CGConfig(0.0, 100, steps, True), Ad, M)
        xr, sr = O.cg(A, b, tol=0.0, restart_iterations=100, max_iterations=steps, left=left)
    else:
        mats = (Ad, Ad.transpose()) if solver in ("bicg", "qmr") else (Ad,)
        s = getattr(spk, solver)(bd, x, spk.BicgstabConfig(0.0, steps, True), *mats, M)
        xr, sr = getattr(O, solver)(A, b, tol=0.0, max_iterations=steps, left=left)
    assert s.computed_iterations == sr.computed_iterations
    # the dot products in another order (2^-53 a term), eight steps of a
    # well-conditioned start
    assert np.linalg.norm(x.numpy() - xr) <= 1e-11 * np.linalg.norm(xr)
    assert np.allclose(s.iteration_residuals, sr.iteration_residuals, rtol=1e-11, atol=0)
