"""ILU(0) factorization and triangular sweeps in tiles, bit for bit against
the oracle where the layout can go wrong: sizes around a tile (2,048 rows)
and a block (4 tiles), chains inside a tile and across tiles, rows wider than
a batch of four entries, rows too long for the short and for the tiled
factorization, rows of very different lengths in one level, rows given in
another order than ascending."""
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


def _banded(O, n, offsets, seed=1):
    """Diagonally dominant, entries at the given column offsets."""
    rng = np.random.default_rng(seed)
    r, c, v = [np.arange(n)], [np.arange(n)], [np.full(n, 2.0 * len(offsets) + 2)]
    for o in offsets:
        i = np.arange(max(0, -o), min(n, n - o))
        r.append(i)
        c.append(i + o)
        v.append(rng.uniform(-1, 1, len(i)))
    return O.make_matrix(n, n, np.concatenate(r), np.concatenate(c), np.concatenate(v))


def _arrow(O, n, width):
    """Two rows and columns of `width` entries among rows of three."""
    rng = np.random.default_rng(3)
    rows, cols = [np.arange(n), np.arange(1, n), np.arange(n - 1)], \
                 [np.arange(n), np.arange(n - 1), np.arange(1, n)]
    far = rng.choice(n - 2, width, replace=False)
    for i in (n // 2, n - 1):
        rows += [np.full(width, i), far]
        cols += [far, np.full(width, i)]
    r, c = np.concatenate(rows), np.concatenate(cols)
    v = np.where(r == c, 4.0 * width, rng.uniform(-1, 1, len(r)))
    return O.make_matrix(n, n, r, c, v)


def _check(O, spk, A, modified=False):
    Lr, Ur = O.ilu0(A, modified)
    Ad = spk.CsrMatrix.from_oracle(A)
    F = (spk.milu0 if modified else spk.ilu0)(Ad)
    r = O.uniform_pm1(5, A.nrows)
    rd = spk.DeviceVector.from_numpy(r)
    y, z = spk.DeviceVector.zeros(A.nrows), spk.DeviceVector.zeros(A.nrows)
    y_ref = O.forward_solve(Lr, r)
    z_ref = O.backward_solve(Ur, y_ref)
    for _ in range(2):  # the second application finds the first one's scratch
        spk.ilu_apply(F, rd, z)
        assert np.array_equal(z.numpy(), z_ref)
    F.forward(rd, y)
    assert np.array_equal(y.numpy(), y_ref)
    F.backward(y, z)
    assert np.array_equal(z.numpy(), z_ref)
    zz = spk.DeviceVector.from_numpy(r)  # in place
    F.apply(zz, zz)
    assert np.array_equal(zz.numpy(), z_ref)
    z32 = spk.DeviceVector.zeros(A.nrows, np.float32)
    F.apply(spk.DeviceVector.from_numpy(r, np.float32), z32)
    # FP32 factors and vector: a few roundings of 2^-24 per entry; the
    # matrices are diagonally dominant, so errors do not grow
    assert np.linalg.norm(z32.numpy() - z_ref) <= 1e-5 * np.linalg.norm(z_ref)
    (lrp, lci, lv), (urp, uci, uv) = F.factors()
    assert np.array_equal(lci, Lr.col_ind) and np.array_equal(lv, Lr.vals)
    assert np.array_equal(uci, Ur.col_ind) and np.array_equal(uv, Ur.vals)


@pytest.mark.parametrize("n", [2, 3, 64, 65, 2047, 2048, 2049, 8191, 8192, 8193, 20000])
def test_chain(O, spk, n):
    """One row a level: every step a single lane."""
    print("chain", n, flush=True)
    _check(O, spk, _banded(O, n, (-1, 1)))


@pytest.mark.parametrize("offsets", [(-2049, 2049), (-8192, -1, 1, 8192), (-100, 3),
                                     (-9000, -5000, -2000, -1, 1, 2000, 5000, 9000)])
def test_dependencies_across_tiles(O, spk, offsets):
    print("offsets", offsets, flush=True)
    for modified in (False, True):
        _check(O, spk, _banded(O, 18001, offsets), modified)


@pytest.mark.parametrize("side", [4, 5, 8, 15, 16])
def test_wide_rows(O, spk, side):
    """4: the short factorization's widest rows; 15: the tiled one's (31
    entries); 16: a launch per level."""
    print("side", side, flush=True)
    near = [k * k + k - 1 for k in range(1, side + 1)]
    _check(O, spk, _banded(O, 5000, [-k for k in near] + near))


@pytest.mark.parametrize("width", [10, 300])
def test_mixed_lengths(O, spk, width):
    print("arrow", width, flush=True)
    _check(O, spk, _arrow(O, 4500, width))


def test_ragged_grids(O, spk):
    for dims in ((13, 11, 9), (45, 3, 31), (100, 37, 3)):
        print("grid", dims, flush=True)
        for modified in (False, True):
            _check(O, spk, O.convdiff_3d(*dims, 1.0, 0.3, 0.2, 0.1), modified)


def test_diagonal_matrix(O, spk):
    """No dependencies: one level."""
    _check(O, spk, _banded(O, 5000, ()))


def test_rows_in_another_order(O, spk):
    """A store whose rows list their columns descending: the factors are
    those of the ascending one."""
    A = O.convdiff_3d(9, 8, 7, 1.0, 0.3, 0.2, 0.1)
    ci, v = np.array(A.col_ind), np.array(A.vals)
    for i in range(A.nrows):
        s = slice(A.row_ptr[i], A.row_ptr[i + 1])
        ci[s], v[s] = ci[s][::-1], v[s][::-1]
    F = spk.ilu0(spk.CsrMatrix.from_host(A.nrows, A.ncols, A.row_ptr, ci, v))
    G = spk.ilu0(spk.CsrMatrix.from_oracle(A))
    for a, b in zip(F.factors(), G.factors()):
        for p, q in zip(a, b):
            assert np.array_equal(p, q)


@pytest.fixture
def sweep_wait(spk):
    from sparkit_amd import _lib

    def limit(ticks):
        _lib.call("spk_set_sweep_wait", ticks)
    yield limit
    limit(0)


@pytest.mark.parametrize("offsets,n,ms", [((-1, 1), 20480, 2),
                                          (tuple(range(-12, 0)) + tuple(range(1, 13)), 6200, 40)])
def test_a_long_chain_is_no_stall(O, spk, sweep_wait, offsets, n, ms):
    """Waits of the last tiles last several times the limit (a tile of 2,048
    dependent rows takes 5 ms to factor, 135 ms with 25 entries a row, 0.6 to
    sweep), in which the tiles before them get on."""
    print("chain", n, "limit", ms, "ms", flush=True)
    A = _banded(O, n, offsets)
    sweep_wait(ms * 100000)
    _check(O, spk, A)


@pytest.mark.parametrize("modified", [False, True])
def test_waits_that_are_given_up(O, spk, sweep_wait, modified):
    """The construction is done again without waits; a sweep says so, and the
    next one is right."""
    print("given up", modified, flush=True)
    A = _banded(O, 20480, (-1, 1))
    Lr, Ur = O.ilu0(A, modified)
    r = O.uniform_pm1(5, A.nrows)
    rd, z = spk.DeviceVector.from_numpy(r), spk.DeviceVector.zeros(A.nrows)
    Ad = spk.CsrMatrix.from_oracle(A)
    sweep_wait(1)
    F = (spk.milu0 if modified else spk.ilu0)(Ad)
    with pytest.raises(spk.SpkError, match="bounded wait"):
        F.apply(rd, z)
    sweep_wait(0)
    assert F.levels() == (A.nrows, A.nrows)
    (lrp, lci, lv), (urp, uci, uv) = F.factors()
    assert np.array_equal(lv, Lr.vals) and np.array_equal(uv, Ur.vals)
    z_ref = O.backward_solve(Ur, O.forward_solve(Lr, r))
    for _ in range(2):
        F.apply(rd, z)
        assert np.array_equal(z.numpy(), z_ref)


def _grid(O, nx, ny, order, points):
    """A 5- or 9-point stencil, its rows in the given order."""
    i = np.arange(nx * ny).reshape(nx, ny)
    x, y = np.indices(i.shape)
    key = {"two colours": (x + y) % 2, "four colours": x % 2 * 2 + y % 2,
           "random": np.random.default_rng(nx).permutation(i.size).reshape(i.shape)}[order]
    at = np.empty(i.size, np.int64)
    at[np.argsort(key.ravel(), kind="stable")] = np.arange(i.size)
    r, c = [at], [at]
    pairs = [(i[1:], i[:-1]), (i[:, 1:], i[:, :-1])]
    if points == 9:
        pairs += [(i[1:, 1:], i[:-1, :-1]), (i[1:, :-1], i[:-1, 1:])]
    for p, q in pairs:
        r += [at[p.ravel()], at[q.ravel()]]
        c += [at[q.ravel()], at[p.ravel()]]
    r, c = np.concatenate(r), np.concatenate(c)
    return O.make_matrix(i.size, i.size, r, c,
                         np.where(r == c, points + 0.0, -0.5 - (r + c) % 7 / 14.0))


@pytest.mark.parametrize("order,points", [("two colours", 5), ("four colours", 9),
                                          ("random", 5), ("random", 9)])
@pytest.mark.parametrize("nx,ny", [(9, 7), (64, 64), (64, 65), (255, 257), (256, 256),
                                   (300, 230)])
def test_few_levels(O, spk, order, points, nx, ny):
    """Around three tiles (4,096 rows) and 65,536 rows, where the sweeps
    change from tiles to a window of levels to a launch per level."""
    print("few levels", order, points, nx, ny, flush=True)
    A = _grid(O, nx, ny, order, points)
    _check(O, spk, A, modified=points == 9)
    F = spk.ilu0(spk.CsrMatrix.from_oracle(A))
    L, U = O.ilu0(A)
    r = O.uniform_pm1(3, A.nrows)
    rd, z = spk.DeviceVector.from_numpy(r), spk.DeviceVector.zeros(A.nrows)
    z_ref = O.backward_solve(U, O.forward_solve(L, r))
    for schedule in ("sync-free", "levels", "auto", "levels", "sync-free"):
        F.schedule = schedule
        for _ in range(2):
            F.apply(rd, z)
            assert np.array_equal(z.numpy(), z_ref)


def _ikj(rp, ci, v, modified):
    """ilu0 of rows that may repeat columns: the first diagonal is the pivot."""
    n, w = len(rp) - 1, np.array(v)
    dp = [rp[i] + list(ci[rp[i]:rp[i + 1]]).index(i) for i in range(n)]
    for i in range(n):
        dropped = 0.0
        for p in range(rp[i], rp[i + 1]):
            k = ci[p]
            if k >= i:
                break
            w[p] = w[p] / w[dp[k]]
            pi = p + 1
            for q in range(dp[k] + 1, rp[k + 1]):
                while pi < rp[i + 1] and ci[pi] < ci[q]:
                    pi += 1
                if pi < rp[i + 1] and ci[pi] == ci[q]:
                    w[pi] = w[pi] - w[p] * w[q]
                elif modified:
                    dropped = dropped + w[p] * w[q]
        if modified:
            w[dp[i]] = w[dp[i]] - dropped
    return w, dp


@pytest.mark.parametrize("modified", [False, True])
def test_repeated_diagonal(O, spk, modified):
    """Rows 5, 50 and 300 have their diagonal twice: factors, forward sweep
    and Jacobi sweeps as ever; the backward solve is refused, on every
    schedule, and at once."""
    A = _banded(O, 400, (-20, -1, 1, 20))
    twice = [5, 50, 300]
    rp, ci, v = [0], [], []
    for i in range(A.nrows):
        s = slice(A.row_ptr[i], A.row_ptr[i + 1])
        for c, x in zip(A.col_ind[s], A.vals[s]):
            ci += [c, c] if c == i and i in twice else [c]
            v += [x, 0.25] if c == i and i in twice else [x]
        rp.append(len(ci))
    rp, ci, v = np.array(rp), np.array(ci), np.array(v)
    F = (spk.milu0 if modified else spk.ilu0)(
        spk.CsrMatrix.from_host(A.nrows, A.nrows, rp, ci, v))
    w, dp = _ikj(rp, ci, v, modified)
    (lrp, lci, lv), (urp, uci, uv) = F.factors()
    for i in range(A.nrows):
        assert np.array_equal(lv[lrp[i]:lrp[i + 1] - 1], w[rp[i]:dp[i]])
        assert np.array_equal(uv[urp[i]:urp[i + 1]], w[dp[i]:rp[i + 1]])
        assert np.array_equal(uci[urp[i]:urp[i + 1]], ci[dp[i]:rp[i + 1]])
    r = O.uniform_pm1(3, A.nrows)
    rd, y = spk.DeviceVector.from_numpy(r), spk.DeviceVector.zeros(A.nrows)
    for schedule in ("auto", "sync-free", "levels"):
        F.schedule = schedule
        F.forward(rd, y)
        x = np.array(r)
        for i in range(A.nrows):
            for p in range(lrp[i], lrp[i + 1] - 1):
                x[i] = x[i] - lv[p] * x[lci[p]]
        assert np.array_equal(y.numpy(), x)
        for call in (F.apply, F.backward):
            with pytest.raises(spk.InvalidArgument, match="diagonal"):
                call(rd, y)
    F.jacobi_sweeps = 1
    F.apply(rd, y)
    d = uv[urp[:-1]]
    low, up = np.array(r), np.zeros(A.nrows)
    for i in range(A.nrows):
        low[i] -= lv[lrp[i]:lrp[i + 1] - 1] @ r[lci[lrp[i]:lrp[i + 1] - 1]]
    for i in range(A.nrows):
        p = slice(urp[i] + 1, urp[i + 1])
        up[i] = (low[i] - uv[p] @ (low / d)[uci[p]]) / d[i]
    assert np.allclose(y.numpy(), up, rtol=1e-13, atol=1e-14)
