"""Learned-SPAI training takes the matrices of a batch through each pass
together, in groups: sizes around the 64-row tiles and 256-row blocks, more
matrices than one group holds, a matrix larger than a group, and row forms
(short rows, one-sided rows)."""
import numpy as np
import pytest
import scipy.sparse as sp

from test_gpu_spai import rand_params

pytestmark = pytest.mark.gpu


def band(n, seed, keep=0.8):
    """n rows, up to four entries on each side of the diagonal at random
    distances, positive diagonal."""
    rng = np.random.default_rng(seed)
    dist = np.unique(rng.integers(1, max(2, n), 4))
    d = [sp.diags(rng.uniform(1.0, 2.0, n))]
    for k in dist:
        for s in (-1, 1):
            if k < n:
                v = rng.uniform(-0.3, 0.3, n - k) * (rng.random(n - k) < keep)
                d.append(sp.diags(v, s * int(k), shape=(n, n)))
    A = sp.csr_matrix(sum(d))
    A.eliminate_zeros()
    A.sort_indices()
    return A


def store(spk, A):
    return spk.CsrMatrix.from_host(A.shape[0], A.shape[1], A.indptr, A.indices, A.data)


SIZES = [2, 3, 63, 64, 65, 255, 256, 257, 1000, 4097]


@pytest.mark.parametrize("sizes", [[2], [65], [64, 2], SIZES, SIZES * 2 + [70000],
                                   [300000, 5, 400000, 257, 400000]])
def test_batch_is_the_weighted_sum_of_its_matrices(spk, sizes):
    """One step over a batch: its loss is the matrices' losses weighted by
    their rows, its gradient the weighted sum of theirs, which the first Adam
    step turns into w -= lr g / (|g| + eps)."""
    print("spai batch", sizes, flush=True)
    mats = [store(spk, band(n, 100 + k)) for k, n in enumerate(sizes)]
    p = rand_params(3, scale3=0.1)
    model = spk.SpaiModel(0)
    model.params = p
    rows = float(sum(sizes))
    loss, grad = 0.0, np.zeros(p.size)
    for A, n in zip(mats, sizes):
        l, g = model.loss_grad(A)
        loss += l * n / rows
        grad += g.astype(np.float64) * (n / rows)
    lr = 1e-3
    hist = model.train(mats, epochs=1, learning_rate=lr, batch_matrices=len(mats),
                       shuffle_seed=1)
    # every row's loss is summed in double, in another order
    assert len(hist) == 1 and abs(hist[0] - loss) <= 1e-9 * loss
    # sums of FP32 partials and of bf16 deltas: dL/dy is scaled before its
    # rounding (2^-9), so |g| sums agree to that on the whole; where the sign
    # is beyond doubt the step is lr to the same accuracy
    big = np.abs(grad) > 0.05 * np.sqrt(np.mean(grad**2)) + 1e-4
    step = (p - model.params)[big].astype(np.float64)
    want = lr * np.sign(grad[big])
    far = np.abs(step - want) > 1e-3 * lr + 2e-7
    assert big.any() and far.mean() <= 0.02, (far.mean(), big.sum())


def test_prediction_beyond_a_group(spk):
    """1.1 million rows (a group holds 2^20): M's values against the loss,
    ||I - M A||^2 / n in double, and equal rows in both parts."""
    nx, ny = 1100, 1000
    A = spk.poisson_2d(nx, ny)
    model = spk.SpaiModel(0)
    model.params = rand_params(3, scale3=0.1)
    M = model.predict(A)
    rp, ci, v = A.download()
    n = A.nrows
    mp, mc, mv = M.download()
    assert np.array_equal(rp, mp) and np.array_equal(ci, mc)
    R = sp.identity(n) - sp.csr_matrix((mv, mc, mp), (n, n)) @ sp.csr_matrix((v, ci, rp), (n, n))
    loss, _ = model.loss_grad(A)
    want = (R.data**2).sum() / n
    assert abs(loss - want) <= 1e-10 * want
    # rows two or more points off the walls have the same features
    inner = 500 * nx + 550
    first = mv[rp[inner]:rp[inner + 1]]
    for i in (2 * nx + 2, (1 << 20) - 7, (1 << 20) + 1, (ny - 3) * nx + 9):
        x = i % nx
        assert 2 <= x < nx - 2
        assert np.array_equal(mv[rp[i]:rp[i + 1]], first), i


def test_rejections_keep_their_order(spk):
    """The first matrix that cannot be trained on names the reason."""
    ok = store(spk, band(70, 1))
    bad = store(spk, sp.csr_matrix(-sp.identity(70)))
    wide = store(spk, sp.csr_matrix(np.eye(3, 4)))
    model = spk.SpaiModel(0)
    for mats, what in (([ok, bad, wide], "positive diagonal"),
                       ([ok, wide, bad], "square matrix")):
        with pytest.raises(spk.InvalidArgument, match=what):
            model.train(mats, epochs=1, learning_rate=1e-3, batch_matrices=2)


def _merged_loss(rp, ci, v, m):
    """The loss of M's values m on A's entries, rows merged list by list (a
    repeated column is met once per entry)."""
    n, total = len(rp) - 1, 0.0
    for i in range(n):
        heads = [[int(rp[ci[p]]), int(rp[ci[p] + 1]), m[p]] for p in range(rp[i], rp[i + 1])]
        while any(h[0] < h[1] for h in heads):
            c = min(ci[h[0]] for h in heads if h[0] < h[1])
            met = [h for h in heads if h[0] < h[1] and ci[h[0]] == c]
            res = (1.0 if c == i else 0.0) - sum(h[2] * v[h[0]] for h in met)
            total += res * res
            for h in met:
                h[0] += 1
    return total / n


def test_a_repeated_diagonal_has_the_same_slots_in_training(spk):
    """Training and prediction read their rows in two forms; both take the
    first of two diagonal entries as the row's."""
    A = band(150, 9, keep=1.0)
    rp, ci, v = [0], [], []
    for i in range(150):
        for p in range(A.indptr[i], A.indptr[i + 1]):
            again = A.indices[p] == i and i % 7 == 3 and A.indptr[i + 1] - p < 5
            ci += [A.indices[p]] * (2 if again else 1)
            v += [A.data[p], 0.75 * A.data[p]][:2 if again else 1]
        rp.append(len(ci))
    rp, ci, v = np.array(rp), np.array(ci), np.array(v)
    Ad = spk.CsrMatrix.from_host(150, 150, rp, ci, v)
    model = spk.SpaiModel(4)
    model.params = rand_params(5)
    m = model.predict(Ad).download()[2]
    loss, _ = model.loss_grad(Ad)
    # the same FP64 values merged in the same order, but for the sum's order
    ref = _merged_loss(rp, ci, v, m)
    assert abs(loss - ref) <= 1e-12 * ref
