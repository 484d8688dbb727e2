"""Device memory from the pool: sizes around its classes and beyond what it
keeps, blocks that come back, threads, and a block freed while work on it is
still queued."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spk():
    import sparkit_amd
    sparkit_amd.init(0)
    return sparkit_amd


@pytest.mark.parametrize("n", [0, 1, 511, 512, 513, 4096, 4097, 8191, 8193, 131072, 131073,
                               1 << 20, (1 << 20) + 1, (1 << 25) + 3])
def test_sizes(spk, n):
    print("pool", n, flush=True)
    rng = np.random.default_rng(n)
    keep = [rng.integers(0, 1 << 30, n).astype(np.float64) for _ in range(2)]
    for _ in range(3):
        a, b = (spk.DeviceVector.from_numpy(k) for k in keep)
        assert a.n == 0 or a.ptr.value != b.ptr.value
        assert np.array_equal(a.numpy(), keep[0]) and np.array_equal(b.numpy(), keep[1])
        del a, b


def test_more_than_the_pool_keeps(spk):
    """3 GB of freed vectors of one size, then many small ones: the pool
    returns the oldest, and every vector still holds its own values."""
    big = [spk.DeviceVector.zeros(1 << 24) for _ in range(24)]
    del big
    small = [spk.DeviceVector.from_numpy(np.full(100 + k, float(k))) for k in range(700)]
    small2 = small[::2]
    del small
    again = [spk.DeviceVector.from_numpy(np.full(100 + k, -1.0)) for k in range(700)]
    for k, v in enumerate(small2):
        assert np.array_equal(v.numpy(), np.full(100 + 2 * k, 2.0 * k))
    for k, v in enumerate(again):
        assert np.array_equal(v.numpy(), np.full(100 + k, -1.0))


def test_freed_while_in_use(spk):
    """multiply's result is dropped and made again while the products are
    queued: each kept one holds its own product."""
    A = spk.poisson_2d(300)
    xs = [spk.uniform_pm1(k, A.nrows) for k in range(40)]
    ref = []
    for x in xs:
        y = spk.multiply(A, x)
        spk.synchronize()
        ref.append(y.numpy())
    kept = []
    for k, x in enumerate(xs):
        for _ in range(5):
            y = spk.multiply(A, xs[(k * 7) % 40])  # dropped at once
        kept.append(spk.multiply(A, x))
    for y, r in zip(kept, ref):
        assert np.array_equal(y.numpy(), r)


def test_threads(spk):
    """Allocation and release from several threads (the calls that queue work
    take turns, as the library asks)."""
    lock, bad = threading.Lock(), []

    def work(seed):
        rng = np.random.default_rng(seed)
        for _ in range(60):
            h = rng.uniform(-1, 1, int(rng.integers(1, 40000)))
            with lock:
                v = spk.DeviceVector.from_numpy(h)
                w = spk.DeviceVector(v.n)
                w.copy_from(v)
            with lock:
                if not np.array_equal(w.numpy(), h):
                    bad.append(seed)
            del v, w  # outside the lock

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_finalize_gives_the_pool_back():
    """Vectors that outlive spk_finalize, and a library started again."""
    import subprocess
    import sys
    code = """
import numpy as np, sparkit_amd as spk
spk.init(0)
for k in range(40):
    v = spk.DeviceVector.from_numpy(np.arange(5000.0))
late = spk.DeviceVector(77)
from sparkit_amd import _lib
_lib.call("spk_finalize")
spk.init(0)
w = spk.DeviceVector.from_numpy(np.arange(5000.0))
del late
for k in range(40):
    v = spk.DeviceVector.from_numpy(np.arange(77.0) + k)
assert np.array_equal(w.numpy(), np.arange(5000.0))
print("ok")
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.stdout.strip().endswith("ok"), r.stderr


def test_a_second_free_is_refused(spk):
    """The pool keeps the block, and the next owners get distinct ones."""
    import ctypes as C

    from sparkit_amd import _lib
    for nbytes in (64, 4096, 1 << 20):
        p = C.c_void_p()
        _lib.call("spk_malloc", C.byref(p), nbytes)
        _lib.call("spk_free", p)
        with pytest.raises(spk.SpkError):
            _lib.call("spk_free", p)
        vs = [spk.DeviceVector(nbytes // 8) for _ in range(40)]
        assert len({v.ptr.value for v in vs}) == 40


@pytest.mark.parametrize("nbytes", [4096, 1 << 20])
def test_a_block_given_back_by_hipfree(spk, nbytes):
    """spk_malloc's memory given to hipFree, its address taken by a smaller
    hipMalloc, and that given to spk_free: it goes to hipFree, and no vector
    of the old size gets it."""
    import ctypes as C

    from sparkit_amd import _lib
    hip = C.CDLL("libamdhip64.so")
    p, q = C.c_void_p(), C.c_void_p()
    held, met = [], False
    for _ in range(60):  # until hipMalloc returns an address of the pool's
        _lib.call("spk_malloc", C.byref(p), nbytes)
        assert hip.hipFree(p) == 0
        assert hip.hipMalloc(C.byref(q), C.c_size_t(nbytes // 4)) == 0
        if q.value == p.value:
            met = True
            break
        held.append(q.value)
    for h in held:
        assert hip.hipFree(C.c_void_p(h)) == 0
    print("address met again:", met, flush=True)
    if met:
        _lib.call("spk_free", q)
        vs = [spk.DeviceVector.from_numpy(np.full(nbytes // 8, float(k))) for k in range(40)]
        for k, v in enumerate(vs):
            assert (v.numpy() == k).all()
        spans = sorted((v.ptr.value, v.ptr.value + nbytes) for v in vs)
        assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))


def test_release_memory(spk):
    """What the pool keeps goes back to the device; what is in use stays."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value
    keep = spk.DeviceVector.from_numpy(np.arange(1 << 20, dtype=np.float64))
    big = [spk.DeviceVector.zeros(1 << 24) for _ in range(8)]  # 1 GiB
    del big
    spk.synchronize()
    before = free()
    spk.release_memory()
    assert free() - before >= 1 << 30
    spk.release_memory()  # nothing left to give
    assert np.array_equal(keep.numpy(), np.arange(1 << 20, dtype=np.float64))
    assert (spk.DeviceVector.from_numpy(np.full(1 << 20, 2.0)).numpy() == 2.0).all()


def test_freed_while_another_stream_reads(spk):
    """A vector freed while work on a second stream is still to read it: what
    the next owners of its block write does not reach that work."""
    import ctypes as C

    from sparkit_amd import _lib
    hip = C.CDLL("libamdhip64.so")
    stream = C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0  # non-blocking
    A = spk.poisson_3d(128)
    u, w = spk.uniform_pm1(1, A.nrows), spk.DeviceVector.zeros(A.nrows)
    n = 5000
    for k in range(5):
        v = spk.DeviceVector.from_numpy(np.full(n, 7.0 + k))
        out = spk.DeviceVector.zeros(n)
        spk.synchronize()
        _lib.call("spk_set_stream", stream)
        try:
            for _ in range(300):  # some milliseconds of products, then the read
                A.spmv(u, w)
            out.copy_from(v)
        finally:
            _lib.call("spk_set_stream", None)
        at = v.ptr.value
        del v
        met = False
        for _ in range(40):  # until the block comes back, as soon as it may
            y = spk.DeviceVector.zeros(n)
            met = met or y.ptr.value == at
            del y
        assert met
        assert hip.hipStreamSynchronize(stream) == 0
        assert (out.numpy() == 7.0 + k).all()
    assert hip.hipStreamDestroy(stream) == 0
