"""The producers' kernels for aligned rows (amdc_quant_q8_v, amdc_swiglu_q8_v, amdc_rmsnorm_q8_r) on an MI355X: the
bits of the kernels for any alignment (rows moved by 4 bytes), which test_producers.py and test_gpu_parity.py hold
to the oracle, at the edges of their workgroups, with zero, infinite and NaN values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows_of(dev, a, off, stride):
    """a's rows on the device, off bytes into a buffer, stride bytes apart."""
    T, n = a.shape
    h = np.zeros(off + T * stride, np.uint8)
    for t in range(T):
        h[off + t * stride:off + t * stride + 4 * n] = a[t].view(np.uint8)
    return dev.DevBuf.of(h)


def rows_from(buf, off, stride, T, nbytes):
    h = buf.download(np.uint8)
    return np.stack([h[off + t * stride:off + t * stride + nbytes] for t in range(T)])


def data(n, T, seed):
    x = (np.random.default_rng(seed).standard_normal((T, n)) * 3).astype(np.float32)
    x[0, :32] = 0.0
    x[-1, n - 32] = np.inf
    x[T // 2, n - 31] = np.nan
    return x


# blocks around one and two workgroups of 32
SIZES = [(1, 1), (31, 3), (32, 1), (33, 2), (65, 5), (544, 1)]


@pytest.mark.parametrize("nb,T", SIZES)
def test_quant(dev, nb, T):
    x = data(32 * nb, T, nb)
    got = []
    # x.s pointer, x.s stride aligned or not; q elsewhere
    for off, pad, qoff in ((0, 16, 0), (4, 16, 0), (0, 4, 0), (0, 0, 4)):
        xs, qs = 128 * nb + pad, 40 * nb + 8
        X, Q = rows_of(dev, x, off, xs), dev.DevBuf(T * qs + 16)
        Q.fill(0xEE)
        dev.quant_q8(X.ptr + off, Q.ptr + qoff, nb, T, xs, qs)
        h = Q.download(np.uint8)
        got.append(rows_from(Q, qoff, qs, T, 40 * nb))
        gaps = [h[:qoff], h[qoff + T * qs:]] + [h[qoff + t * qs + 40 * nb:qoff + (t + 1) * qs] for t in range(T)]
        assert all((gap == 0xEE).all() for gap in gaps)
    assert all(np.array_equal(g, got[0]) for g in got)


@pytest.mark.parametrize("nb,T", SIZES)
@pytest.mark.parametrize("withq", [True, False])
def test_swiglu(dev, nb, T, withq):
    n = 32 * nb
    a, b = data(n, T, nb), data(n, T, nb + 1)[:, ::-1].copy()
    got = []
    for off, pad in ((0, 16), (4, 16), (0, 4)):
        s, qs = 4 * n + pad, 40 * nb + 8
        A, B, Q = rows_of(dev, a, off, s), rows_of(dev, b, off, s), dev.DevBuf(T * qs)
        Q.fill(0xEE)
        dev.swiglu_q8(A.ptr + off, B.ptr + off, n, Q if withq else None, T, s, qs)
        h = A.download(np.uint8)
        assert all((h[off + t * s + 4 * n:off + (t + 1) * s] == 0).all() for t in range(T))
        got.append((rows_from(A, off, s, T, 4 * n), Q.download(np.uint8)))
    assert all(np.array_equal(g[0], got[0][0]) and np.array_equal(g[1], got[0][1]) for g in got)


# 2^19 values and more in 96 rows and more of 1024 and more take the row kernel: one row short of it, on it, past it;
# rows of whole passes of 1024 and with a rest of 32
@pytest.mark.parametrize("n,T", [(4096, 127), (4096, 128), (992, 530), (1024, 512), (2080, 253), (5120, 103), (8192, 95), (5472, 96)])
@pytest.mark.parametrize("withq", [True, False])
def test_rmsnorm(dev, n, T, withq):
    nb, x = n // 32, data(n, T, T)
    w = np.random.default_rng(n).standard_normal((1, n)).astype(np.float32)
    got = []
    for off, pad in ((0, 16), (4, 16), (0, 4)):
        s, qs = 4 * n + pad, 40 * nb + 8
        X, W, Y, Q = rows_of(dev, x, off, s), rows_of(dev, w, 0, 4 * n), dev.DevBuf(off + T * s), dev.DevBuf(T * qs)
        Y.fill(0xEE), Q.fill(0xEE)
        dev.rmsnorm_q8(X.ptr + off, W, Y.ptr + off, n, 1e-6, Q if withq else None, T, s, s, qs)
        h = Y.download(np.uint8)[off:].reshape(T, s)
        assert (h[:, 4 * n:] == 0xEE).all()
        got.append((h[:, :4 * n].copy(), Q.download(np.uint8)))
    assert all(np.array_equal(g[0], got[0][0]) and np.array_equal(g[1], got[0][1]) for g in got)
