"""The wide-tile prefill GEMM (amdc_gemmw_*) on an MI355X, every kind, at the sizes where its tiles, groups and
splits end: against the oracle within 1e-5 of sum |terms| (the GPU bar of test_gpu_parity.py), and bit for bit on
the exact cases (exactcase.py), where any wrong index moves y by at least 1/2."""
import numpy as np
import pytest

import exactcase
from amdc import synth
from test_gpu_parity import TOL, Case, rel_err

KINDS = [synth.KIND_Q4_0, synth.KIND_Q8_0, synth.KIND_Q4_K, synth.KIND_Q6_K]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
# rows around a 128-row tile, one / two / three super-groups (an odd count leaves the second group without its
# last), tokens around 64 and 128, splits that leave a workgroup a single super-group
@pytest.mark.parametrize("rows,nb,T,ks", [(1, 8, 33, 0), (127, 16, 63, 0), (128, 24, 64, 0), (129, 40, 65, 0), (257, 24, 128, 2),
                                          (300, 72, 129, 3), (130, 104, 200, 7)])
@pytest.mark.parametrize("kern", [0, 5])  # as dispatched (the 64-row kernels at these sizes), and the wide tiles
def test_edges(dev, orc, kind, rows, nb, T, ks, kern):
    c = Case(dev, orc, kind, rows, nb, T, seed=rows + T)
    c.quant()
    g = np.random.default_rng(T)
    bias, res = g.standard_normal(rows).astype(np.float32), g.standard_normal((T, rows)).astype(np.float32)
    B, R = dev.DevBuf.of(bias), dev.DevBuf.of(res)
    dev.set_tuning(gemm_kernel=kern, gemm_ksplit=ks)
    try:
        c.Y.fill(0xFF)
        dev.gemm(kind, c.W, c.Q, c.Y, rows, nb, T, c.xs, rows, rows, bias=B, res=R)
        assert dev.last_kernel() == "amdc_gemm_reduce" or dev.last_kernel().startswith("amdc_gemmw" if kern else "amdc_gemmh")
    finally:
        dev.set_tuning()
    y = c.y_gpu()
    for t in range(T):
        want = orc.epilogue(c.y_oracle(t), bias, res[t])
        assert rel_err(y[t], want, c.mag(t) + np.abs(bias) + np.abs(res[t])) < TOL, t


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [synth.KIND_Q4_0, synth.KIND_Q8_0])
@pytest.mark.parametrize("nb", [1, 7, 9, 21])
@pytest.mark.parametrize("T,kern", [(70, 0), (40, 5), (70, 5)])
def test_ragged_blocks(dev, orc, kind, nb, T, kern):
    """Rows whose last super-group is partly filled."""
    rows = 140
    c = Case(dev, orc, kind, rows, nb, T, seed=nb)
    c.quant()
    c.Y.fill(0xFF)
    dev.set_tuning(gemm_kernel=kern)
    try:
        dev.gemm(kind, c.W, c.Q, c.Y, rows, nb, T, c.xs, rows)
    finally:
        dev.set_tuning()
    y = c.y_gpu()
    for t in range(T):
        assert rel_err(y[t], c.y_oracle(t), c.mag(t)) < TOL, t


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
def test_many_tiles_exact(dev, orc, kind):
    """More tiles than the device holds at once (128 tokens in two groups, unsplit) against the exact sums, spot-checked over
    every row and token tile."""
    rows, nb, T = 128 * 130 + 5, 16, 128 * 4 + 3
    src = exactcase.gguf(kind, rows, 32 * nb, seed=kind)
    x = exactcase.activations(T, 32 * nb, seed=kind + 1)
    xs = (40 * nb + 255) // 256 * 256
    W, X, Q, Y = dev.DevBuf.of(dev.repack(kind, src, rows, 32 * nb)), dev.DevBuf.of(x), dev.DevBuf(T * xs), dev.DevBuf(4 * T * rows)
    dev.quant_q8(X, Q, nb, T, 128 * nb, xs)
    Y.fill(0xFF)
    dev.gemm(kind, W, Q, Y, rows, nb, T, xs, rows)
    y = Y.download(np.float32).reshape(T, rows)
    xq = orc.quant_q8(x)
    for t in range(0, T, 37):
        assert np.array_equal(y[t], exactcase.exact_y(orc, kind, src, rows, nb, xq[t])), t
    assert np.isfinite(y).all()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [synth.KIND_Q4_0, synth.KIND_Q4_K, synth.KIND_Q6_K])
@pytest.mark.parametrize("nb", [16, 24])
def test_two_workgroups_exact(dev, orc, kind, nb):
    """Two workgroups per CU (amdc_gemmw_*_i128; test_host_choice.py: these sizes take it): whole rounds of 170 row tiles x 3
    token tiles and two row tiles in as many splits as super-groups, the last row tile and token tile ragged; against the
    exact sums, and rows in strides with a bias and a residual."""
    rows, T, ys, rs = 22003, 257, 22016, 22010
    src = exactcase.gguf(kind, rows, 32 * nb, seed=kind + nb)
    x = exactcase.activations(T, 32 * nb, seed=nb)
    xs = (40 * nb + 255) // 256 * 256
    g = np.random.default_rng(nb)
    bias, res = g.integers(-9, 10, rows).astype(np.float32), g.integers(-9, 10, (T, rs)).astype(np.float32)
    W, X, Q, Y, B, R = (dev.DevBuf.of(dev.repack(kind, src, rows, 32 * nb)), dev.DevBuf.of(x), dev.DevBuf(T * xs), dev.DevBuf(4 * T * ys),
                        dev.DevBuf.of(bias), dev.DevBuf.of(res))
    dev.quant_q8(X, Q, nb, T, 128 * nb, xs)
    xq = orc.quant_q8(x)
    Y.fill(0xFF)
    dev.gemm(kind, W, Q, Y, rows, nb, T, xs, rows)
    y = Y.download(np.float32)[:T * rows].reshape(T, rows).copy()
    assert np.isfinite(y).all()
    Y.fill(0xEE)
    dev.gemm(kind, W, Q, Y, rows, nb, T, xs, ys, rs, bias=B, res=R)
    z = Y.download(np.float32).reshape(T, ys)
    assert (z[:, rows:].view(np.uint32) == 0xEEEEEEEE).all()
    assert np.array_equal(z[:, :rows], res[:, :rows] + (y + bias))
    for t in (0, 1, 63, 64, 127, 128, 191, 255, 256):
        assert np.array_equal(y[t], exactcase.exact_y(orc, kind, src, rows, nb, xq[t])), t


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("kern", [4, 5])
@pytest.mark.parametrize("T", [40, 70, 150])
@pytest.mark.parametrize("ks", [1, 2])  # whole K, every tile split
def test_strides(dev, orc, kind, kern, T, ks):
    """Rows of y, res and xq further apart than they are long: the bits of the packed call, nothing written between."""
    rows, nb, ys, rs = 140, 24, 160, 150
    c = Case(dev, orc, kind, rows, nb, T, seed=T)
    c.quant()
    g = np.random.default_rng(T)
    bias, res = g.standard_normal(rows).astype(np.float32), g.standard_normal((T, rs)).astype(np.float32)
    xs = c.xs + 272
    q = np.full((T, xs), 0x5A, np.uint8)
    q[:, :40 * nb] = c.xq
    B, R, RP, Q, Y = dev.DevBuf.of(bias), dev.DevBuf.of(res), dev.DevBuf.of(np.ascontiguousarray(res[:, :rows])), dev.DevBuf.of(q), dev.DevBuf(4 * T * ys)
    dev.set_tuning(gemm_kernel=kern, gemm_ksplit=ks)
    try:
        dev.gemm(kind, c.W, c.Q, c.Y, rows, nb, T, c.xs, rows, rows, bias=B, res=RP)
        Y.fill(0xEE)
        dev.gemm(kind, c.W, Q, Y, rows, nb, T, xs, ys, rs, bias=B, res=R)
    finally:
        dev.set_tuning()
    z = Y.download(np.uint32).reshape(T, ys)
    assert (z[:, rows:] == 0xEEEEEEEE).all()
    assert np.array_equal(z[:, :rows], c.Y.download(np.uint32).reshape(T, rows))


@pytest.mark.gpu
def test_noalloc_falls_back(dev, orc):
    """A call whose image does not fit the fixed workspace beside its partial sums, but the 64-row kernels' does."""
    kind, rows, nb, T = synth.KIND_Q4_K, 64, 544, 1664
    c = Case(dev, orc, kind, rows, nb, T, seed=5)
    c.quant()
    assert T * nb * 72 <= dev.SCRATCH_BYTES < T * nb * 76
    c.Y.fill(0xFF)
    dev.op_gemv_noalloc(kind, c.W, c.Q, c.Y, rows, nb, T, c.xs, rows)
    y = c.y_gpu()
    for t in range(0, T, 111):
        assert rel_err(y[t], c.y_oracle(t), c.mag(t)) < TOL, t


# ---------------------------------------------------------------- infinities, NaN, zeros

D_OFF = {synth.KIND_Q4_0: (18, 0), synth.KIND_Q8_0: (34, 0), synth.KIND_Q4_K: (144, 0), synth.KIND_Q6_K: (210, 208)}  # block bytes, its d


def special_weights(kind, rows, nb, seed):
    """(bytes, rows with a special scale): infinite and NaN d, Q4_K: dmin, in one block of a row each; Q4_K: a row
    whose sub-block scales are all 0 (its products are 0 beside an infinite min term)."""
    size, off = D_OFF[kind]
    src = synth.gguf(kind, rows, 32 * nb, seed).reshape(rows, -1).copy()
    n = src.shape[1] // size
    f16 = np.array([np.inf, -np.inf, np.nan], np.float16).view(np.uint8).reshape(3, 2)
    for i in range(3):
        o = min(i, n - 1) * size + off
        src[5 + i, o:o + 2] = f16[i]
        if kind == synth.KIND_Q4_K:
            src[9 + i, o + 2:o + 4] = f16[i]
    if kind == synth.KIND_Q4_K:
        for g in range(n):  # sc 0..3 = 0, mn 0..3 kept; sc 4..7 = 0, mn 4..7 their low 4 bits
            h = src[20, g * size + 4:g * size + 16]
            h[0:4], h[4:8], h[8:12] = 0, h[4:8] & 63, h[8:12] & 0xF0
    return src.reshape(-1), list(range(5, 12)) + [20]


def special_tokens(xq, nb):
    """Tokens 3 .. 12 of the Q8 rows xq get special blocks; their numbers."""
    q = xq[:, :32 * nb].view(np.int8)
    d = xq[:, 32 * nb:36 * nb].view(np.float32)
    a = xq[:, 36 * nb:40 * nb].view(np.int32)

    def block(t, b, val, dd):
        q[t, 32 * b:32 * b + 32], d[t, b], a[t, b] = val, dd, 32 * val

    d[3, 4], d[4, 1], d[5, 9] = np.inf, -np.inf, np.nan
    for b in range(nb):
        block(6, b, 0, 0.0)     # the zero token
        block(9, b, 2, 1.0)     # d_a asum = 64: one significant bit
        block(10, b, b % 3, 1.0)  # some blocks 0 under every min
        block(12, b, 1, 1e-20)
    block(7, 2, 127, 1e37)      # d_a asum overflows to an infinity of each sign
    block(8, 3, -127, 1e37)
    block(11, 0, 127, 1e28)     # large and finite
    return list(range(3, 13))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("T,ks", [(40, 0), (70, 0), (150, 0), (150, 2)])
def test_special_values(dev, orc, kind, T, ks):
    """Infinite, NaN and zero blocks in activations and weights: infinities of the same sign and NaN at the same
    places as from the 64-row kernels, whose min term is in f32; the other rows and tokens keep their bits."""
    rows, nb = 140, 24
    src, srows = special_weights(kind, rows, nb, seed=kind + T)
    xq = orc.quant_q8(synth.activations(T, 32 * nb, kind + T)).reshape(T, 40 * nb).copy()
    clean_src, clean_xq = synth.gguf(kind, rows, 32 * nb, kind + T), xq.copy()
    stok = special_tokens(xq, nb)
    xs = (40 * nb + 255) // 256 * 256

    def run(s, x, kern):
        pad = np.zeros((T, xs), np.uint8)
        pad[:, :40 * nb] = x
        W, Q, Y = dev.DevBuf.of(dev.repack(kind, s, rows, 32 * nb)), dev.DevBuf.of(pad), dev.DevBuf(4 * T * rows)
        Y.fill(0x55)
        dev.set_tuning(gemm_kernel=kern, gemm_ksplit=ks)
        try:
            dev.gemm(kind, W, Q, Y, rows, nb, T, xs, rows)
        finally:
            dev.set_tuning()
        return Y.download(np.float32).reshape(T, rows)

    want, got, clean = run(src, xq, 4), run(src, xq, 5), run(clean_src, clean_xq, 5)
    for cls in (np.isnan, np.isposinf, np.isneginf):
        bad = np.argwhere(cls(got) != cls(want))
        assert len(bad) == 0, (cls.__name__, len(bad), bad[:5].tolist(), [(float(got[t, r]), float(want[t, r])) for t, r in bad[:5]])
    rest = [r for r in range(rows) if r not in srows]
    other = [t for t in range(T) if t not in stok]
    assert np.array_equal(got[np.ix_(other, rest)].view(np.uint32), clean[np.ix_(other, rest)].view(np.uint32))
    for t in stok:
        if t in (6, 9, 10, 12):
            mag = orc.gemv_f64(synth.GGML[kind], src, rows, nb, xq[t])[1][rest]
            assert rel_err(got[t, rest], want[t, rest], mag) < TOL, t
    assert np.isinf(want).any() and np.isnan(want).any() and np.all(got[6, rest] == 0.0)


@pytest.mark.gpu
# the image alone exceeds it (Q4_K, nb = 544 and 1584: 128- and 64-token tiles), or the image and the partial sums
# (128 tokens in two groups; two independent workgroups, whole rounds and a split tail; the longest rows)
@pytest.mark.parametrize("kind,rows,nb,T", [(synth.KIND_Q4_K, 64, 544, 1664), (synth.KIND_Q6_K, 628, 184, 3903), (synth.KIND_Q8_0, 802, 1184, 646),
                                            (synth.KIND_Q4_0, 15261, 552, 831), (synth.KIND_Q4_K, 290, 1584, 504), (synth.KIND_Q6_K, 1500, 2048, 380)])
def test_noalloc_in_pieces(dev, kind, rows, nb, T):
    """A GEMM whose workspace exceeds the fixed one gives the bits of amdc_op_gemv there too."""
    g = np.random.default_rng(rows)
    xs = (40 * nb + 255) // 256 * 256
    n = dev.mat_bytes(kind, rows, 32 * nb)
    chunk = g.integers(0, 100, min(n, 48 << 20), dtype=np.uint8)  # bytes below 100: every f16 in them is finite
    W, Q, Y = dev.DevBuf(n), dev.DevBuf(T * xs), dev.DevBuf(4 * T * rows)
    for o in range(0, n, len(chunk)):
        W.upload(chunk[:min(len(chunk), n - o)], o)
    X = dev.DevBuf.of(synth.activations(T, 32 * nb, rows))
    R, B = dev.DevBuf.of(g.standard_normal((T, rows)).astype(np.float32)), dev.DevBuf.of(g.standard_normal(rows).astype(np.float32))
    dev.quant_q8(X, Q, nb, T, 128 * nb, xs)
    out = []
    for f in (dev.op_gemv, dev.op_gemv_noalloc):
        Y.fill(0xFF)
        f(kind, W, Q, Y, rows, nb, T, xs, rows, rows, bias=B, res=R)
        out.append(Y.download(np.uint32))
    assert np.isfinite(out[0].view(np.float32)).all()
    assert np.array_equal(out[0], out[1]), f"{int((out[0] != out[1]).sum())} of {out[0].size} outputs differ"
