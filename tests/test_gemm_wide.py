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
def test_edges(dev, orc, kind, rows, nb, T, ks):
    c = Case(dev, orc, kind, rows, nb, T, seed=rows + T)
    c.quant()
    g = np.random.default_rng(T)
    bias, res = g.standard_normal(rows).astype(np.float32), g.standard_normal((T, rows)).astype(np.float32)
    B, R = dev.DevBuf.of(bias), dev.DevBuf.of(res)
    dev.set_tuning(gemm_ksplit=ks)
    try:
        c.Y.fill(0xFF)
        dev.gemm(kind, c.W, c.Q, c.Y, rows, nb, T, c.xs, rows, rows, bias=B, res=R)
    finally:
        dev.set_tuning()
    y = c.y_gpu()
    for t in range(T):
        want = orc.epilogue(c.y_oracle(t), bias, res[t])
        assert rel_err(y[t], want, c.mag(t) + np.abs(bias) + np.abs(res[t])) < TOL, t


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [synth.KIND_Q4_0, synth.KIND_Q8_0])
@pytest.mark.parametrize("nb", [1, 7, 9, 21])
def test_ragged_blocks(dev, orc, kind, nb):
    """Rows whose last super-group is partly filled."""
    rows, T = 140, 70
    c = Case(dev, orc, kind, rows, nb, T, seed=nb)
    c.quant()
    dev.gemm(kind, c.W, c.Q, c.Y, rows, nb, T, c.xs, rows)
    y = c.y_gpu()
    for t in range(T):
        assert rel_err(y[t], c.y_oracle(t), c.mag(t)) < TOL, t


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
def test_many_tiles_exact(dev, orc, kind):
    """More tiles than the device holds at once (the third form for all but Q8_0: whole rounds and a split tail)
    against the exact sums, spot-checked over every row and token tile."""
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
