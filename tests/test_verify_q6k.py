"""The Q6_K verify GEMV (amdc_gemv_q6_k_v8 / _v16) on an MI355X: every token's bits are the decode GEMV's, at the edges of
its row groups, tiles, ranges and token halves, on ordinary weights and on the extremes of the format (weights -32 and
31 on scales -128 and 127 with activations of -127 and 127: the largest half dots)."""
import subprocess
import sys

import numpy as np
import pytest

from amdc import synth

pytestmark = pytest.mark.gpu
Q6 = synth.KIND_Q6_K


def extremes(rows, ng, seed):
    """GGUF Q6_K super-blocks (ql 128, qh 64, int8 scales 16, f16 d) of 0 and 63 with extreme scales."""
    g = np.random.default_rng(seed)
    b = np.zeros((rows, ng, 210), np.uint8)
    b[..., :192] = np.where(g.random((rows, ng, 1)) < 0.5, 0, 255)
    b[..., 192:208] = np.where(g.random((rows, ng, 16)) < 0.5, 128, 127)
    b[..., 208:] = np.frombuffer(np.float16(0.01).tobytes(), np.uint8)
    return b.reshape(-1)


@pytest.mark.parametrize("rows,nb,ks", [(1, 8, 0), (63, 56, 0), (65, 64, 0), (17, 72, 0), (64, 136, 2), (130, 264, 0), (130, 264, 3), (48, 520, 16)])
@pytest.mark.parametrize("T", [2, 7, 8, 9, 16])
@pytest.mark.parametrize("extreme", [False, True])
def test_bits_of_decode(dev, rows, nb, ks, T, extreme):
    src = extremes(rows, nb // 8, nb) if extreme else synth.gguf(Q6, rows, 32 * nb, rows + nb)
    x = synth.activations(T, 32 * nb, T)
    if extreme:
        x = np.sign(x).astype(np.float32)
        x[0] = 1.0
    xs = (40 * nb + 255) // 256 * 256
    W, X, Q = dev.DevBuf.of(dev.repack(Q6, src, rows, 32 * nb)), dev.DevBuf.of(x), dev.DevBuf(T * xs)
    Q.fill(0)
    dev.quant_q8(X, Q, nb, T, 128 * nb, xs)
    one, Y = dev.DevBuf(4 * rows), dev.DevBuf(4 * T * rows + 256)
    want = []
    dev.set_tuning(form=2)
    for t in range(T):
        dev.gemv(Q6, W, Q.ptr + t * xs, one, rows, nb)
        want.append(one.download(np.uint32).copy())
    try:
        dev.set_tuning(gemm_ksplit=ks if ks else 1)  # (a split set: the MFMA kernels at any size)
        Y.fill(0xEE)
        dev.gemv_t(Q6, W, Q, Y, rows, nb, T, xs, rows)
        y = Y.download(np.uint32)
        assert (y[T * rows:] == 0xEEEEEEEE).all()
        assert np.array_equal(y[:T * rows].reshape(T, rows), np.stack(want))
        dev.set_tuning()
        dev.gemv_t(Q6, W, Q, Y, rows, nb, T, xs, rows)  # as dispatched
        assert np.array_equal(Y.download(np.uint32)[:T * rows].reshape(T, rows), np.stack(want))
    finally:
        dev.set_tuning()


@pytest.mark.parametrize("rows,nb,T", [(4096, 128, 16), (3200, 344, 4)])
def test_first_call_under_capture(rows, nb, T):
    """In a fresh process, whose workspace holds nothing yet: a captured call replays with the eager call's bits."""
    code = f"""
import sys; sys.path[:0] = {sys.path!r}
import numpy as np, amdc as dev
from amdc import synth
dev.open_device()
rows, nb, T = {rows}, {nb}, {T}
xs = (40 * nb + 255) // 256 * 256
g = np.random.default_rng(1)
W = dev.DevBuf.of(np.resize(dev.repack(4, synth.gguf(4, 40, 32 * nb, 1), 40, 32 * nb), dev.mat_bytes(4, rows, 32 * nb)))
X, Q, Y = dev.DevBuf.of(synth.activations(T, 32 * nb, 2)), dev.DevBuf(T * xs), dev.DevBuf(4 * T * rows)
Q.fill(0)
dev.quant_q8(X, Q, nb, T, 128 * nb, xs)
S = dev.Stream()
S.sync()
G = dev.Graph(S, lambda s: dev.gemv_t(4, W, Q, Y, rows, nb, T, xs, rows, stream=s))
out = []
for rep in range(3):
    Y.fill(0xEE); G.launch(); S.sync(); out.append(Y.download(np.uint32))
    Y.fill(0xEE); dev.gemv_t(4, W, Q, Y, rows, nb, T, xs, rows); out.append(Y.download(np.uint32))
assert all(np.array_equal(o, out[0]) for o in out)
print("same")
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "same" in r.stdout, r.stderr[-800:]
