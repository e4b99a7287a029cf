"""The single-shot decode GEMV of Q8_0 and Q6_K (amdc_gemv_q8_0_s1 / _s2, amdc_gemv_q6_k_s1, and on an f32 vector
_xs1 / _xs2l; _s1l and so on: nontemporal loads) on an MI355X: bit for bit the persistent form's results (which test_gpu_k8.py holds to the oracle), at the
sizes where lanes, super-groups per lane, workgroups and the rule that chooses them end."""
import numpy as np
import pytest

from amdc import synth

pytestmark = pytest.mark.gpu
Q8, Q6 = synth.KIND_Q8_0, synth.KIND_Q6_K


@pytest.fixture(autouse=True)
def _tuning_reset(dev):
    dev.set_tuning()
    yield
    dev.set_tuning()


# super-groups: one, a full 4 lanes, one past; 64 and 65 (Q8_0: two per lane; Q6_K: the persistent form), 128 and 129;
# rows: one, a workgroup's less and plus one, enough workgroups for the fused kernels' second item (and 16 and 48 blocks)
CASES = [(Q8, 1, 1), (Q8, 63, 32), (Q8, 65, 33), (Q8, 5, 512), (Q8, 9, 513), (Q8, 7, 1017), (Q8, 5, 1024), (Q8, 3, 1025), (Q8, 12289, 64),
         (Q8, 12300, 125), (Q8, 3073, 192), (Q8, 3073, 193), (Q6, 1, 8), (Q6, 65, 32), (Q6, 63, 40), (Q6, 5, 512), (Q6, 3, 520),
         (Q6, 6200, 160), (Q6, 20000, 64), (Q6, 65535, 40), (Q6, 65536, 40), (Q6, 65536, 56), (Q6, 33, 112), (Q6, 70, 224), (Q8, 9, 576)]


@pytest.mark.parametrize("kind,rows,nb", CASES)
@pytest.mark.parametrize("special", [False, True])
def test_bits_of_the_persistent_form(dev, kind, rows, nb, special):
    # a few distinct rows repeated: the weights' generator is slow
    per = min(rows, 37)
    src = dev.repack(kind, synth.gguf(kind, per, 32 * nb, rows + nb), per, 32 * nb)
    rb = src.nbytes // per
    W = dev.DevBuf.of(np.resize(src.reshape(per, rb), (rows, rb)))
    x = synth.activations(1, 32 * nb, nb)
    if special:
        x[0, 3], x[0, 32 * nb - 1] = np.inf, np.nan
    xs = (40 * nb + 255) // 256 * 256
    g = np.random.default_rng(rows)
    bias, res = g.standard_normal(rows).astype(np.float32), g.standard_normal(rows).astype(np.float32)
    X, Q, Q2, B, R = dev.DevBuf.of(x), dev.DevBuf(xs), dev.DevBuf(xs), dev.DevBuf.of(bias), dev.DevBuf.of(res)
    Y = dev.DevBuf(4 * rows + 256)
    Q.fill(0), Q2.fill(0)
    dev.quant_q8(X, Q, nb, 1, 0, 0)

    def run(f, *a, **k):
        Y.fill(0xEE)
        f(kind, W, *a, Y, rows, nb, **k)
        y = Y.download(np.uint32)
        assert (y[rows:] == 0xEEEEEEEE).all()
        return y[:rows]

    for ep in ({}, {"bias": B, "res": R}):
        dev.set_tuning(form=2)
        want = run(dev.gemv, Q, **ep)
        dev.set_tuning()
        assert np.array_equal(run(dev.gemv, Q, **ep), want)
        assert np.array_equal(run(dev.gemv_x, X, **ep), want)
        assert np.array_equal(run(dev.gemv_x, X, q8=Q2, **ep), want)
        assert np.array_equal(Q2.download(np.uint8)[:40 * nb], Q.download(np.uint8)[:40 * nb])


@pytest.mark.parametrize("kind,rows,nb,on_q8,on_f32", [
    # 10, 15 and 21 super-groups on 16 and 32 lanes: no row on half its lanes; 16 of 16 with more than 3 workgroups per CU: one
    (Q8, 25000, 80, "q8_0_s1", "q8_0_xs1"), (Q8, 13000, 113, "q8_0_s1", "q8_0_xs1"), (Q8, 9919, 162, "q8_0_s1", "q8_0_s1"), (Q8, 13000, 128, "q8_0_s1l", "q8_0_xs2l"),
    # whole lines: 8 super-groups (Q8_0), 14 (Q6_K)
    (Q8, 100, 64, "q8_0_s1l", "q8_0_xs1l"), (Q8, 100, 72, "q8_0_s1", "q8_0_xs1"), (Q6, 100, 112, "q6_k_s1l", "q6_k_xs1l"), (Q6, 100, 128, "q6_k_s1", "q6_k_xs1"),
    # more than 16 super-groups, 2^16 blocks quantized in all and one workgroup more
    (Q8, 3272, 160, "q8_0_s1", "q8_0_xs1l"), (Q8, 3280, 160, "q8_0_s1", "q8_0_xs1"), (Q6, 3272, 160, "q6_k_s1", "q6_k_xs1l"), (Q6, 3280, 160, "q6_k_s1", "q6_k_xs1"),
    # more than 64 super-groups; many rows
    (Q8, 4095, 544, "q8_0_s2", "q8_0_s2"), (Q8, 4096, 544, "q8_0_p2", "q8_0_p2"), (Q8, 64, 576, "q8_0_s2l", "q8_0_s2l"), (Q6, 64, 520, "q6_k_p2", "q6_k_p2"),
    (Q6, 65536, 40, "q6_k_s1", "q6_k_xs1")])
def test_choice(dev, kind, rows, nb, on_q8, on_f32):
    if dev.cu_count() != 256:
        pytest.skip("the lines of the rule are those of 256 CUs")
    W, X, Q, Y = dev.DevBuf(dev.mat_bytes(kind, rows, 32 * nb)), dev.DevBuf.of(synth.activations(1, 32 * nb, 1)), dev.DevBuf(40 * nb), dev.DevBuf(4 * rows)
    W.fill(0)
    dev.quant_q8(X, Q, nb)
    dev.gemv(kind, W, Q, Y, rows, nb)
    assert dev.last_kernel() == "amdc_gemv_" + on_q8
    dev.gemv_x(kind, W, X, Y, rows, nb)
    assert dev.last_kernel() == "amdc_gemv_" + on_f32


@pytest.mark.parametrize("kind", [Q8, Q6])
def test_result_over_the_vector(dev, kind):
    """y written onto x: x is quantized before any result is written."""
    rows, nb = 1500, 48
    W = dev.DevBuf.of(dev.repack(kind, synth.gguf(kind, rows, 32 * nb, 3), rows, 32 * nb))
    x = synth.activations(1, 32 * nb, 4)
    X, Y = dev.DevBuf.of(x), dev.DevBuf(4 * rows)
    dev.gemv_x(kind, W, X, Y, rows, nb)
    want = Y.download(np.uint32)
    for off in (0, 16):
        Z = dev.DevBuf.of(x)
        dev.gemv_x(kind, W, Z, Z.ptr + off, min(rows, 32 * nb - off // 4), nb)
        assert np.array_equal(Z.download(np.uint32)[off // 4:][:rows], want)
