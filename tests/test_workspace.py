"""Which calls ask for the library's device workspace, on the CPU against a HIP runtime that does nothing
(capi/hip_stub.c). Calls on the shared workspace must be ordered by the caller; the others may overlap on the device."""
import os
import subprocess
import sys

import pytest

from amdc import synth

HERE = os.path.dirname(os.path.abspath(__file__))
Q6 = synth.KIND_Q6_K


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-w", os.path.join(HERE, "capi", "hip_stub.c"), "-o", str(d / "libamdhip64.so.7")], check=True)
    return str(d)


def workspace(stub, calls):
    """The bytes of device memory that each call of gemv_t(kind, rows, nb, T) asks for, each in a library just opened."""
    code = f"""
import sys; sys.path[:0] = {sys.path!r}
import ctypes as C, amdc
hip = C.CDLL("libamdhip64.so.7")
for kind, rows, nb, T in {calls!r}:
    n = C.c_size_t.in_dll(hip, "stub_bytes"); n.value = 0
    l = C.c_uint.in_dll(hip, "stub_launches"); l.value = 0
    assert amdc.lib().amdc_open(None) == 0
    amdc.gemv_t(kind, 4096, 8192, 12288, rows, nb, T, 40 * nb + 256, rows)
    assert l.value
    print(n.value)
    amdc.lib().amdc_close()
"""
    env = dict(os.environ, LD_LIBRARY_PATH=stub)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=60, env=env)
    assert r.returncode == 0, r.stderr[-800:]
    return [int(v) for v in r.stdout.split()]


def test_q6k_without(stub):
    """Q6_K calls on the few-vector kernel, and of rows of at most 4 tiles of 64 blocks that fill the CUs unsplit, use none."""
    calls = [(Q6, 4096, 344, 4), (Q6, 8192, 64, 8),  # few vectors
             (Q6, 8192, 128, 8), (Q6, 11008, 128, 6), (Q6, 16384, 128, 8), (Q6, 13000, 160, 8), (Q6, 16000, 192, 4), (Q6, 16000, 192, 8),
             (Q6, 64, 128, 16), (Q6, 4096, 128, 16), (Q6, 16000, 128, 9), (Q6, 8192, 192, 16), (Q6, 11008, 256, 16)]
    assert workspace(stub, calls) == [0] * len(calls)


def test_q6k_split(stub):
    """Longer rows are split: the smallest workspace (1 MiB) or the next powers of two that hold ranges x T x rows sums."""
    assert workspace(stub, [(Q6, 5120, 544, 5), (Q6, 5120, 544, 16), (Q6, 1024, 544, 2)]) == [1 << 20, 4 << 20, 1 << 20]
