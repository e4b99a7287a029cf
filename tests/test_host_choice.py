"""The host library's choices, on the CPU against a HIP runtime that does nothing (capi/hip_stub.c): which calls ask for the
device workspace (calls on it must be ordered by the caller; the others may overlap on the device), and which prefill
GEMM runs."""
import os
import subprocess
import sys

import pytest

from amdc import synth

HERE = os.path.dirname(os.path.abspath(__file__))
Q4, Q8, Q4K, Q6 = synth.KIND_Q4_0, synth.KIND_Q8_0, synth.KIND_Q4_K, synth.KIND_Q6_K


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    d = tmp_path_factory.mktemp("hip")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-w", os.path.join(HERE, "capi", "hip_stub.c"), "-o", str(d / "libamdhip64.so.7")], check=True)
    return str(d)


def launched(stub, calls):
    """Of each call of op(kind, rows, nb, T), in a library just opened: the bytes of device memory it asks for, and its kernels."""
    code = f"""
import sys; sys.path[:0] = {sys.path!r}
import ctypes as C, amdc
hip = C.CDLL("libamdhip64.so.7")
for op, kind, rows, nb, T in {calls!r}:
    n, l = C.c_size_t.in_dll(hip, "stub_bytes"), C.c_uint.in_dll(hip, "stub_launches")
    n.value = l.value = 0
    assert amdc.lib().amdc_open(None) == 0
    getattr(amdc, op)(kind, 4096, 8192, 12288, rows, nb, T, 40 * nb + 256, rows)
    names = (C.c_char_p * 16).in_dll(hip, "stub_name")
    print(n.value, *[names[i].decode()[5:] for i in range(l.value)])
    amdc.lib().amdc_close()
"""
    env = dict(os.environ, LD_LIBRARY_PATH=stub)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=60, env=env)
    assert r.returncode == 0, r.stderr[-800:]
    got = [line.split() for line in r.stdout.splitlines()]
    assert len(got) == len(calls) and all(len(g) > 1 for g in got)
    return [(int(g[0]), g[1:]) for g in got]


def workspace(stub, calls):
    return [n for n, _ in launched(stub, [("gemv_t",) + c for c in calls])]


def test_q6k_without(stub):
    """Q6_K calls on the few-vector kernel, and of rows of at most 4 tiles of 64 blocks that fill the CUs unsplit, use none."""
    calls = [(Q6, 4096, 344, 4), (Q6, 8192, 64, 8),  # few vectors
             (Q6, 8192, 128, 8), (Q6, 11008, 128, 6), (Q6, 16384, 128, 8), (Q6, 13000, 160, 8), (Q6, 16000, 192, 4), (Q6, 16000, 192, 8),
             (Q6, 64, 128, 16), (Q6, 4096, 128, 16), (Q6, 16000, 128, 9), (Q6, 8192, 192, 16), (Q6, 11008, 256, 16)]
    assert workspace(stub, calls) == [0] * len(calls)


def test_q6k_split(stub):
    """Longer rows are split: the smallest workspace (1 MiB) or the next powers of two that hold ranges x T x rows sums."""
    assert workspace(stub, [(Q6, 5120, 544, 5), (Q6, 5120, 544, 16), (Q6, 1024, 544, 2)]) == [1 << 20, 4 << 20, 1 << 20]


def test_gemm_kernel(stub):
    """Small matrices take the 64-row kernels: at most 2^22 weights times token tiles of 64, Q4_K 3 2^21 up to 64 tokens; 65 to 96
    tokens on 2^21 to 2^22 weights the 128-token tile of a kind that has one."""
    want = [((Q8, 2048, 64, 64), "gemmh_q8_0_m64_n64"), ((Q8, 2049, 64, 64), "gemmw_q8_0_n64"), ((Q4, 2049, 64, 64), "gemmw_q4_0_n64"),
            ((Q4K, 4096, 48, 48), "gemmh_m64_n64"), ((Q4K, 3072, 64, 64), "gemmh_m64_n64"), ((Q4K, 3073, 64, 64), "gemmw_q4_k_n64"),
            ((Q8, 1400, 64, 65), "gemmh_q8_0_m64_n128"), ((Q6, 2048, 48, 80), "gemmh_q6_k_m64_n128"), ((Q4K, 2048, 64, 96), "gemmh_m64_n128"),
            ((Q4, 1400, 64, 65), "gemmw_q4_0_"), ((Q8, 1024, 64, 65), "gemmh_q8_0_m64_n64"), ((Q8, 2049, 64, 65), "gemmw_q8_0_"),
            ((Q8, 1400, 64, 97), "gemmw_q8_0_"), ((Q6, 1024, 64, 128), "gemmh_q6_k_m64_n64"), ((Q4K, 1025, 64, 128), "gemmw_q4_k_")]
    for (call, kernel), (_, names) in zip(want, launched(stub, [("gemm",) + c for c, _ in want])):
        assert any(n.startswith(kernel) for n in names), (call, kernel, names)


def test_two_workgroups(stub):
    """22003 rows, 257 tokens: two workgroups per CU, whole rounds and a split tail (test_gemm_wide.py runs them)."""
    kinds = {Q4: "q4_0", Q4K: "q4_k", Q6: "q6_k"}
    calls = [("gemm", k, 22003, nb, 257) for k in kinds for nb in (16, 24)]
    assert [n for _, n in launched(stub, calls)] == [["gemmw_prep", f"gemmw_{kinds[c[1]]}_i128", "gemm_reduce"] for c in calls]
