"""The workloads that the kernels' speed is judged on: what a decode engine has this library do.

A case is a dict of plain values; "path" says which part of the engine it is:

  step      a batch-1 decode step: every GEMV of one layer and the head, each on an f32 vector, captured once as
            a HIP graph and replayed (the library's own graph entry points), as a serving loop runs it
  gemv      one decode GEMV on an f32 vector, launched eagerly: what a host without graphs pays per operator
  batch     T vectors through one matrix: quantize the T rows, then the dispatcher (the verify kernels for the few
            vectors of a speculative step, the prefill GEMM for a prompt chunk)
  producers the fused Q8 producers of a prompt chunk: RMSNorm + Q8 and SwiGLU + Q8 over T rows

The sizes are those of the repository's benchmark configurations (7B-class 4096 / 11008 / 32000 and 27B-class
5120 / 17408 / 152064) and generic ones between and around them. draw() spreads over the same ranges.

The weights are random GGUF blocks in the benchmark's distributions, the activations normal with a few large
channels, as hidden states have. exact() dequantizes the GGUF blocks and multiplies in 64 bits; the Q8 quantization
of the activations is part of the operators' definition (d = amax / 127, q = round half away of x / d, in f32) and
is applied as defined.
"""
import os
import sys
from concurrent.futures import ThreadPoolExecutor

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amd.c_amd"))
import amdc  # noqa: E402

KIND = {"q4_0": amdc.KIND_Q4_0, "q8_0": amdc.KIND_Q8_0, "q4_k": amdc.KIND_Q4_K, "q6_k": amdc.KIND_Q6_K}
# weights per GGUF block, bytes per block
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q4_k": (256, 144), "q6_k": (256, 210)}
EPS = 1e-6


def listed():
    return [
        # a host without graphs: the attention output projection of a 7B-class layer, one eager launch
        {"name": "gemv_o_7b_q4_0", "path": "gemv", "kind": "q4_0", "rows": 4096, "cols": 4096, "res": True},
        # a decode step of a 7B-class Q4_0 file: wqkv, o, gate|up, down and the head, replayed
        {"name": "step_7b_q4_0", "path": "step", "mix": "q4_0", "hidden": 4096, "ffn": 11008, "vocab": 32000},
        # a decode step of a 27B-class Q4_K_M file: Q4_K attention and gate|up, Q6_K attn_v, ffn_down and head
        {"name": "step_27b_q4_k_m", "path": "step", "mix": "q4_k_m", "hidden": 5120, "ffn": 17408, "vocab": 152064},
        # a decode step of a small Q8_0 model (a draft model): every launch is short
        {"name": "step_draft_q8_0", "path": "step", "mix": "q8_0", "hidden": 2048, "ffn": 5632, "vocab": 32000},
        # speculative verify of 8 tokens: Q4_K gate / up
        {"name": "verify8_up_q4_k", "path": "batch", "kind": "q4_k", "rows": 17408, "cols": 5120, "T": 8, "res": False},
        # speculative verify of 5 tokens: Q6_K ffn_down with the residual
        {"name": "verify5_down_q6_k", "path": "batch", "kind": "q6_k", "rows": 5120, "cols": 17408, "T": 5, "res": True},
        # the end of a prompt: a short, ragged chunk
        {"name": "prefill77_up_q4_0", "path": "batch", "kind": "q4_0", "rows": 11008, "cols": 4096, "T": 77, "res": False},
        # the prompt chunk of the benchmark: Q4_K gate / up
        {"name": "prefill256_up_q4_k", "path": "batch", "kind": "q4_k", "rows": 17408, "cols": 5120, "T": 256, "res": False},
        # the same chunk through the Q6_K ffn_down of a Q4_K_M file
        {"name": "prefill256_down_q6_k", "path": "batch", "kind": "q6_k", "rows": 5120, "cols": 17408, "T": 256, "res": True},
        # a chunk of a 7B-class Q8_0 file
        {"name": "prefill384_down_q8_0", "path": "batch", "kind": "q8_0", "rows": 4096, "cols": 11008, "T": 384, "res": True},
        # a long prompt at once: gate|up as one matrix, the largest call
        {"name": "prefill1024_gateup_q4_k", "path": "batch", "kind": "q4_k", "rows": 34816, "cols": 5120, "T": 1024, "res": False},
        # the producers between the GEMMs of a chunk
        {"name": "producers256_27b", "path": "producers", "hidden": 5120, "ffn": 17408, "T": 256},
    ]


def _log(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    path = rng.choice(["step", "gemv", "batch", "batch", "batch", "batch", "producers"])
    if path == "step":
        mix = rng.choice(["q4_0", "q4_k_m", "q8_0"])
        hidden = 256 * rng.randint(8, 20)
        return {"path": path, "mix": mix, "hidden": hidden, "ffn": 256 * rng.randint(20, 68), "vocab": int(_log(rng, 16000, 100000))}
    kind = rng.choice(["q4_0", "q8_0", "q4_k", "q6_k"])
    rows = int(_log(rng, 1000, 36000))
    unit = BLOCK[kind][0]
    cols = unit * max(1, round(_log(rng, 1536, 17408) / unit))
    if path == "gemv":
        return {"path": path, "kind": kind, "rows": rows, "cols": cols, "res": rng.random() < 0.5}
    if path == "producers":
        return {"path": path, "hidden": 32 * rng.randint(64, 192), "ffn": 32 * rng.randint(128, 544), "T": int(_log(rng, 16, 640))}
    # vectors: from a speculative step's few to a whole chunk; the matrix smaller where the chunk is long
    T = int(_log(rng, 2, 1000))
    rows = min(rows, max(1000, int(17e10 / (T * cols))))
    return {"path": path, "kind": kind, "rows": rows, "cols": cols, "T": T, "res": rng.random() < 0.5}


# ---------------------------------------------------------------- inputs

def _mats(case):
    """(name, kind, rows, cols, residual) of a step's GEMVs, in the order an engine runs them."""
    h, f, v = case["hidden"], case["ffn"], case["vocab"]
    if case["mix"] == "q4_k_m":
        return [("attn_in", "q4_k", h + h // 5 // 32 * 32, h, False), ("attn_v", "q6_k", h // 5, h, False), ("attn_out", "q4_k", h, h + h // 5 // 256 * 256, True),
                ("gate_up", "q4_k", 2 * f, h, False), ("down", "q6_k", h, f, True), ("head", "q6_k", v, h, False)]
    k = case["mix"]
    return [("qkv", k, 3 * h, h, False), ("o", k, h, h, True), ("gate_up", k, 2 * f, h, False), ("down", k, h, f, True), ("head", k, v, h, False)]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 13)
    return g


def _gguf(kind, rows, cols, g):
    """Random GGUF blocks on the GPU, rows * cols / block of them: (n, bytes) uint8. Small normal scales, uniform quants."""
    per, size = BLOCK[kind]
    n = rows * cols // per
    blk = torch.randint(0, 256, (n, size), dtype=torch.uint8, device="cuda", generator=g)

    def f16(scale, count):
        d = torch.randn((n, count), device="cuda", generator=g).abs_().mul_(scale).half()
        return d.view(torch.uint8).view(n, 2 * count)

    if kind == "q4_0":
        blk[:, 0:2] = f16(0.02, 1)
    elif kind == "q8_0":
        blk[:, 0:2] = f16(0.004, 1)
    elif kind == "q4_k":
        blk[:, 0:4] = f16(0.01, 2)
    else:
        blk[:, 208:210] = f16(0.0005, 1)
    return blk


def _acts(T, n, g):
    """T x n f32 activations: normal, about one channel in 200 twenty times larger."""
    x = torch.randn((T, n), device="cuda", generator=g)
    big = torch.rand((n,), device="cuda", generator=g) < 0.005
    return torch.where(big, 20.0 * x, x).contiguous()


def _device_matrix(kind, rows, cols, blk):
    """The matrix as the engine holds it: repacked on the host (rows dealt to threads) and uploaded."""
    src = blk.cpu().numpy().reshape(rows, -1)
    parts = max(1, min(16, rows // 256))
    cut = [rows * i // parts for i in range(parts + 1)]
    with ThreadPoolExecutor(parts) as pool:
        got = list(pool.map(lambda i: torch.from_numpy(amdc.repack(KIND[kind], src[cut[i]:cut[i + 1]].reshape(-1), cut[i + 1] - cut[i], cols)), range(parts)))
    return torch.cat(got).cuda()


def _xs(cols):
    return (40 * (cols // 32) + 255) // 256 * 256


_engine_stream = None


def _stream():
    """The engine's one stream, on which its graphs are captured and replayed."""
    global _engine_stream
    if _engine_stream is None:
        _engine_stream = amdc.Stream()
    return _engine_stream


def prepare(case, seed):
    amdc.open_device()
    g = _gen(seed)
    if case["path"] == "producers":
        T, h, f = case["T"], case["hidden"], case["ffn"]
        s = {"case": case, "x": _acts(T, h, g), "w": 1.0 + 0.1 * torch.randn((h,), device="cuda", generator=g), "gate": _acts(T, f, g), "up": _acts(T, f, g)}
        s["y"], s["a"] = torch.empty((T, h), device="cuda"), torch.empty((T, f), device="cuda")
        s["yq"] = torch.zeros((T, _xs(h)), dtype=torch.uint8, device="cuda")
        s["aq"] = torch.zeros((T, _xs(f)), dtype=torch.uint8, device="cuda")
        return s
    if case["path"] == "step":
        ops = []
        for _, kind, rows, cols, res in _mats(case):
            w = _device_matrix(kind, rows, cols, _gguf(kind, rows, cols, g))
            x = _acts(1, cols, g)[0].contiguous()
            r = torch.randn((rows,), device="cuda", generator=g) if res else None
            ops.append((KIND[kind], w, x, torch.empty((rows,), device="cuda"), rows, cols // 32, r, torch.empty((_xs(cols),), dtype=torch.uint8, device="cuda")))

        def launch(stream):
            for kind, w, x, y, rows, nb, r, q in ops:
                amdc.gemv_x(kind, w.data_ptr(), x.data_ptr(), y.data_ptr(), rows, nb, res=r.data_ptr() if r is not None else None, q8=q.data_ptr(), stream=stream)

        torch.cuda.synchronize()
        st = _stream()
        launch(st.s)  # the workspaces of these sizes, before the capture
        st.sync()
        return {"case": case, "ops": ops, "graph": amdc.Graph(st, launch), "y": [o[3] for o in ops]}
    kind, rows, cols = case["kind"], case["rows"], case["cols"]
    T = case.get("T", 1)
    w = _device_matrix(kind, rows, cols, _gguf(kind, rows, cols, g))
    x = _acts(T, cols, g)
    r = torch.randn((T, rows), device="cuda", generator=g) if case["res"] else None
    return {"case": case, "w": w, "x": x, "r": r, "q": torch.zeros((T, _xs(cols)), dtype=torch.uint8, device="cuda"), "y": torch.empty((T, rows), device="cuda")}


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "step":
        state["graph"].launch()
        return state["y"]
    stream = torch.cuda.current_stream().cuda_stream
    if path == "producers":
        T, h, f = case["T"], case["hidden"], case["ffn"]
        amdc.rmsnorm_q8(state["x"].data_ptr(), state["w"].data_ptr(), state["y"].data_ptr(), h, EPS, state["yq"].data_ptr(), T, 4 * h, 4 * h, _xs(h), stream)
        state["a"].copy_(state["gate"])  # the SwiGLU works in place on the gate GEMM's output
        amdc.swiglu_q8(state["a"].data_ptr(), state["up"].data_ptr(), f, state["aq"].data_ptr(), T, 4 * f, _xs(f), stream)
        return {"y": state["y"], "yq": state["yq"], "a": state["a"], "aq": state["aq"]}
    kind, rows, nb = KIND[case["kind"]], case["rows"], case["cols"] // 32
    w, x, q, y, r = (state[k].data_ptr() if state[k] is not None else None for k in ("w", "x", "q", "y", "r"))
    if path == "gemv":
        amdc.gemv_x(kind, w, x, y, rows, nb, res=r, q8=q, stream=stream)
    else:
        T, xs = case["T"], _xs(case["cols"])
        amdc.quant_q8(x, q, nb, T, 128 * nb, xs, stream)
        amdc.op_gemv(kind, w, q, y, rows, nb, T, xs, rows, rows if r is not None else 0, res=r, stream=stream)
    return state["y"]


# ---------------------------------------------------------------- what a pass cannot do without, and its result in 64 bits

def _mat_work(kind, rows, cols, T, res):
    per, size = BLOCK[kind]
    return rows * cols // per * size + 4 * T * cols + 4 * T * rows * (2 if res else 1), 2 * T * rows * cols


def work(case):
    if case["path"] == "producers":
        T, h, f = case["T"], case["hidden"], case["ffn"]
        # x and w in, y and its Q8 copy out; gate and up in, the product and its Q8 copy out
        return {"bytes": T * h * 8 + 4 * h + T * h // 32 * 40 + T * f * 12 + T * f // 32 * 40, "flops": 10 * T * (h + f)}
    if case["path"] == "step":
        each = [_mat_work(k, r, c, 1, s) for _, k, r, c, s in _mats(case)]
    else:
        each = [_mat_work(case["kind"], case["rows"], case["cols"], case.get("T", 1), case["res"])]
    return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}


def tolerance(case):
    # exact integer block dots, then f32 sums over the blocks of a row: 0.8e-7 (decode) to 2.5e-7 (prefill) against 64 bits measured
    return {"rel": 1e-6, "max": 4e-5}


def _dequant(kind, blk):
    """GGUF blocks (n, bytes) -> (n, weights) f64."""
    n = blk.shape[0]

    def f16(lo):
        return blk[:, lo:lo + 2].contiguous().view(torch.float16).double()

    if kind == "q4_0":
        b = blk[:, 2:].to(torch.int16)
        return f16(0) * (torch.cat([b & 15, b >> 4], 1).double() - 8.0)
    if kind == "q8_0":
        return f16(0) * blk[:, 2:].contiguous().view(torch.int8).double()
    if kind == "q4_k":
        s = blk[:, 4:16].to(torch.int16)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        b = blk[:, 16:].to(torch.int16).view(n, 4, 1, 32)
        q = torch.cat([b & 15, b >> 4], 2).view(n, 8, 32).double()
        return ((f16(0) * sc)[:, :, None] * q - (f16(2) * mn)[:, :, None]).view(n, 256)
    ql, qh = blk[:, 0:128].to(torch.int16).view(n, 2, 2, 32), blk[:, 128:192].to(torch.int16).view(n, 2, 1, 32)
    lo = torch.cat([ql & 15, ql >> 4], 2)
    hi = torch.cat([(qh >> (2 * m)) & 3 for m in range(4)], 2)
    q = (lo | (hi << 4)).view(n, 16, 16).double() - 32.0
    sc = blk[:, 192:208].contiguous().view(torch.int8).double()
    return ((f16(208) * sc)[:, :, None] * q).view(n, 256)


def _quantized(x):
    """The activations as the operators define their Q8 copy, as f64 (d q per block of 32)."""
    b = x.cpu().view(x.shape[0], -1, 32)
    d = b.abs().amax(2, keepdim=True) / torch.tensor(127.0)
    v = torch.where(d > 0, b / torch.where(d > 0, d, torch.ones_like(d)), torch.zeros_like(b)).double()
    return (d.double() * (v.sign() * (v.abs() + 0.5).floor())).view(x.shape).cuda()


def _product(kind, rows, cols, blk, x):
    """T x rows f64: the quantized activations times the dequantized weights, a slice of rows at a time."""
    a = _quantized(x)
    y = torch.empty((x.shape[0], rows), dtype=torch.float64, device="cuda")
    per = cols // BLOCK[kind][0]
    step = max(1, (1 << 28) // (8 * cols))
    for r in range(0, rows, step):
        e = min(rows, r + step)
        y[:, r:e] = a @ _dequant(kind, blk[r * per:e * per]).view(e - r, cols).t()
    return y


def exact(case, seed):
    g = _gen(seed)
    if case["path"] == "producers":
        T, h, f = case["T"], case["hidden"], case["ffn"]
        x = _acts(T, h, g).double()
        w = (1.0 + 0.1 * torch.randn((h,), device="cuda", generator=g)).double()
        gate, up = _acts(T, f, g).double(), _acts(T, f, g).double()
        y = x / (x.square().mean(1, keepdim=True) + EPS).sqrt() * w
        return {"y": y, "yq": None, "a": gate / (1.0 + (-gate).exp()) * up, "aq": None}
    if case["path"] == "step":
        out = []
        for _, kind, rows, cols, res in _mats(case):
            blk = _gguf(kind, rows, cols, g)
            y = _product(kind, rows, cols, blk, _acts(1, cols, g))[0]
            out.append(y + torch.randn((rows,), device="cuda", generator=g).double() if res else y)
        return out
    kind, rows, cols, T = case["kind"], case["rows"], case["cols"], case.get("T", 1)
    blk = _gguf(kind, rows, cols, g)
    y = _product(kind, rows, cols, blk, _acts(T, cols, g))
    return y + torch.randn((T, rows), device="cuda", generator=g).double() if case["res"] else y
