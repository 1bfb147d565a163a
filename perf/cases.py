"""The work that programs bring to this library, as cases that can be timed and checked.

Each case is one pass through the public entry points (``vkblas_amd.gemm_async`` /
``gemm_ex_async`` or the hipBLAS ABI of ``vkblas_amd.hipblas()``), with operands and handle in
hand before the call:

``linear``     y = x W^T + bias, W stored N x K (PyTorch's ``linear``), engine entry with the bias epilogue
``train``      the three products of a linear layer's training step (y, dx, and dW accumulated
               in fp32), hipBLAS GemmEx
``attention``  q k^T / sqrt(d) and p v over batch x heads, hipBLAS GemmStridedBatchedEx
``decode``     a gated MLP's gate, up and down projections for a few tokens (weights N x K), engine entry
``xw``         y = x w with the weight stored K x N (PyTorch's ``x @ w``), engine entry
``square``     C = A B, column-major, hipblasSgemm (fp32) or GemmEx
``longk``      a small product over a very long K (a weight gradient over many samples), engine entry

Sizes are those of the repository's benchmark, configurations and tests where it has them, and
generic layer sizes elsewhere.
"""
import ctypes
import math

import torch

import vkblas_amd as vk
from vkblas_amd import hipblas_abi as hb

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
ENGINE = {"f32": vk.DT_F32, "f16": vk.DT_F16, "bf16": vk.DT_BF16}
HIP = {"f32": hb.HIP_R_32F, "f16": hb.HIP_R_16F, "bf16": hb.HIP_R_16BF}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # the smallest call: one layer of a small fp32 network on a small batch; launch latency
        {"name": "linear_f32_small", "op": "linear", "dtype": "f32", "m": 64, "n": 128, "k": 256},
        # an output layer over an odd number of classes: C's rows have no alignment
        {"name": "linear_f16_classes", "op": "linear", "dtype": "f16", "m": 128, "n": 32003, "k": 1024},
        # a training step of a small fp32 layer whose sizes are multiples of no tile
        {"name": "train_f32_ragged", "op": "train", "dtype": "f32", "m": 200, "n": 500, "k": 784},
        # a training step of a mid-size transformer layer on a short batch: too few tiles to fill the chip
        {"name": "train_bf16_mid", "op": "train", "dtype": "bf16", "m": 512, "n": 4096, "k": 1024},
        # a training step of a large transformer layer on 8192 tokens: the largest case
        {"name": "train_bf16_large", "op": "train", "dtype": "bf16", "m": 8192, "n": 11008, "k": 4096},
        # attention products of a training batch
        {"name": "attention_bf16", "op": "attention", "dtype": "bf16", "batch": 64, "s": 1024, "d": 64},
        # the same for an odd sequence length: the rows of p have no alignment
        {"name": "attention_f16_odd", "op": "attention", "dtype": "f16", "batch": 96, "s": 197, "d": 64},
        # a prompt of 2047 tokens through a large projection (the benchmark's ragged shape)
        {"name": "linear_f16_prompt", "op": "linear", "dtype": "f16", "m": 2047, "n": 14336, "k": 4096},
        # the benchmark's headline product
        {"name": "square_f32", "op": "square", "dtype": "f32", "n": 4096},
        # one token through an MLP: its three weights are read once
        {"name": "decode_f16_one", "op": "decode", "dtype": "f16", "m": 1, "n": 14336, "k": 4096},
        # a batch of 32 sequences decoding against a weight stored K x N (the benchmark's wide decode)
        {"name": "xw_f16_batch", "op": "xw", "dtype": "f16", "m": 32, "n": 8192, "k": 8192},
        # the benchmark's long reduction, K split by the planner
        {"name": "longk_f16", "op": "longk", "dtype": "f16", "m": 256, "n": 256, "k": 65536},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi):
    """A size between lo and hi: a multiple of 64, a multiple of 8, or any number."""
    v = _log(rng, lo, hi)
    step = rng.choice((64, 64, 8, 1))
    return int(min(hi, max(lo, step * max(1, round(v / step)))))


def draw(rng):
    while True:
        op = rng.choice(("linear", "linear", "train", "train", "attention", "decode", "xw", "square", "longk"))
        dtype = rng.choice(("f16", "bf16", "f32"))
        c = {"op": op, "dtype": dtype}
        if op == "linear":
            c.update(m=_size(rng, 8, 4096), n=_size(rng, 64, 32768), k=_size(rng, 64, 8192))
        elif op == "train":
            c.update(m=_size(rng, 64, 8192), n=_size(rng, 64, 11008), k=_size(rng, 64, 8192))
        elif op == "attention":
            c.update(batch=int(_log(rng, 4, 128)), s=_size(rng, 32, 2048), d=rng.choice((32, 64, 72, 80, 96, 128)))
        elif op == "decode":
            c.update(m=int(_log(rng, 1, 65)), n=64 * int(_log(rng, 16, 225)), k=64 * int(_log(rng, 16, 129)))
        elif op == "xw":
            c.update(m=int(_log(rng, 1, 65)), n=64 * int(_log(rng, 16, 225)), k=64 * int(_log(rng, 16, 225)))
        elif op == "square":
            c.update(n=_size(rng, 96, 4096))
        else:
            c.update(m=64 * int(_log(rng, 1, 9)), n=64 * int(_log(rng, 1, 9)), k=1024 * int(_log(rng, 8, 129)))
        w = work(c)
        flops = 137.5e9 if dtype == "f32" else 2.21e12   # no more than the largest listed of the type
        if w["flops"] <= flops and 2e5 <= w["bytes"] <= 8e8:
            return c


def work(case):
    es = SIZE[case["dtype"]]
    op = case["op"]
    if op == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": es * (m * k + n * k + m * n + n), "flops": 2 * m * n * k}
    if op == "train":
        m, n, k = case["m"], case["n"], case["k"]
        # x, W and dy read once, y and dx written once, dW (fp32) read and written
        return {"bytes": es * 2 * (m * k + m * n) + es * n * k + 8 * n * k, "flops": 6 * m * n * k}
    if op == "attention":
        b, s, d = case["batch"], case["s"], case["d"]
        return {"bytes": es * b * (4 * s * d + 2 * s * s), "flops": 4 * b * s * s * d}
    if op == "decode":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": es * (3 * n * k + 2 * m * k + 3 * m * n), "flops": 6 * m * n * k}
    if op == "square":
        n = case["n"]
        return {"bytes": es * 3 * n * n, "flops": 2 * n ** 3}
    m, n, k = case["m"], case["n"], case["k"]
    es_c = 4 if op == "longk" else es
    return {"bytes": es * (m * k + n * k) + es_c * m * n, "flops": 2 * m * n * k}


def tolerance(case):
    # About four times what results differ by from float64 rounded to the result's type, over 42
    # cases: two correct orders of the fp32 sums turn a rare last bit of a 16-bit result (rel up
    # to 1.5e-5 in fp16 and 5.1e-5 in bf16, max one spacing of the type: 9.8e-4 and 7.8e-3), and
    # move an fp32 one by up to 1.1e-6 (max 1e-5), sums of 16-bit products by 2.2e-7.
    if case["dtype"] == "f32":
        return {"rel": 5e-6, "max": 5e-5}
    if case["op"] == "longk":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 6e-5, "max": 4e-3} if case["dtype"] == "f16" else {"rel": 2e-4, "max": 0.03}


_handle = None


def _hipblas():
    """The process's hipBLAS handle, on the stream that PyTorch runs on."""
    global _handle
    abi = vk.hipblas()
    if _handle is None:
        _handle = abi.create()
    if abi.hipblasSetStream(_handle, torch.cuda.current_stream().cuda_stream) != hb.HIPBLAS_STATUS_SUCCESS:
        raise RuntimeError("hipblasSetStream failed")
    return abi, _handle


def _inputs(case, seed):
    """The operands, by name: unit-scale activations, weights that keep that scale."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = TORCH[case["dtype"]]
    op = case["op"]

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, device="cuda", generator=g) * scale).to(dt)

    if op == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"x": normal(m, k), "w": normal(n, k, scale=k ** -0.5), "bias": normal(n, scale=0.1)}
    if op == "train":
        m, n, k = case["m"], case["n"], case["k"]
        return {"x": normal(m, k), "w": normal(n, k, scale=k ** -0.5), "dy": normal(m, n, scale=0.1),
                "dw": torch.randn(n, k, device="cuda", generator=g) * 0.1 * m ** 0.5}
    if op == "attention":
        b, s, d = case["batch"], case["s"], case["d"]
        q, kk, v = normal(b, s, d), normal(b, s, d), normal(b, s, d)
        p = torch.softmax(torch.randn(b, s, s, device="cuda", generator=g), dim=-1).to(dt)
        return {"q": q, "k": kk, "v": v, "p": p}
    if op == "decode":
        m, n, k = case["m"], case["n"], case["k"]
        return {"x": normal(m, k), "gate": normal(n, k, scale=k ** -0.5), "up": normal(n, k, scale=k ** -0.5),
                "h": normal(m, n, scale=0.5), "down": normal(k, n, scale=n ** -0.5)}
    if op == "square":
        n = case["n"]
        u = torch.rand(2, n, n, device="cuda", generator=g) * 2 - 1
        return {"a": u[0].to(dt).contiguous(), "b": u[1].to(dt).contiguous()}
    m, n, k = case["m"], case["n"], case["k"]
    if op == "xw":
        return {"x": normal(m, k), "w": normal(k, n, scale=k ** -0.5)}
    # longk: A^T B over k samples, both stored k x features
    return {"a": normal(k, m), "b": normal(k, n)}


def prepare(case, seed):
    vk.load()
    s = {"case": case}
    s.update(_inputs(case, seed))
    dt = TORCH[case["dtype"]]

    def empty(*shape, dtype=dt):
        return torch.empty(*shape, device="cuda", dtype=dtype)

    op = case["op"]
    if op in ("linear", "xw"):
        s["y"] = empty(case["m"], case["n"])
    elif op == "train":
        s["y"], s["dx"] = empty(case["m"], case["n"]), empty(case["m"], case["k"])
    elif op == "attention":
        s["scores"] = empty(case["batch"], case["s"], case["s"])
        s["ctx"] = empty(case["batch"], case["s"], case["d"])
    elif op == "decode":
        s["y_gate"], s["y_up"] = empty(case["m"], case["n"]), empty(case["m"], case["n"])
        s["y"] = empty(case["m"], case["k"])
    elif op == "square":
        s["c"] = empty(case["n"], case["n"])
    else:
        s["c"] = empty(case["m"], case["n"], dtype=torch.float32)
    if op in ("train", "attention", "square"):
        s["abi"], s["handle"] = _hipblas()
        s["one"], s["zero"] = ctypes.c_float(1.0), ctypes.c_float(0.0)
        s["scale"] = ctypes.c_float(case["d"] ** -0.5 if op == "attention" else 1.0)
    return s


def _ok(status):
    if status != hb.HIPBLAS_STATUS_SUCCESS:
        raise RuntimeError(f"hipBLAS call failed: {status}")


def _gemm_ex(s, ta, tb, m, n, k, a, lda, b, ldb, beta, c, ldc, ct):
    """hipblasGemmEx, column-major, fp32 compute."""
    t = HIP[s["case"]["dtype"]]
    _ok(s["abi"].hipblasGemmEx(s["handle"], ta, tb, m, n, k, ctypes.byref(s["one"]), a.data_ptr(), t, lda,
                               b.data_ptr(), t, ldb, ctypes.byref(beta), c.data_ptr(), ct, ldc,
                               hb.HIPBLAS_COMPUTE_32F, hb.HIPBLAS_GEMM_DEFAULT))


def run(s):
    case = s["case"]
    op, et = case["op"], ENGINE[case["dtype"]]
    N, T = hb.HIPBLAS_OP_N, hb.HIPBLAS_OP_T
    stream = torch.cuda.current_stream().cuda_stream
    if op == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        vk.gemm_ex_async(et, et, vk.OP_N, vk.OP_T, m, n, k, 1.0, s["x"].data_ptr(), k, s["w"].data_ptr(), k, 0.0,
                         s["y"].data_ptr(), n, bias=s["bias"].data_ptr(), bias_type=et, stream=stream)
        return s["y"]
    if op == "train":
        m, n, k, t = case["m"], case["n"], case["k"], HIP[case["dtype"]]
        # row-major y = x W^T, dx = dy W, dW += dy^T x, as hipBLAS's column-major products
        _gemm_ex(s, T, N, n, m, k, s["w"], k, s["x"], k, s["zero"], s["y"], n, t)
        _gemm_ex(s, N, N, k, m, n, s["w"], k, s["dy"], n, s["zero"], s["dx"], k, t)
        _gemm_ex(s, N, T, k, n, m, s["x"], k, s["dy"], n, s["one"], s["dw"], k, hb.HIP_R_32F)
        return {"y": s["y"], "dx": s["dx"], "dw": s["dw"]}
    if op == "attention":
        b, L, d, t = case["batch"], case["s"], case["d"], HIP[case["dtype"]]
        batched = s["abi"].hipblasGemmStridedBatchedEx
        _ok(batched(s["handle"], T, N, L, L, d, ctypes.byref(s["scale"]), s["k"].data_ptr(), t, d, L * d,
                    s["q"].data_ptr(), t, d, L * d, ctypes.byref(s["zero"]), s["scores"].data_ptr(), t, L, L * L, b,
                    hb.HIPBLAS_COMPUTE_32F, hb.HIPBLAS_GEMM_DEFAULT))
        _ok(batched(s["handle"], N, N, d, L, L, ctypes.byref(s["one"]), s["v"].data_ptr(), t, d, L * d,
                    s["p"].data_ptr(), t, L, L * L, ctypes.byref(s["zero"]), s["ctx"].data_ptr(), t, d, L * d, b,
                    hb.HIPBLAS_COMPUTE_32F, hb.HIPBLAS_GEMM_DEFAULT))
        return {"scores": s["scores"], "ctx": s["ctx"]}
    if op == "decode":
        m, n, k = case["m"], case["n"], case["k"]
        for w, y in (("gate", "y_gate"), ("up", "y_up")):
            vk.gemm_async(et, et, vk.OP_N, vk.OP_T, m, n, k, 1.0, s["x"].data_ptr(), k, s[w].data_ptr(), k, 0.0,
                          s[y].data_ptr(), n, stream=stream)
        vk.gemm_async(et, et, vk.OP_N, vk.OP_T, m, k, n, 1.0, s["h"].data_ptr(), n, s["down"].data_ptr(), n, 0.0,
                      s["y"].data_ptr(), k, stream=stream)
        return {"gate": s["y_gate"], "up": s["y_up"], "y": s["y"]}
    if op == "xw":
        m, n, k = case["m"], case["n"], case["k"]
        vk.gemm_async(et, et, vk.OP_N, vk.OP_N, m, n, k, 1.0, s["x"].data_ptr(), k, s["w"].data_ptr(), n, 0.0,
                      s["y"].data_ptr(), n, stream=stream)
        return s["y"]
    if op == "square":
        n = case["n"]
        if case["dtype"] == "f32":
            _ok(s["abi"].hipblasSgemm(s["handle"], N, N, n, n, n, ctypes.byref(s["one"]), s["a"].data_ptr(), n,
                                      s["b"].data_ptr(), n, ctypes.byref(s["zero"]), s["c"].data_ptr(), n))
        else:
            _gemm_ex(s, N, N, n, n, n, s["a"], n, s["b"], n, s["zero"], s["c"], n, HIP[case["dtype"]])
        return s["c"]
    m, n, k = case["m"], case["n"], case["k"]
    vk.gemm_async(et, vk.DT_F32, vk.OP_T, vk.OP_N, m, n, k, 1.0, s["a"].data_ptr(), m, s["b"].data_ptr(), n, 0.0,
                  s["c"].data_ptr(), n, stream=stream)
    return s["c"]


def exact(case, seed):
    """What run() returns, in float64 by PyTorch."""
    v = {name: t.double() for name, t in _inputs(case, seed).items()}
    op = case["op"]
    if op == "linear":
        return v["x"] @ v["w"].t() + v["bias"]
    if op == "train":
        return {"y": v["x"] @ v["w"].t(), "dx": v["dy"] @ v["w"], "dw": v["dw"] + v["dy"].t() @ v["x"]}
    if op == "attention":
        # one product at a time: the batch's scores in float64 may be large
        scores = torch.stack([a @ b.t() for a, b in zip(v["q"], v["k"])]) * case["d"] ** -0.5
        return {"scores": scores, "ctx": torch.stack([a @ b for a, b in zip(v["p"], v["v"])])}
    if op == "decode":
        return {"gate": v["x"] @ v["gate"].t(), "up": v["x"] @ v["up"].t(), "y": v["h"] @ v["down"].t()}
    if op == "square":
        # column-major A B is, read row by row, B A
        return v["b"] @ v["a"]
    if op == "xw":
        return v["x"] @ v["w"]
    return v["a"].t() @ v["b"]
