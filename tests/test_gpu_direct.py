"""gemm_direct_kernel (small tiles, fragments straight from memory) at the
edges of its tiles: one past and one short of a tile, one k, K around its K
step (16 fp32, 32 16-bit) and around a whole round of loads in flight, every
layout and type pair, odd leading dimensions with NaN in the padding,
operands one element off any alignment, batches, beta with C in place or
apart, a bias; against the CPU oracle.  C's padding must come back untouched.  Split-K
pass 1 with a ragged last slice."""
import numpy as np
import pytest
import torch

import oracle
from gpu_helpers import (BACK, BF16_BOUND, CONV, ENGINE, F16_BOUND, f32_bound, normwise, patterns,
                         to_dev_as as _dev)

pytestmark = pytest.mark.gpu

TYPES = [("f32", "f32"), ("f32", "f16"), ("f32", "bf16"), ("f16", "f16"), ("f16", "f32"), ("bf16", "bf16"),
         ("bf16", "f32")]
# M, N, K, batch.  64 x 64 tiles from 144 of them on, else 32 x 32 (fp32 with
# fewer than 128 of those: 16 x 32)
SHAPES = [(33, 32, 1, 1), (65, 47, 15, 1), (95, 33, 33, 2), (129, 65, 64, 3),   # 16 x 32 (fp32) / 32 x 32
          (193, 191, 129, 4),                                                   # 32 x 32
          (65, 64, 257, 72), (129, 127, 511, 36), (193, 321, 1027, 7)]           # 64 x 64


@pytest.mark.parametrize("form", ["plain", "apart", "in_place"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("op_a,op_b", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("ab,ct", TYPES)
def test_direct(ab, ct, op_a, op_b, shape, form):
    import vkblas_amd as vk
    M, N, K, batch = shape
    print(f"[case] direct {ab}>{ct} op={op_a}{op_b} {shape} {form}", flush=True)
    r = np.random.default_rng(M + 3 * N + 7 * K + batch)
    # odd leading dimensions, every matrix one element off its buffer's start
    ra, ca = (K, M) if op_a else (M, K)
    rb, cb = (N, K) if op_b else (K, N)
    lda, ldb, ldc = ca + 1 - ca % 2 + 2, cb + 1 - cb % 2 + 4, N + 1 - N % 2 + 2
    sa, sb, sc = lda * ra + 1, ldb * rb + 3, ldc * M + 5

    def operand(rows, cols, ld, stride):
        x = np.full(1 + stride * batch, np.nan, np.float32)
        for i in range(batch):
            x[1 + i * stride:][:ld * rows].reshape(rows, ld)[:, :cols] = r.uniform(-1, 1, (rows, cols))
        return x
    a, b = CONV[ab](operand(ra, ca, lda, sa)), CONV[ab](operand(rb, cb, ldb, sb))
    c0 = CONV[ct](r.uniform(-1, 1, 1 + sc * batch).astype(np.float32))
    cin = CONV[ct](r.uniform(-1, 1, 1 + sc * batch).astype(np.float32))
    bias = CONV[ab](r.uniform(-1, 1, N).astype(np.float32))
    alpha, beta = 1.25, 0.0 if form == "plain" else -0.5
    if form == "plain":                  # beta == 0 never reads C
        for i in range(batch):
            c0[1 + i * sc:][:ldc * M].reshape(M, ldc)[:, :N] = CONV[ct](np.full(1, np.nan, np.float32))[0]
    want = c0.copy()
    for i in range(batch):
        src = (cin if form == "apart" else want)[1 + i * sc:][:ldc * M].copy()
        out = want[1 + i * sc:][:ldc * M].copy()
        oracle.ref_gemm_epi_rm(ab, ct, op_a, op_b, M, N, K, np.ascontiguousarray(a[1 + i * sa:][:lda * ra]), lda,
                               np.ascontiguousarray(b[1 + i * sb:][:ldb * rb]), ldb, alpha, beta, src, ldc, out, ldc,
                               BACK[ab](bias))
        want[1 + i * sc:][:ldc * M] = out
    dt = ENGINE
    dA, dB, dC, dI, dBias = _dev(a, ab), _dev(b, ab), _dev(c0, ct), _dev(cin, ct), _dev(bias, ab)
    ea, ec = dA.element_size(), dC.element_size()
    vk.gemm_ex_async(dt[ab], dt[ct], op_a, op_b, M, N, K, alpha, dA.data_ptr() + ea, lda, dB.data_ptr() + ea, ldb,
                     beta, dC.data_ptr() + ec, ldc, batch=batch, stride_a=sa, stride_b=sb, stride_c=sc,
                     c_in=dI.data_ptr() + ec if form == "apart" else None, ldc_in=ldc if form == "apart" else 0,
                     stride_c_in=sc if form == "apart" else 0, bias=dBias.data_ptr(), bias_type=dt[ab])
    torch.cuda.synchronize()
    assert vk.last_kernel() == vk.KERNEL_DIRECT, vk.last_kernel()
    got = patterns(dC)
    bound = BF16_BOUND if ct == "bf16" else F16_BOUND if "f16" in (ab, ct) or ab == "bf16" else f32_bound(K)
    for i in range(batch):
        g = BACK[ct](got[1 + i * sc:][:ldc * M]).reshape(M, ldc)
        w = BACK[ct](want[1 + i * sc:][:ldc * M]).reshape(M, ldc)
        assert np.array_equal(g[:, N:], w[:, N:]), "C padding written"
        assert np.all(np.isfinite(g[:, :N]))
        assert normwise(g[:, :N], w[:, :N]) <= bound, i


@pytest.mark.parametrize("form", ["plain", "in_place"])
@pytest.mark.parametrize("M,N,K,split", [(33, 35, 1000, 3), (97, 65, 2003, 4), (193, 129, 777, 2)])
@pytest.mark.parametrize("op_a,op_b", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("ab,ct", [("f32", "f32"), ("f16", "f16"), ("bf16", "f32")])
def test_direct_split(ab, ct, op_a, op_b, M, N, K, split, form):
    """pass 1 of a caller's split: slices that start past k 0, the last one shorter"""
    import vkblas_amd as vk
    print(f"[case] direct split {ab}>{ct} op={op_a}{op_b} {M}x{N}x{K}/{split} {form}", flush=True)
    r = np.random.default_rng(M + 3 * N + 7 * K)
    ra, lda = (K, M) if op_a else (M, K)
    rb, ldb = (N, K) if op_b else (K, N)
    a, b, c = (CONV[t](r.uniform(-1, 1, 1 + n).astype(np.float32))
               for t, n in ((ab, ra * lda), (ab, rb * ldb), (ct, M * N)))
    beta = 0.0 if form == "plain" else -0.5
    want = c[1:].copy()
    oracle.ref_gemm_epi_rm(ab, ct, op_a, op_b, M, N, K, a[1:].copy(), lda, b[1:].copy(), ldb, 1.25, beta, want.copy(),
                           N, want, N, None)
    dA, dB, dC = _dev(a, ab), _dev(b, ab), _dev(c, ct)
    vk.gemm_async(ENGINE[ab], ENGINE[ct], op_a, op_b, M, N, K, 1.25, dA.data_ptr() + dA.element_size(), lda,
                  dB.data_ptr() + dB.element_size(), ldb, beta, dC.data_ptr() + dC.element_size(), N, split_k=split)
    assert (vk.last_path(), vk.last_kernel()) == (vk.PATH_SPLITK, vk.KERNEL_DIRECT), vk.last_kernel()
    got = patterns(dC)
    assert got[0] == c[0], "the element in front of C written"
    bound = BF16_BOUND if ct == "bf16" else f32_bound(K) if ab == "f32" else F16_BOUND
    assert normwise(BACK[ct](got[1:].copy()), BACK[ct](want)) <= bound


# type, op_a, op_b, M, N, K, batch, kernel: both sides of the lines in tiles of 64 x 64
@pytest.mark.parametrize("ab,op_a,op_b,M,N,K,batch,kernel", [
    ("f32", 0, 1, 576, 64, 320, 15, "DIRECT"), ("f32", 0, 1, 576, 64, 320, 16, "GENERIC"),      # whole tiles, NT: 144
    ("f16", 0, 1, 320, 192, 192, 6, "DIRECT"), ("f16", 0, 1, 256, 384, 192, 4, "GENERIC"),      # 16 bits: 96
    ("f32", 1, 0, 640, 64, 128, 16, "DIRECT"), ("f32", 1, 0, 768, 64, 128, 16, "GENERIC"),      # others: 192
    ("f32", 1, 0, 448, 64, 64, 20, "DIRECT"), ("f32", 1, 0, 576, 64, 64, 16, "GENERIC"),        # a short K: 144
    # edges, K below 512 bytes: 256 tiles
    ("f16", 1, 1, 343, 13, 5, 42, "DIRECT"), ("f16", 1, 1, 343, 13, 5, 43, "GENERIC_CHECKED"),
    ("f32", 0, 0, 7, 509, 127, 32, "DIRECT"), ("f32", 0, 0, 7, 509, 127, 33, "GENERIC_CHECKED"),
    ("f32", 0, 0, 7, 509, 128, 33, "DIRECT")])
def test_line_against_the_generic_kernel(ab, op_a, op_b, M, N, K, batch, kernel):
    import vkblas_amd as vk
    print(f"[case] line {ab} op={op_a}{op_b} {M}x{N}x{K} x{batch}", flush=True)
    r = np.random.default_rng(M + 3 * N + 7 * K)
    lda, ldb = (M if op_a else K), (K if op_b else N)
    a, b = (CONV[ab](r.uniform(-1, 1, batch * n).astype(np.float32)) for n in (M * K, N * K))
    want = CONV[ab](np.zeros(M * N, np.float32))
    oracle.ref_gemm_epi_rm(ab, ab, op_a, op_b, M, N, K, a[-M * K:].copy(), lda, b[-N * K:].copy(), ldb, 1.25, 0.0,
                           want.copy(), N, want, N, None)
    dA, dB, dC = _dev(a, ab), _dev(b, ab), _dev(CONV[ab](np.zeros(batch * M * N, np.float32)), ab)
    vk.gemm_async(ENGINE[ab], ENGINE[ab], op_a, op_b, M, N, K, 1.25, dA.data_ptr(), lda, dB.data_ptr(), ldb, 0.0,
                  dC.data_ptr(), N, batch=batch, stride_a=M * K, stride_b=N * K, stride_c=M * N)
    assert vk.last_kernel() == getattr(vk, "KERNEL_" + kernel), vk.last_kernel()
    got = patterns(dC)[-M * N:].copy()
    assert normwise(BACK[ab](got), BACK[ab](want)) <= (f32_bound(K) if ab == "f32" else F16_BOUND)
