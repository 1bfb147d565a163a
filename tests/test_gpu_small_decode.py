"""Decode plans on either side of the lines between gemm_direct_kernel and the decode
kernels: vkblas_last_kernel names the kernel that ran, vkblas_last_path stays the
plan's, and the result agrees with the CPU oracle."""
import numpy as np
import pytest
import torch

import oracle
from gpu_helpers import BACK, BF16_BOUND, CONV, ENGINE, F16_BOUND, f32_bound, normwise, patterns

pytestmark = pytest.mark.gpu

# type, op_b (1: weight N x K), M, N, K, whether gemm_direct_kernel runs it
CASES = [
    ("f32", 1, 64, 128, 256, True), ("f32", 1, 17, 1000, 1028, True), ("f32", 0, 16, 260, 33, True),
    ("f16", 1, 17, 1000, 1032, True), ("bf16", 0, 4, 776, 7, True), ("f16", 0, 64, 136, 33, True),
    ("f32", 1, 16, 128, 256, False),        # up to 16 rows against N x K
    ("f32", 1, 20, 28, 13, False), ("f16", 0, 8, 24, 64, False),        # fewer than 32 columns
    ("f16", 1, 40, 1000, 2056, False), ("f16", 0, 40, 1000, 2056, False),   # K past 2048
    ("f32", 0, 16, 4096, 260, False), ("bf16", 1, 64, 8192, 520, False),    # weight past the line
]
# the lines in N (8192, 16-bit K x N 16384), in K (fp32 1280), in tiles (16-bit N x K) and
# of one or two rows
LINES = [
    ("f32", 1, 17, 8192, 8, True), ("f32", 1, 17, 8200, 8, False), ("f32", 0, 4, 8192, 16, True),
    ("f32", 0, 4, 8200, 16, False), ("f16", 1, 20, 8192, 16, True), ("f16", 1, 20, 8200, 16, False),
    ("f16", 0, 2, 16384, 24, True), ("f16", 0, 2, 16392, 24, False), ("bf16", 0, 8, 42616, 32, False),
    ("f32", 1, 33, 96, 1280, True), ("f32", 1, 33, 96, 1284, False), ("f32", 0, 16, 40, 1284, False),
    ("f16", 1, 33, 4096, 520, True), ("f16", 1, 33, 4104, 520, False), ("f16", 1, 33, 4104, 512, True),
    ("f32", 0, 2, 256, 32, False), ("f32", 0, 2, 256, 36, True), ("f32", 0, 3, 256, 32, True),
]


def _run(ab, op_b, M, N, K, lda, ldb, kernel):
    import vkblas_amd as vk
    r = np.random.default_rng(M + 3 * N + 7 * K)
    rows_b, cols_b = (N, K) if op_b else (K, N)
    a, b = (CONV[ab](r.uniform(-1, 1, n).astype(np.float32)) for n in (M * K, rows_b * cols_b))
    want = CONV[ab](np.zeros(M * N, np.float32))
    oracle.ref_gemm_epi_rm(ab, ab, 0, op_b, M, N, K, a, K, b, cols_b, 1.25, 0.0, want.copy(), N, want, N, None)
    t = ENGINE[ab]
    dt = torch.float32 if ab == "f32" else torch.int16
    dA, dB = (torch.empty((rows - 1) * ld + cols, dtype=dt, device="cuda:0")
              for rows, cols, ld in ((M, K, lda), (rows_b, cols_b, ldb)))
    for d, h, rows, cols, ld in ((dA, a, M, K, lda), (dB, b, rows_b, cols_b, ldb)):
        d.as_strided((rows, cols), (ld, 1)).copy_(torch.from_numpy(h.view(np.int16) if ab != "f32" else h)
                                                  .reshape(rows, cols))
    dC = torch.zeros(M * N, dtype=dt, device="cuda:0")
    vk.gemm_async(t, t, 0, op_b, M, N, K, 1.25, dA.data_ptr(), lda, dB.data_ptr(), ldb, 0.0, dC.data_ptr(), N)
    assert vk.last_path() == vk.PATH_SKINNY
    assert vk.last_kernel() == kernel, vk.last_kernel()
    bound = f32_bound(K) if ab == "f32" else F16_BOUND if ab == "f16" else BF16_BOUND
    assert normwise(BACK[ab](patterns(dC)), BACK[ab](want)) <= bound


@pytest.mark.parametrize("case", CASES + LINES, ids=lambda c: "{}_op{}_{}x{}x{}_{}".format(*c))
def test_kernel_and_result(case):
    import vkblas_amd as vk
    ab, op_b, M, N, K, direct = case
    print(f"[case] small decode {case}", flush=True)
    _run(ab, op_b, M, N, K, K + -K % 8, (K if op_b else N) + -(K if op_b else N) % 8,
         vk.KERNEL_DIRECT if direct else vk.KERNEL_SKINNY)


@pytest.mark.parametrize("ab,op_b,M,N,K,lda,ldb", [
    ("f16", 0, 3, 64, 64, 1 << 25, 64),         # the last token of each of three sequences of 8192 x 4096
    ("f32", 0, 3, 64, 64, 1 << 24, 64), ("f32", 0, 2, 64, 40, 40, 1 << 24),
    ("bf16", 1, 17, 64, 64, 1 << 25, 64)])
def test_rows_gigabytes_apart(ab, op_b, M, N, K, lda, ldb):
    """Leading dimensions past gemm_direct_kernel's 32-bit offsets: the decode kernels'."""
    import vkblas_amd as vk
    print(f"[case] small decode, far rows {ab} op_b={op_b} {M}x{N}x{K} lda={lda} ldb={ldb}", flush=True)
    _run(ab, op_b, M, N, K, lda, ldb, vk.KERNEL_SKINNY)
