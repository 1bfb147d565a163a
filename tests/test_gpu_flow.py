"""gemm_flow_kernel (16-bit, 128x128 and 128x64 tiles) at the edges of its
tiles and forms: K of one step, one short of and one past it in 16-byte chunks,
past its stages; M and N one past and one short of a tile where the layout takes
them; the form for few, for one wave of and for many tiles; NaN in the padding of
every operand, C without any alignment, beta with C in place or apart, a bias;
against the CPU oracle.  C's padding must come back untouched.  Split-K pass 1 with a
ragged last slice, and the calls that add to C instead of the pipelined kernel."""
import numpy as np
import pytest
import torch

import oracle
from gpu_helpers import (BACK, BF16_BOUND, CONV, ENGINE, F16_BOUND, f32_bound, normwise, patterns,
                         to_dev_as as _dev)

pytestmark = pytest.mark.gpu

# M, N, K, batch (an MN-major operand's M or N is rounded up to a multiple of 8,
# K to one of 8 unless both are MN-major):
SHAPES = [(257, 63, 65, 40), (129, 127, 191, 40),      # 128 x 64 tiles: N of one, few of 128 x 128
          (641, 1153, 328, 4),                         # 128 x 128, three stages, eight waves (240 tiles)
          (1301, 703, 40, 1), (1601, 1537, 64, 1),     # three stages, one step: 128 x 64, eight waves
          (129, 129, 57, 96),                          # one stage (384 tiles, a single partial step)
          (257, 255, 72, 72), (130, 257, 200, 50)]     # two stages


@pytest.mark.parametrize("form", ["plain", "apart", "in_place"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("op_a,op_b", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("ab,ct", [("f16", "f16"), ("f16", "f32"), ("bf16", "bf16"), ("bf16", "f32")])
def test_flow(ab, ct, op_a, op_b, shape, form):
    import vkblas_amd as vk
    M, N, K, batch = shape
    M, N = (-(-M // 8) * 8 if op_a else M), (N if op_b else -(-N // 8) * 8)
    K = K if op_a and not op_b else -(-K // 8) * 8
    print(f"[case] flow {ab}>{ct} op={op_a}{op_b} {M}x{N}x{K} x{batch} {form}", flush=True)
    r = np.random.default_rng(M + 3 * N + 7 * K + batch)
    ra, ca = (K, M) if op_a else (M, K)
    rb, cb = (N, K) if op_b else (K, N)
    lda, ldb, ldc = -(-ca // 8) * 8 + 8, -(-cb // 8) * 8 + 8, N + 1 - N % 2 + 2
    # strides short of the last row's padding: the next matrix starts in it
    sa, sb, sc = lda * ra, ldb * rb, ldc * M + 5

    def operand(rows, cols, ld, stride):
        x = np.full(stride * batch, np.nan, np.float32)
        for i in range(batch):
            x[i * stride:][:ld * rows].reshape(rows, ld)[:, :cols] = r.uniform(-1, 1, (rows, cols))
        return x
    a, b = CONV[ab](operand(ra, ca, lda, sa)), CONV[ab](operand(rb, cb, ldb, sb))
    c0 = CONV[ct](r.uniform(-1, 1, 1 + sc * batch).astype(np.float32))
    cin = CONV[ct](r.uniform(-1, 1, 1 + sc * batch).astype(np.float32))
    bias = CONV[ab](r.uniform(-1, 1, N).astype(np.float32))
    alpha, beta = 1.25, 0.0 if form == "plain" else -0.5
    if form == "plain":                  # beta == 0 never reads C
        for i in range(batch):
            c0[1 + i * sc:][:ldc * M].reshape(M, ldc)[:, :N] = CONV[ct](np.full(1, np.nan, np.float32))[0]
    picked = sorted({0, batch // 2, batch - 1})
    rows = np.unique(np.array([0, 1, 63, 64, 127, 128, M // 2, M - 2, M - 1], np.int32))
    rows = rows[rows < M].astype(np.int32)
    want = c0.copy()
    for i in picked:
        src = (cin if form == "apart" else want)[1 + i * sc:][:ldc * M].copy()
        out = want[1 + i * sc:][:ldc * M].copy()
        oracle.ref_gemm_epi_rm(ab, ct, op_a, op_b, M, N, K, np.ascontiguousarray(a[i * sa:][:lda * ra]), lda,
                               np.ascontiguousarray(b[i * sb:][:ldb * rb]), ldb, alpha, beta, src, ldc, out, ldc,
                               BACK[ab](bias), rows=rows)
        want[1 + i * sc:][:ldc * M] = out
    dt = ENGINE
    dA, dB, dC, dI, dBias = _dev(a, ab), _dev(b, ab), _dev(c0, ct), _dev(cin, ct), _dev(bias, ab)
    ec = dC.element_size()
    vk.gemm_ex_async(dt[ab], dt[ct], op_a, op_b, M, N, K, alpha, dA.data_ptr(), lda, dB.data_ptr(), ldb,
                     beta, dC.data_ptr() + ec, ldc, batch=batch, stride_a=sa, stride_b=sb, stride_c=sc,
                     c_in=dI.data_ptr() + ec if form == "apart" else None, ldc_in=ldc if form == "apart" else 0,
                     stride_c_in=sc if form == "apart" else 0, bias=dBias.data_ptr(), bias_type=dt[ab])
    torch.cuda.synchronize()
    assert vk.last_kernel() == vk.KERNEL_FLOW, vk.last_kernel()
    got = patterns(dC)
    first = c0.view(np.uint8).reshape(-1)
    for i in range(batch):
        g = got[1 + i * sc:][:ldc * M].reshape(M, ldc)
        w = want[1 + i * sc:][:ldc * M].reshape(M, ldc)
        assert np.array_equal(g[:, N:], w[:, N:]), "C padding written"
        assert np.all(np.isfinite(BACK[ct](np.ascontiguousarray(g[:, :N]).reshape(-1)))), i
        if i in picked:
            gb = BACK[ct](np.ascontiguousarray(g[rows, :N]).reshape(-1))
            wb = BACK[ct](np.ascontiguousarray(w[rows, :N]).reshape(-1))
            assert normwise(gb, wb) <= (BF16_BOUND if ct == "bf16" else F16_BOUND), i
    # the element in front of C
    assert np.array_equal(got.view(np.uint8).reshape(-1)[:ec], first[:ec])


@pytest.mark.parametrize("form", ["plain", "in_place"])
@pytest.mark.parametrize("M,N,K,split", [(520, 520, 600, 3), (1032, 264, 2056, 4)])
@pytest.mark.parametrize("op_a,op_b", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("ab,ct", [("f16", "f16"), ("bf16", "f32")])
def test_flow_split(ab, ct, op_a, op_b, M, N, K, split, form):
    """pass 1 of a caller's split: slices that start past k 0, the last one shorter"""
    import vkblas_amd as vk
    print(f"[case] flow split {ab}>{ct} op={op_a}{op_b} {M}x{N}x{K}/{split} {form}", flush=True)
    _adds(vk, ab, ct, op_a, op_b, M, N, K, 0.0 if form == "plain" else -0.5, split, vk.PATH_SPLITK, vk.KERNEL_FLOW)


@pytest.mark.parametrize("M,N,K,beta,kernel", [
    (1024, 1024, 512, -0.5, "FLOW"), (256, 4096, 1024, 1.0, "FLOW"), (200, 8192, 128, 1.0, "FLOW"),
    (1024, 1024, 512, 0.0, "PIPE128_4"), (256, 4096, 1152, 1.0, "PIPE128_4")])
@pytest.mark.parametrize("ab,ct", [("f16", "f16"), ("bf16", "f32")])
@pytest.mark.parametrize("op_a,op_b", [(0, 1), (1, 0)])
def test_adds_to_c(op_a, op_b, ab, ct, M, N, K, beta, kernel):
    """one wave of 128 x 128 tiles: this kernel where beta adds to C in place after at most
    1024 k, else the pipelined one"""
    import vkblas_amd as vk
    print(f"[case] adds {ab}>{ct} op={op_a}{op_b} {M}x{N}x{K} beta={beta}", flush=True)
    _adds(vk, ab, ct, op_a, op_b, M, N, K, beta, 0, vk.PATH_TILE128, getattr(vk, "KERNEL_" + kernel))


def _adds(vk, ab, ct, op_a, op_b, M, N, K, beta, split, path, kernel):
    r = np.random.default_rng(M + 3 * N + 7 * K)
    lda, ldb = (M if op_a else K), (K if op_b else N)
    a, b, c = (CONV[t](r.uniform(-1, 1, n).astype(np.float32)) for t, n in ((ab, M * K), (ab, N * K), (ct, M * N)))
    rows = oracle.sample_rows(M, 16)
    want = c.copy()
    oracle.ref_gemm_epi_rm(ab, ct, op_a, op_b, M, N, K, a, lda, b, ldb, 1.25, beta, c, N, want, N, None, rows=rows)
    dA, dB, dC = _dev(a, ab), _dev(b, ab), _dev(c, ct)
    vk.gemm_async(ENGINE[ab], ENGINE[ct], op_a, op_b, M, N, K, 1.25, dA.data_ptr(), lda, dB.data_ptr(), ldb, beta,
                  dC.data_ptr(), N, split_k=split)
    assert (vk.last_path(), vk.last_kernel()) == (path, kernel), (vk.last_path(), vk.last_kernel())
    got = BACK[ct](patterns(dC)).reshape(M, N)
    assert np.all(np.isfinite(got))
    assert normwise(got[rows], BACK[ct](want).reshape(M, N)[rows]) <= (BF16_BOUND if ct == "bf16" else F16_BOUND)


@pytest.mark.parametrize("beta,M,N,K", [(0.0, 1304, 704, 200), (1.0, 1024, 1024, 512)])
def test_keeps_negative_zero(beta, M, N, K):
    """no bias adds nothing, not even 0.0 to -0.0: -1 times a zero product, plus a C of -0.0"""
    import vkblas_amd as vk
    print(f"[case] flow -0.0 beta={beta}", flush=True)
    a = torch.zeros(M, K, dtype=torch.float16, device="cuda:0")
    b = torch.ones(N, K, dtype=torch.float16, device="cuda:0")
    c = torch.full((M, N), -0.0, dtype=torch.float16, device="cuda:0")
    vk.gemm_async(vk.DT_F16, vk.DT_F16, 0, 1, M, N, K, -1.0, a.data_ptr(), K, b.data_ptr(), K, beta, c.data_ptr(), N)
    torch.cuda.synchronize()
    assert vk.last_kernel() == vk.KERNEL_FLOW, vk.last_kernel()
    assert bool((c == 0).all()) and bool(torch.signbit(c).all())
