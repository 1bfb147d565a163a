"""The pipelined kernels' epilogue that adds beta's matrix: C in place, apart with
16-byte rows (read as row segments) and apart off that alignment (read through the
MFMA layout), with a bias, on whole and on shifted edge tiles of both tile sizes and
every result type; against the CPU oracle.  C's padding must come back untouched.
Batches with the scalars in device memory."""
import numpy as np
import pytest
import torch

import oracle
from gpu_helpers import (BACK, BF16_BOUND, CONV, ENGINE, F16_BOUND, f32_bound, normwise, patterns,
                         to_dev_as as _dev)

pytestmark = pytest.mark.gpu

# tile override (1: 128 x 128, 2: 256 x 256), M, N, K
SHAPES = [(2, 512, 256, 256), (2, 264, 520, 256), (1, 128, 256, 256), (1, 200, 264, 256)]


@pytest.fixture(autouse=True)
def reset_override():
    import vkblas_amd as vk
    yield
    vk.set_override(-1, False)


@pytest.mark.parametrize("form", ["in_place", "apart", "apart_unaligned"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("op_a,op_b", [(0, 1), (1, 0)])
@pytest.mark.parametrize("ab,ct", [("f32", "f32"), ("f16", "f16"), ("f16", "f32"), ("bf16", "bf16"), ("bf16", "f32")])
def test_add(ab, ct, op_a, op_b, shape, form):
    import vkblas_amd as vk
    tile, M, N, K = shape
    print(f"[case] pipe add {ab}>{ct} op={op_a}{op_b} {shape} {form}", flush=True)
    r = np.random.default_rng(M + 3 * N)
    lda, ldb, ldc = (M if op_a else K), (K if op_b else N), N + 8
    ldi = N + (12 if form == "apart_unaligned" else 16)
    u = lambda n: r.uniform(-1, 1, n).astype(np.float32)   # noqa: E731
    a, b = CONV[ab](u(M * K)), CONV[ab](u(N * K))
    c, cin = CONV[ct](u(M * ldc)), CONV[ct](u(M * ldi + 4))
    off = 4 if form == "apart_unaligned" and ct != "f32" else 1 if form == "apart_unaligned" else 0
    bias = CONV[ab](u(N))
    src, lds = (c.copy(), ldc) if form == "in_place" else (cin[off:off + M * ldi].copy(), ldi)
    want = c.copy()
    oracle.ref_gemm_epi_rm(ab, ct, op_a, op_b, M, N, K, a, lda, b, ldb, 1.25, -0.5, src, lds, want, ldc, BACK[ab](bias))
    dt = ENGINE
    dA, dB, dC, dI, dBias = _dev(a, ab), _dev(b, ab), _dev(c, ct), _dev(cin, ct), _dev(bias, ab)
    vk.set_override(tile, False)
    vk.gemm_ex_async(dt[ab], dt[ct], op_a, op_b, M, N, K, 1.25, dA.data_ptr(), lda, dB.data_ptr(), ldb, -0.5,
                     dC.data_ptr(), ldc, c_in=None if form == "in_place" else dI.data_ptr() + off * dI.element_size(),
                     ldc_in=0 if form == "in_place" else ldi, bias=dBias.data_ptr(), bias_type=dt[ab])
    torch.cuda.synchronize()
    if form != "apart_unaligned" or ct != "f32":   # fp32 off 16 bytes goes to the generic kernel
        assert vk.last_kernel() in (vk.KERNEL_PIPE256, vk.KERNEL_PIPE128, vk.KERNEL_PIPE128_4), vk.last_kernel()
    got = patterns(dC)
    g, w = (BACK[ct](x).reshape(M, ldc) for x in (got, want))
    assert np.array_equal(g[:, N:], w[:, N:]), "C padding written"
    bound = BF16_BOUND if ct == "bf16" else f32_bound(K) if ab == "f32" else F16_BOUND
    assert normwise(g[:, :N], w[:, :N]) <= bound


@pytest.mark.parametrize("form", ["in_place", "apart"])
@pytest.mark.parametrize("shape", [(2, 264, 520, 256), (1, 200, 264, 256)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("ab,ct", [("f32", "f32"), ("f16", "f16"), ("bf16", "f32")])
def test_add_batch_device_scalars(ab, ct, shape, form):
    import vkblas_amd as vk
    tile, M, N, K = shape
    batch = 3
    print(f"[case] pipe add batch {ab}>{ct} {shape} {form}", flush=True)
    r = np.random.default_rng(M + 5 * N)
    ldc, ldi = N + 8, N + 16
    sc, si = M * ldc + 16, M * ldi + 8
    u = lambda n: r.uniform(-1, 1, n).astype(np.float32)   # noqa: E731
    a, b = CONV[ab](u(batch * M * K)), CONV[ab](u(batch * N * K))
    c, cin = CONV[ct](u(batch * sc)), CONV[ct](u(batch * si))
    want = c.copy()
    for i in range(batch):
        src, lds = (want[i * sc:][:M * ldc].copy(), ldc) if form == "in_place" else (cin[i * si:][:M * ldi].copy(), ldi)
        out = want[i * sc:][:M * ldc].copy()
        oracle.ref_gemm_epi_rm(ab, ct, 0, 1, M, N, K, a[i * M * K:][:M * K].copy(), K, b[i * N * K:][:N * K].copy(), K,
                               1.25, -0.5, src, lds, out, ldc, None)
        want[i * sc:][:M * ldc] = out
    dA, dB, dC, dI = _dev(a, ab), _dev(b, ab), _dev(c, ct), _dev(cin, ct)
    scalars = torch.tensor([1.25, -0.5], device="cuda:0")
    vk.set_override(tile, False)
    vk.gemm_ex_async(ENGINE[ab], ENGINE[ct], 0, 1, M, N, K, 0.0, dA.data_ptr(), K, dB.data_ptr(), K, 0.0, dC.data_ptr(),
                     ldc, batch=batch, stride_a=M * K, stride_b=N * K, stride_c=sc, scalar_mode=vk.SCALAR_DEV_F32,
                     alpha_dev=scalars.data_ptr(), beta_dev=scalars.data_ptr() + 4,
                     c_in=dI.data_ptr() if form == "apart" else None, ldc_in=ldi if form == "apart" else 0,
                     stride_c_in=si if form == "apart" else 0)
    assert vk.last_kernel() in (vk.KERNEL_PIPE256, vk.KERNEL_PIPE128, vk.KERNEL_PIPE128_4), vk.last_kernel()
    got = patterns(dC)
    bound = BF16_BOUND if ct == "bf16" else f32_bound(K) if ab == "f32" else F16_BOUND
    for i in range(batch):
        g, w = (BACK[ct](x[i * sc:(i + 1) * sc].copy()) for x in (got, want))
        assert np.array_equal(g[M * ldc:], w[M * ldc:]), "between the matrices written"
        g, w = g[:M * ldc].reshape(M, ldc), w[:M * ldc].reshape(M, ldc)
        assert np.array_equal(g[:, N:], w[:, N:]), "C padding written"
        assert normwise(g[:, :N], w[:, :N]) <= bound, i


@pytest.mark.parametrize("tile,ct", [(2, "f16"), (2, "f32"), (1, "f16"), (1, "f32")])
def test_keeps_negative_zero(tile, ct):
    """no bias adds nothing, not even 0.0 to -0.0: -1 times a zero product, plus a C of -0.0"""
    import vkblas_amd as vk
    print(f"[case] pipe add -0.0 tile={tile} {ct}", flush=True)
    M, N, K = 512, 256, 256
    a = torch.zeros(M, K, dtype=torch.float16, device="cuda:0")
    b = torch.ones(N, K, dtype=torch.float16, device="cuda:0")
    c = torch.full((M, N), -0.0, dtype=torch.float16 if ct == "f16" else torch.float32, device="cuda:0")
    vk.set_override(tile, False)
    vk.gemm_async(vk.DT_F16, ENGINE[ct], 0, 1, M, N, K, -1.0, a.data_ptr(), K, b.data_ptr(), K, 1.0, c.data_ptr(), N)
    torch.cuda.synchronize()
    assert vk.last_kernel() in (vk.KERNEL_PIPE256, vk.KERNEL_PIPE128, vk.KERNEL_PIPE128_4), vk.last_kernel()
    assert bool((c == 0).all()) and bool(torch.signbit(c).all())


@pytest.mark.parametrize("K", [1024, 16512])
def test_add_large(K):
    """an fp32 C of 64 MiB that is stored to stay in the caches, and past them where the
    operands of the call drive it out (in all more than 320 MiB)"""
    import vkblas_amd as vk
    M = N = 4096
    print(f"[case] pipe add {M}x{N}x{K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.randn(K, 4096, device="cuda", generator=g).bfloat16() for _ in range(2))
    c = torch.randn(M, N, device="cuda", generator=g)
    rows = oracle.sample_rows(M, 8)
    want = c.cpu().numpy().reshape(-1)
    hc = want.copy()
    oracle.ref_gemm_epi_rm("bf16", "f32", 1, 0, M, N, K, patterns(a).reshape(-1), M, patterns(b).reshape(-1), N, 1.25, -0.5,
                           hc, N, want, N, None, rows=rows)
    vk.set_override(2, False)
    vk.gemm_async(vk.DT_BF16, vk.DT_F32, 1, 0, M, N, K, 1.25, a.data_ptr(), M, b.data_ptr(), N, -0.5, c.data_ptr(), N,
                  split_k=1)
    assert vk.last_kernel() == vk.KERNEL_PIPE256, vk.last_kernel()
    got = patterns(c)
    assert np.all(np.isfinite(got))
    assert normwise(got[rows], want.reshape(M, N)[rows]) <= F16_BOUND
