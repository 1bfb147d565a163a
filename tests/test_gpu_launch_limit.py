"""A launch holds less than 2^32 threads: past that HIP runs a few workgroups and reports
success.  Such calls run on a kernel that needs fewer, or are refused."""
import numpy as np
import pytest
import torch

import oracle
from gpu_helpers import f32_bound, normwise, to_dev

pytestmark = pytest.mark.gpu


def _equal_products(M, N, K, batch):
    """batch products of the same two operands, fp32 NN; the result matrices and the oracle's"""
    import vkblas_amd as vk
    print(f"[case] {batch} matrices of {M}x{N}x{K}", flush=True)
    r = np.random.default_rng(1)
    a, b = (r.uniform(-1, 1, n).astype(np.float32) for n in (M * K, K * N))
    want = np.zeros(M * N, np.float32)
    oracle.ref_gemm_f32_rm(0, 0, M, N, K, a, K, b, N, 1.0, 0.0, want, N)
    dA, dB = to_dev(a), to_dev(b)
    dC = torch.empty(batch, M * N, device="cuda:0")
    vk.gemm_async(vk.DT_F32, vk.DT_F32, 0, 0, M, N, K, 1.0, dA.data_ptr(), K, dB.data_ptr(), N, 0.0, dC.data_ptr(), N,
                  batch=batch, stride_a=0, stride_b=0, stride_c=M * N)
    torch.cuda.synchronize()
    return dC, want


def test_more_matrices_than_small_tiles():
    """2^22 + 1 matrices of 33 x 33: 4 tiles of 32 x 32 each are too many, one of 64 x 64 is not"""
    import vkblas_amd as vk
    dC, want = _equal_products(33, 33, 128, (1 << 22) + 1)
    assert vk.last_kernel() == vk.KERNEL_GENERIC_CHECKED, vk.last_kernel()
    assert normwise(dC[0].cpu().numpy(), want) <= f32_bound(128)
    assert torch.equal(dC, dC[:1].expand_as(dC))


@pytest.mark.parametrize("extra", [0, 1])
def test_more_matrices_than_any_tile(extra):
    import vkblas_amd as vk
    with pytest.raises(vk.VkblasError):
        _equal_products(8, 8, 8, (1 << 24) + extra)


def test_more_weight_rows_than_the_gemv():
    """one token against 2^26 + 64 weight rows of 8: not the GEMV kernel's 64 threads per row"""
    import vkblas_amd as vk
    N, K = (1 << 26) + 64, 8
    print(f"[case] 1x{N}x{K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randint(-4, 5, (1, K), device="cuda", generator=g).half()
    w = torch.randint(-4, 5, (N, K), device="cuda", generator=g).half()
    y = torch.full((1, N), float("nan"), device="cuda", dtype=torch.float16)
    vk.gemm_async(vk.DT_F16, vk.DT_F16, 0, 1, 1, N, K, 1.0, x.data_ptr(), K, w.data_ptr(), K, 0.0, y.data_ptr(), N)
    torch.cuda.synchronize()
    assert vk.last_path() != vk.PATH_SKINNY
    # small whole numbers: exact in fp16 and fp32
    assert torch.equal(y[0], (w.float() * x.float()).sum(1).half())
