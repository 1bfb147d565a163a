"""The generic kernel's branch-free edge loads: M and N below one 16-byte vector, one
past and one short of a tile, K of one, one short of and one past a K step, odd
leading dimensions with NaN in the padding, operands one element off any alignment,
every layout, type pair and tile; against the CPU oracle.  C's padding must come back
untouched."""
import numpy as np
import pytest
import torch

import oracle
from gpu_helpers import (BACK, BF16_BOUND, CONV, ENGINE, F16_BOUND, f32_bound, normwise, patterns,
                         to_dev_as as _dev)

pytestmark = pytest.mark.gpu

# tile override (0: 64 x 64, 1: 128 x 128, 2: 256 x 256), M, N, K, split
SHAPES = [(0, 3, 5, 1, 1), (0, 65, 63, 31, 1), (0, 9, 129, 65, 1), (1, 129, 127, 63, 1), (1, 2, 131, 33, 1),
          (1, 250, 7, 100, 1), (2, 257, 255, 67, 1),
          (0, 5, 3, 300, 1), (1, 131, 2, 129, 1), (0, 70, 6, 7, 1),       # fewer than a vector along M, N, K
          # slices of whole K steps, the last one shorter than a vector (fp16 64 + 64 + 5, fp32 4 x 32 + 5)
          (0, 65, 63, 133, 5), (1, 129, 3, 133, 5)]


@pytest.fixture(autouse=True)
def reset_override():
    import vkblas_amd as vk
    yield
    vk.set_override(-1, False)


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("op_a,op_b", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("ab,ct", [("f32", "f32"), ("f16", "f16"), ("f16", "f32"), ("bf16", "bf16"), ("bf16", "f32")])
def test_generic_edges(ab, ct, op_a, op_b, shape):
    import vkblas_amd as vk
    tile, M, N, K, split = shape
    print(f"[case] generic {ab}>{ct} op={op_a}{op_b} {shape}", flush=True)
    r = np.random.default_rng(M + 3 * N + 7 * K)
    ra, ca = (K, M) if op_a else (M, K)
    rb, cb = (N, K) if op_b else (K, N)
    lda, ldb, ldc = ca + 1 - ca % 2 + 2, cb + 1 - cb % 2 + 4, N + 1 - N % 2 + 2

    def operand(rows, cols, ld):
        x = np.full(1 + ld * rows, np.nan, np.float32)
        x[1:].reshape(rows, ld)[:, :cols] = r.uniform(-1, 1, (rows, cols))
        return CONV[ab](x)
    a, b = operand(ra, ca, lda), operand(rb, cb, ldb)
    c = CONV[ct](r.uniform(-1, 1, 1 + M * ldc).astype(np.float32))
    want = c[1:].copy()
    oracle.ref_gemm_epi_rm(ab, ct, op_a, op_b, M, N, K, a[1:].copy(), lda, b[1:].copy(), ldb, 1.25, -0.5, want.copy(),
                           ldc, want, ldc, None)
    dt = ENGINE
    dA, dB, dC = _dev(a, ab), _dev(b, ab), _dev(c, ct)
    vk.set_override(tile, True)
    vk.gemm_async(dt[ab], dt[ct], op_a, op_b, M, N, K, 1.25, dA.data_ptr() + dA.element_size(), lda,
                  dB.data_ptr() + dB.element_size(), ldb, -0.5, dC.data_ptr() + dC.element_size(), ldc, split_k=split)
    torch.cuda.synchronize()
    assert vk.last_kernel() == vk.KERNEL_GENERIC_CHECKED, vk.last_kernel()
    got = patterns(dC)
    assert np.array_equal(got[:1], c[:1]), "the element in front of C written"
    g, w = (BACK[ct](np.ascontiguousarray(x)).reshape(M, ldc) for x in (got[1:], want))
    assert np.array_equal(g[:, N:], w[:, N:]), "C padding written"
    assert np.all(np.isfinite(g[:, :N]))
    bound = BF16_BOUND if ct == "bf16" else f32_bound(K) if ab == "f32" else F16_BOUND
    assert normwise(g[:, :N], w[:, :N]) <= bound
