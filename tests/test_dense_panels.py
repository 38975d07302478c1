"""dense_i8 / dense_u8s8 on the panel kernels (gemm_i8_panel256.hip,
gemm_i8_panel128.hip, gemm_i8_skinny.hip), bit for bit against the oracle:
tile edges, odd numbers of 64-byte K slices, part panels, and A's extreme
values with columns whose sums are large."""
import numpy as np
import pytest

from tests.test_gpu_parity import _dense_inputs
from tests.test_qformats import assert_same, dev, host

pytestmark = pytest.mark.gpu
F32 = np.float32

# up to 128 rows: one workgroup per panel (1, 2, 4 and 8 row blocks); above,
# 128-tiles, and 256-tiles once they give every CU one
SHAPES = [(1, 10, 64), (17, 33, 100), (50, 128, 784), (64, 16, 320), (113, 200, 1000), (128, 257, 192),
          (129, 16, 64), (144, 130, 128), (300, 250, 456), (513, 384, 832), (4081, 4090, 192)]


@pytest.mark.parametrize("unsigned_a", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_dense_shapes(ane, oracle, M, N, K, unsigned_a):
    import torch

    A, B, bias, Mp, Kp = _dense_inputs(M, N, K, M + N + K, unsigned_a)
    if N > 20:
        B[:, 3], B[:, 17] = 127, -128
    A[0] = 255 if unsigned_a else -128
    Bp = oracle.pack_b(B, Kp, N)
    want = oracle.dense_i8(M, N, K, F32(0.01), F32(0.02), 1 if M % 2 else 0, A, Bp, bias, unsigned_a=unsigned_a)
    C = torch.full((Mp * N + 8,), 7.0, device="cuda")
    ane.dense_i8(M, N, K, 0.01, 0.02, M % 2 == 1, dev(A), dev(Bp), dev(bias), C, unsigned_a=unsigned_a)
    got = host(C)
    assert_same(got[:Mp * N], np.asarray(want, F32).reshape(-1)[:Mp * N])
    assert (got[Mp * N:] == 7.0).all()


@pytest.mark.parametrize("unsigned_a", [False, True])
def test_panels_past_32_bit_offsets(ane, oracle, unsigned_a):
    """B just over 2 GiB: the general kernel (gemm_i8.hip), which keeps 64-bit
    offsets.  Three stretches of panels against the oracle; the last crosses the
    2 GiB line."""
    import torch

    M, K, P = 16, 4096, 32769  # panels of 64 KiB
    N = 16 * P
    g = torch.Generator(device="cuda").manual_seed(5)
    Bp = torch.empty((P, 16 * K), dtype=torch.int8, device="cuda")
    for p in range(0, P, 4096):
        n = min(4096, P - p)
        Bp[p:p + n] = torch.randint(-128, 128, (n, 16 * K), generator=g, dtype=torch.int8, device="cuda")
    A, _, _, _, _ = _dense_inputs(M, 16, K, 7, unsigned_a)
    A[0] = 255 if unsigned_a else -128
    bias = torch.randn(N, generator=g, device="cuda")
    C = torch.full((M * N + 8,), 7.0, device="cuda")
    ane.dense_i8(M, N, K, 0.01, 0.02, False, dev(A), Bp, bias, C, unsigned_a=unsigned_a)
    assert (host(C[M * N:]) == 7.0).all()
    C = C[:M * N].view(M, N)
    for p0, n in ((0, 3), (16383, 4), (P - 5, 5)):
        cols = slice(16 * p0, 16 * (p0 + n))
        want = oracle.dense_i8(M, 16 * n, K, F32(0.01), F32(0.02), 0, A, host(Bp[p0:p0 + n]).ravel(), host(bias[cols]),
                               unsigned_a=unsigned_a)
        assert_same(host(C[:, cols].contiguous()), np.asarray(want, F32).reshape(M, 16 * n))
    del Bp, C
    torch.cuda.empty_cache()
