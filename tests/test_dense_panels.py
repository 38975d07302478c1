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
