"""cblas_igemm's operand pre-pass and fused epilogue (ane_amd/csrc/igemm.hip), bit
for bit against the oracle: edges of the 128-row x 128-k tiles, row and column sums
as partials and (where they do not fit or are more than 16, or beta is not zero)
as cleared sums, the epilogue of every contraction kernel, and operands at odd
addresses."""
import numpy as np
import pytest

from tests.test_convert_kernels import at_offset
from tests.test_gpu_parity import IGEMM_VARIANT, _igemm_case
from tests.test_qformats import assert_same, dev, host

pytestmark = pytest.mark.gpu
F32 = np.float32


# few-row kernel and 64-tiles; (1, 40, 1024): more partials than the workspace has
# room for; 16 and 17 k-tiles on both
@pytest.mark.parametrize("kind", ["igemm", "ugemm", "usgemm"])
@pytest.mark.parametrize("flags", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,K", [(63, 65, 320), (65, 63, 256), (1, 40, 1024), (129, 257, 576), (130, 1300, 64),
                                   (400, 900, 1100), (70, 200, 2048), (70, 200, 2112), (257, 600, 2048),
                                   (257, 600, 2112)])
def test_tiles_and_sums(ane, oracle, kind, flags, M, N, K):
    for beta, sem in ((0.0, 0), (0.25, 0), (0.0, 1), (-0.5, 1)):
        lda = K + 1 if not flags & 1 else M + 3
        ldb = N + 5 if not flags & 2 else K + 9
        if flags & 1 and sem == 0:
            lda = max(lda, K)
        A, B, C = _igemm_case(kind, flags, M, N, K, lda, ldb, N + 1, seed=M + N + K + flags)
        if flags & 1 and sem == 1:
            A = np.resize(A, K * lda)
        want = oracle.cblas_igemm(IGEMM_VARIANT[kind], flags, M, N, K, lda, ldb, N + 1, -1.5, beta, A, B, C,
                                  semantics=sem)
        Cd = dev(C)
        ka, pa = at_offset(A, 1)
        kb, pb = at_offset(B, 3)
        ane.cblas_igemm(kind, flags, M, N, K, lda, ldb, N + 1, -1.5, beta, pa, pb, Cd, blas=bool(sem))
        assert_same(host(Cd), want)


# with 256 CUs: 128-tiles on a 3-stage ring (192), 128-tiles (289), 256-tiles (256),
# and the general kernel (few columns, more few-row workgroups than CUs)
@pytest.mark.parametrize("kind", ["igemm", "ugemm", "usgemm"])
@pytest.mark.parametrize("pad", [1, 4])
@pytest.mark.parametrize("M,N,K", [(1500, 2000, 320), (2100, 2100, 192), (4081, 4092, 128), (4100, 100, 192)])
def test_epilogue_of_the_large_tiles(ane, oracle, kind, M, N, K, pad):
    """beta = 0, so the contraction writes C: 16-byte stores (ldc % 4 == 0) or single ones."""
    A, B, C = _igemm_case(kind, 2, M, N, K, K + 3, K + 5, N + pad, seed=M + N + K)
    oracle.set_threads(0)
    try:
        want = oracle.cblas_igemm(IGEMM_VARIANT[kind], 2, M, N, K, K + 3, K + 5, N + pad, 0.75, 0.0, A, B, C)
    finally:
        oracle.set_threads(1)
    Cd = dev(C)
    ane.cblas_igemm(kind, 2, M, N, K, K + 3, K + 5, N + pad, 0.75, 0.0, dev(A), dev(B), Cd)
    assert_same(host(Cd), want)


@pytest.mark.parametrize("which,flags", [("A", 0), ("A", 1), ("B", 2), ("B", 0)])
@pytest.mark.parametrize("M,N,K,at", [(300, 700, 512, 0), (300, 700, 512, 160000), (40, 64, 128, 48), (500, 900, 320, 16)])
def test_c_over_an_operand(ane, oracle, which, flags, M, N, K, at):
    """igemm with beta = 0 whose C covers A or B (from byte `at` of C on): the
    operand is read whole before C is written, also where it could be read in
    place (A without transA, B with transB)."""
    import torch

    lda, ldb, ldc = (K if not flags & 1 else M + 16), (N if not flags & 2 else K + 16), N + 4
    if flags & 1:
        lda = -(-max(lda, K) // 16) * 16
    A, B, C = _igemm_case("igemm", flags, M, N, K, lda, ldb, ldc, seed=M + N + K + flags)
    for sem in (0, 1):
        if flags & 1 and sem == 1:
            A = np.resize(A, K * lda)
        want = oracle.cblas_igemm(0, flags, M, N, K, lda, ldb, ldc, 0.5, 0.0, A, B, np.zeros_like(C), semantics=sem)
        over = A if which == "A" else B
        buf = torch.zeros(max(M * ldc * 4, at + over.size), dtype=torch.uint8, device="cuda")
        buf[at:at + over.size] = dev(over.view(np.uint8))
        a = buf.data_ptr() + at if which == "A" else dev(A)
        b = buf.data_ptr() + at if which == "B" else dev(B)
        ane.cblas_igemm("igemm", flags, M, N, K, lda, ldb, ldc, 0.5, 0.0, a, b, buf, blas=bool(sem))
        got = host(buf)[:M * ldc * 4].view(F32).reshape(M, ldc)
        assert_same(got[:, :N], np.asarray(want).reshape(M, ldc)[:, :N])
