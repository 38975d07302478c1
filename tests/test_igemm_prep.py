"""cblas_igemm's operand pre-pass and fused epilogue (ane_amd/csrc/igemm.hip), bit
for bit against the oracle: edges of the 64-row x 256-k tiles, row and column sums
as partials and (where they do not fit, or beta is not zero) as cleared sums, the
epilogue of every contraction kernel, and operands at odd addresses."""
import numpy as np
import pytest

from tests.test_convert_kernels import at_offset
from tests.test_gpu_parity import IGEMM_VARIANT, _igemm_case
from tests.test_qformats import assert_same, dev, host

pytestmark = pytest.mark.gpu
F32 = np.float32


# few-row kernel, 64/128-row contraction tiles, 128-tiles on a part of the CUs;
# (1, 40, 1024): more partials than the workspace has room for
@pytest.mark.parametrize("kind", ["igemm", "ugemm", "usgemm"])
@pytest.mark.parametrize("flags", [0, 1, 2, 3])
@pytest.mark.parametrize("M,N,K", [(63, 65, 320), (65, 63, 256), (1, 40, 1024), (129, 257, 576), (130, 1300, 64),
                                   (400, 900, 1100)])
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
