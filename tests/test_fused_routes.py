"""dense_fused_i8 on the 64 x 64 contraction tiles (gemm_i8_tile64.hip) and on the
two-pass quantizer's unaligned rows (quantize_fused.hip), bit for bit against the
oracle: tile edges, an odd number of 64-byte K halves, rows of any length, and
the capture rule after calls that took the two-pass route."""
import numpy as np
import pytest

from tests import data
from tests.test_qformats import assert_same, dev, host

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("M,N,K", [(129, 1300, 100), (192, 1344, 129), (300, 700, 333), (257, 2003, 450),
                                   (130, 4100, 65), (513, 641, 1155), (200, 1999, 1)])
@pytest.mark.parametrize("offset", [0, 1])
def test_tiles_and_rows(ane, oracle, M, N, K, offset):
    import torch

    A, B = data.gemm_inputs(M, N, K, seed=M + N + K)
    want = oracle.dense_fused_i8(M, N, K, F32(0.5), bool(M % 2), A, B)
    a, b = (torch.zeros(v.size + 8, device="cuda") for v in (A, B))
    a[offset:offset + A.size].copy_(dev(A.ravel()))
    b[offset:offset + B.size].copy_(dev(B.ravel()))
    C = torch.full((M * N + 4,), 7.0, device="cuda")
    ane.dense_fused_i8(M, N, K, 0.5, bool(M % 2), a[offset:], b[offset:], C)
    got = host(C)
    assert_same(got[:M * N].reshape(M, N), want)
    assert (got[M * N:] == 7.0).all()


def test_capture_follows_the_last_eager_stream(ane, oracle):
    """256 x 2048 x 2048 is captured with its grid-wide wait on the stream of the
    last uncaptured call only, whichever route that call took; elsewhere the
    captured call takes the two-pass route.  Both replay to the same bits."""
    import torch

    M, N, K = 256, 2048, 2048
    A, B = data.gemm_inputs(M, N, K, seed=31)
    want = oracle.dense_fused_i8(M, N, K, F32(1.0), True, A, B)
    dA, dB, C = dev(A), dev(B), torch.zeros(M * N, device="cuda")
    ws = torch.empty(ane.dense_fused_i8_workspace_size(M, N, K), dtype=torch.uint8, device="cuda")
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    ane.dense_fused_i8(M, N, K, 1.0, True, dA, dB, C, workspace=ws, stream=s1)
    assert_same(host(C).reshape(M, N), want)
    for s, waits in ((s2, False), (s1, True)):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            ane.dense_fused_i8(M, N, K, 1.0, True, dA, dB, C, workspace=ws, stream=s, check_wait=False)
        for _ in range(3):
            C.fill_(float("nan"))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            ane.dense_fused_i8_status(ws, stream=s)
            assert_same(host(C).reshape(M, N), want)
            # the wait record counts the workgroups that met (0: two-pass)
            count = int(host(ws[256 + 8192:256 + 8196]).view(np.uint32)[0])
            assert (count > 0) == waits
        del g


def test_capture_after_a_wait_on_another_stream(ane, oracle):
    """A kernel with a grid-wide wait ran on s1 (16 x 4096 x 4096, taken eagerly
    too); an uncaptured 256 x 2048 x 2048 on s2, which takes the two-pass route,
    makes s2 the stream to capture on: the captured call keeps its wait."""
    import torch

    M, N, K = 256, 2048, 2048
    A, B = data.gemm_inputs(M, N, K, seed=37)
    want = oracle.dense_fused_i8(M, N, K, F32(1.0), True, A, B)
    dA, dB, C = dev(A), dev(B), torch.zeros(M * N, device="cuda")
    ws = torch.empty(ane.dense_fused_i8_workspace_size(M, N, K), dtype=torch.uint8, device="cuda")
    x, w, y = (torch.randn(n, device="cuda") for n in (16 * 4096, 4096 * 4096, 16 * 4096))
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    ane.dense_fused_i8(16, 4096, 4096, 1.0, True, x, w, y, stream=s1)
    ane.dense_fused_i8(M, N, K, 1.0, True, dA, dB, C, workspace=ws, stream=s2)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s2):
        ane.dense_fused_i8(M, N, K, 1.0, True, dA, dB, C, workspace=ws, stream=s2, check_wait=False)
    for _ in range(3):
        C.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        ane.dense_fused_i8_status(ws, stream=s2)
        assert_same(host(C).reshape(M, N), want)
        assert int(host(ws[256 + 8192:256 + 8196]).view(np.uint32)[0]) > 0


def test_two_pass_calls_do_not_wait_for_each_other(ane, oracle):
    """With no grid-wide wait in flight, a two-pass call on one stream does not
    run behind what another stream had queued before its own two-pass call."""
    import torch

    M, N, K = 256, 2048, 2048
    A, B = data.gemm_inputs(M, N, K, seed=41)
    want = oracle.dense_fused_i8(M, N, K, F32(1.0), True, A, B)
    dA, dB, C = dev(A), dev(B), [torch.zeros(M * N, device="cuda") for _ in range(2)]
    ws = [torch.empty(ane.dense_fused_i8_workspace_size(M, N, K), dtype=torch.uint8, device="cuda") for _ in range(2)]
    x, y = torch.randn(8192, 8192, device="cuda"), torch.empty(8192, 8192, device="cuda")
    busy, others = torch.cuda.Stream(), [torch.cuda.Stream() for _ in range(4)]

    def call(i, s):
        ane.dense_fused_i8(M, N, K, 1.0, True, dA, dB, C[i], workspace=ws[i], stream=s, check_wait=False)

    def backlog():  # a few hundred milliseconds on `busy`
        with torch.cuda.stream(busy):
            for _ in range(30):
                torch.mm(x, x, out=y)
        return busy.record_event()

    def independent(s):  # not on busy's hardware queue
        end = backlog()
        with torch.cuda.stream(s):
            C[1].zero_()
        s.record_event().synchronize()
        free = not end.query()
        torch.cuda.synchronize()
        return free

    for s in [busy] + others:
        call(0, s)
    backlog()
    torch.cuda.synchronize()
    s = next(s for s in others if independent(s))
    call(1, others[0] if s is not others[0] else others[1])
    torch.cuda.synchronize()
    end = backlog()
    call(0, busy)
    call(1, s)
    s.record_event().synchronize()
    assert not end.query()
    torch.cuda.synchronize()
    for c in C:
        assert_same(host(c).reshape(M, N), want)
