"""The panel packer and the per-row quantizer (ane_amd/csrc/quantize.hip) at
the edges of their work splits, bit for bit against the oracle: 64 x 256 tiles
and unaligned rows, one-wave and one-workgroup rows and their register limits."""
import numpy as np
import pytest

from tests.test_qformats import dev, host

pytestmark = pytest.mark.gpu
F32 = np.float32


def at_offset(a, nbytes):
    """a on the device starting nbytes past a 256-byte boundary."""
    import torch

    raw = np.ascontiguousarray(a).reshape(-1).view(np.uint8)
    buf = torch.zeros(raw.size + 256, dtype=torch.uint8, device="cuda")
    buf[nbytes:nbytes + raw.size] = torch.from_numpy(raw).cuda()
    return buf, buf.data_ptr() + nbytes


@pytest.mark.parametrize("offset", [0, 1, 8])
@pytest.mark.parametrize("K,N", [(64, 256), (63, 255), (65, 257), (1, 1), (4, 16), (130, 1000), (67, 31), (1000, 48)])
def test_pack_b_tiles(ane, oracle, K, N, offset):
    import torch

    B = np.random.default_rng(K * N).integers(-128, 128, size=(K, N), dtype=np.int8)
    ref = oracle.pack_b(B, K, N)
    keep, src = at_offset(B, offset)
    for dst_off in (0, 4):
        out = torch.full((ref.size + 64,), 77, dtype=torch.int8, device="cuda")
        ane.pack_b_i8(K, N, src, out.data_ptr() + dst_off)
        got = host(out)
        np.testing.assert_array_equal(got[dst_off:dst_off + ref.size], ref)
        assert (got[:dst_off] == 77).all() and (got[dst_off + ref.size:] == 77).all()


def test_pack_b_more_rows_than_a_launch(ane):
    """2^30 + 5 rows of one column: more 64-row tiles than one launch holds (1 GiB
    in, 16 GiB out, compared on the device)."""
    import torch

    K = (1 << 30) + 5
    src = torch.randint(-128, 128, (K,), dtype=torch.int8, device="cuda")
    out = torch.full((-(-K // 4) * 64,), 77, dtype=torch.int8, device="cuda")
    ane.pack_b_i8(K, 1, src, out)
    groups = out.view(torch.int32).view(-1, 16)  # a column's four rows per word
    col = groups[:, 0].contiguous().view(torch.int8)
    assert torch.equal(col[:K], src) and not col[K:].any()
    assert not groups[:, 1:].any()
    del src, out, groups, col
    torch.cuda.empty_cache()


# 1024 rows: one wave per row up to 2048 values; fewer rows or longer ones: a
# workgroup per row, held in registers up to 8192 values
@pytest.mark.parametrize("rows,cols", [(1024, 16), (1027, 100), (1025, 2048), (1024, 2064), (3, 8192), (2, 8200),
                                       (1, 1), (5, 1030), (1026, 272)])
@pytest.mark.parametrize("offset", [0, 4])
def test_channelwise_rows(ane, oracle, rows, cols, offset):
    import torch

    cpad = max(16, -(-cols // 16) * 16)
    x = np.random.default_rng(rows + cols).standard_normal((rows, cpad)).astype(F32)
    x[rows // 2] = 0.0
    if rows > 4:
        x[1, 3] = np.nan
        x[2, 5] = np.inf
        x[3] *= F32(1e-40)
    q_ref, s_ref = oracle.channelwise(x.reshape(-1), rows, cols)
    keep, src = at_offset(x, offset)
    q = torch.zeros(rows * cpad + 16, dtype=torch.int8, device="cuda")
    s = torch.zeros(rows, dtype=torch.float32, device="cuda")
    ane.check(ane.lib().ane_hip_quantize_channelwise(rows, cols, src, q.data_ptr() + offset, s.data_ptr(), 0))
    np.testing.assert_array_equal(host(q)[offset:offset + rows * cpad], np.asarray(q_ref).reshape(-1))
    np.testing.assert_array_equal(host(s).view(np.uint32)[~np.isnan(s_ref)], s_ref.view(np.uint32)[~np.isnan(s_ref)])
    assert np.array_equal(np.isnan(host(s)), np.isnan(s_ref))
