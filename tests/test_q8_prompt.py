"""The prompt form of the G-mode product (ane_amd/csrc/q8_0_prompt.hip), bit for
bit against the oracle: edges of the 64-row and 32/64-token tiles, block counts
that leave a part stage or fewer than a stage, rows at any even alignment, and
scales that are infinite, denormal, negative or NaN."""
import numpy as np
import pytest

from tests import data
from tests.test_qformats import assert_same, dev, host, weights_at

pytestmark = pytest.mark.gpu


def run(ane, N, K, T, W, x, offset=0):
    import torch

    keep, Wd = weights_at(W, offset)
    y = torch.full((T * N + 8,), 7.0, device="cuda")
    ane.q8_0_mul_mat(N, K, T, dev(x), Wd, y)
    got = host(y)
    assert (got[T * N:] == 7.0).all()
    return got[:T * N].reshape(T, N)


# K: whole stages of 512, part stages, under one stage, odd block counts
# (rows that are only 2-byte aligned); N and T around the tile edges.  Aligned
# rows (offset 0) with several stages: 136 blocks (the last stage half full) and
# 64 blocks on 195 workgroups; the other whole-stage shapes are too few
# workgroups for this kernel at offset 0
@pytest.mark.parametrize("N,K,T", [(64, 512, 64), (65, 1024, 65), (63, 544, 33), (1, 32, 70), (130, 480, 100),
                                   (200, 4128, 31), (64, 96, 5), (300, 2080, 129), (1000, 11008, 17), (7, 160, 200),
                                   (200, 4352, 100), (100, 4352, 20), (4100, 2048, 130)])
@pytest.mark.parametrize("offset", [0, 6])
def test_shapes(ane, oracle, N, K, T, offset):
    W = data.q8_0_weights(N, K, seed=N + K)
    x = data.activations(T, K, seed=T)
    assert_same(run(ane, N, K, T, W, x, offset), oracle.q8_0_mul_mat_g(N, K, T, x, W))


@pytest.mark.parametrize("K", [544, 1024, 4352])
def test_special_scales(ane, oracle, K):
    N, T = 70, 72
    W = data.q8_0_weights(N, K, seed=3).reshape(N, K // 32, 34).copy()
    for r, bits in ((1, 0x7C00), (2, 0x0001), (3, 0x8000), (4, 0xFC00), (5, 0x7E00), (6, 0xB123)):
        W[r, -1, :2] = np.array([bits], np.uint16).view(np.uint8)
    x = data.activations(T, K, seed=5)
    x[2, 40] = np.inf
    x[3, K - 1] = np.nan
    x[4] = 0.0
    x[5] *= np.float32(1e-38)
    x[71, :32] = -np.inf
    W = W.reshape(N, -1)
    assert_same(run(ane, N, K, T, W, x), oracle.q8_0_mul_mat_g(N, K, T, x, W))
