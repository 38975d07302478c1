"""The many-token R-mode product (ane_amd/csrc/rmode_mul_mat.hip) through the
ggml hook, bit for bit against the oracle's GEMV per token: edges of the row
and token tiles, block counts that leave a part stage, weights at any even
offset, and inputs with infinities, denormals and zeros."""
import numpy as np
import pytest

from tests import data
from tests.test_qformats import assert_same, dev, host, weights_at

pytestmark = pytest.mark.gpu


def run_node(ane, q4, N, K, T, W, x):
    import torch

    y = torch.full((T, N), float("nan"), device="cuda")
    a = ane.ggml_tensor(ane.GgmlType.Q4_0 if q4 else ane.GgmlType.Q8_0, [K, N], W)
    b = ane.ggml_tensor(ane.GgmlType.F32, [K, T], x)
    d = ane.ggml_tensor(ane.GgmlType.F32, [N, T], y, op=ane.GgmlOp.MUL_MAT, src=(a, b))
    be = ane.GgmlBackend(q8_mode=1)  # R arithmetic for Q8_0
    be.compute(d)
    out = host(y)
    be.close()
    return out


def want(oracle, q4, N, K, W, x):
    f = (lambda v: oracle.q_gemv("q4_0", N, K, v, W)) if q4 else (lambda v: oracle.q8_0_gemv(N, K, v, W))
    return np.stack([f(v) for v in x])


# (N, K, T): each tile shape of the dispatch (by rows and tokens), its edges,
# and K of 1 to 5 blocks over the 4-block stages
SHAPES = [(16, 32, 2), (1, 64, 3), (17, 128, 16), (33, 160, 17), (100, 416, 31), (300, 512, 33), (4096, 128, 64),
          (8200, 96, 65), (2050, 256, 130), (9000, 160, 33), (16400, 64, 70),
          # two and three tokens on aligned rows ((N + T) % 8 == 0), both sides of
          # the rule that leaves them to the GEMVs (256 CUs)
          (4094, 256, 2), (4110, 1280, 2), (4109, 1280, 3), (8206, 256, 2), (8206, 1280, 2), (33005, 256, 3)]


@pytest.mark.parametrize("q4", [True, False])
@pytest.mark.parametrize("N,K,T", SHAPES)
def test_tokens_match_the_gemv(ane, oracle, q4, N, K, T):
    W = data.q_weights("q4_0", N, K, seed=N + T) if q4 else data.q8_0_weights(N, K, seed=N + T)
    x = data.activations(T, K, seed=K + T)
    off = (N + T) % 8 * 2  # weights at any even offset of their 16-byte granule
    keep, Wd = weights_at(W, off)
    assert_same(run_node(ane, q4, N, K, T, Wd, dev(x)), want(oracle, q4, N, K, W, x))


@pytest.mark.parametrize("q4", [True, False])
def test_special_values(ane, oracle, q4):
    N, K, T = 40, 224, 21
    W = (data.q_weights("q4_0", N, K, seed=3) if q4 else data.q8_0_weights(N, K, seed=3)).reshape(N, K // 32, -1)
    W = W.copy()
    for r, bits in ((1, 0x7C00), (2, 0x0001), (3, 0x8000), (4, 0xFC00), (5, 0x7E00)):  # inf, denormal, -0, -inf, NaN
        W[r, 2, :2] = np.array([bits], np.uint16).view(np.uint8)
    x = data.activations(T, K, seed=5)
    x[2, 70] = np.inf
    x[3, 5] = -np.inf
    x[4] = 0.0
    x[5] *= np.float32(1e-38)
    x[6, ::3] = -0.0
    x[20, 33] = np.nan
    W = W.reshape(N, -1)
    keep, Wd = weights_at(W, 6)
    assert_same(run_node(ane, q4, N, K, T, Wd, dev(x)), want(oracle, q4, N, K, W, x))


def test_odd_weights_address_takes_the_gemv(ane, oracle):
    """Q4_0 rows at an odd address keep the per-token GEMV."""
    N, K, T = 24, 64, 3
    W = data.q_weights("q4_0", N, K, seed=8)
    x = data.activations(T, K, seed=9)
    keep, Wd = weights_at(W, 7)
    assert_same(run_node(ane, True, N, K, T, Wd, dev(x)), want(oracle, True, N, K, W, x))


@pytest.mark.parametrize("q4", [True, False])
@pytest.mark.parametrize("K,T", [(64, 3), (256, 40)])
def test_outputs_over_earlier_inputs(ane, oracle, q4, K, T):
    """y one row before x in one buffer: token t's outputs replace token
    t-1's inputs, and each token still sees its own (one GEMV per token)."""
    import torch

    W = data.q_weights("q4_0", K, K, seed=K) if q4 else data.q8_0_weights(K, K, seed=K)
    x = data.activations(T, K, seed=T)
    keep, Wd = weights_at(W, 0)
    buf = torch.zeros((T + 1, K), device="cuda")
    buf[1:].copy_(dev(x))
    a = ane.ggml_tensor(ane.GgmlType.Q4_0 if q4 else ane.GgmlType.Q8_0, [K, K], Wd)
    b = ane.ggml_tensor(ane.GgmlType.F32, [K, T], buf[1:])
    d = ane.ggml_tensor(ane.GgmlType.F32, [K, T], buf[:T], op=ane.GgmlOp.MUL_MAT, src=(a, b))
    be = ane.GgmlBackend(q8_mode=1)
    be.compute(d)
    got = host(buf)[:T]
    be.close()
    assert_same(got, want(oracle, q4, K, K, W, x))
