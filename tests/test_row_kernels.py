"""The ggml node kernels' short-row, flat and swept forms, bit for bit: the
softmax of many short rows (decode_ref.hip, k_softmax_short) at the edges of
its register sizes, the contiguous elementwise forms (ggml_backend.hip,
k_flat_ew / k_row_ew), SiLU's vectors and RoPE over several sweeps of rows."""
import numpy as np
import pytest

from tests.test_ggml_ops import host, rnd, same, softmax_oracle
from tests.test_ggml_ops import dev as _dev

pytestmark = pytest.mark.gpu
F32 = np.float32


_keep = []  # a node holds addresses only: its tensors live until the test ends


def dev(a):
    _keep.append(_dev(a))
    return _keep[-1]


@pytest.fixture(autouse=True)
def _release():
    yield
    _keep.clear()


def compute(ane, op, ne, out, src, params=(), nb=None):
    t = ane.GgmlType.F32
    be = ane.GgmlBackend()
    be.compute(ane.ggml_tensor(t, ne, out, op=getattr(ane.GgmlOp, op), src=src, nb=nb,
                               op_params=ane.ggml_op_params(*params)))
    import torch

    torch.cuda.synchronize()
    be.close()


# from four rows per CU (1024 on 256 CUs) the 16-lane rows; 8, 16, 32 and 64 registers
@pytest.mark.parametrize("n", [1, 15, 16, 17, 128, 129, 250, 257, 512, 520, 1024, 1025])
@pytest.mark.parametrize("masked", [False, True])
def test_softmax_short_rows(ane, oracle, n, masked):
    H, T = 3, 347  # 1041 rows: the last workgroup is partly filled
    X = rnd((H, T, n), n, 6.0)
    X[0, 1, :] = F32(-3e38)
    X[0, 2, n // 2] = F32(np.inf)
    M = np.zeros((T, n), F32)
    M[3, : n // 2] = -np.inf
    M[4, n // 3:] = F32(-2.5)
    scale = F32(0.0883)
    out = dev(np.full(X.shape, np.nan, F32))
    x = ane.ggml_tensor(ane.GgmlType.F32, [n, T, H], dev(X))
    m = ane.ggml_tensor(ane.GgmlType.F32, [n, T], dev(M)) if masked else None
    compute(ane, "SOFT_MAX", [n, T, H], out, (x, m), (float(scale), 0.0))
    pre = (X * scale).astype(F32)
    if masked:
        pre = pre + M
    rows = np.r_[0:6, T:T + 3, 2 * T + 300:3 * T]  # heads, specials and the last rows
    flat, got = pre.reshape(-1, n), host(out).reshape(-1, n)
    ok = [r for r in rows if not (np.isinf(flat[r]).any() and not np.isneginf(flat[r]).any()) and
          not np.isneginf(flat[r]).all()]
    same(got[ok], softmax_oracle(oracle, flat[ok]))
    # every row against the kernel that takes a few rows at a time
    few = dev(np.full((7, n), np.nan, F32))
    for r0 in (0, 500, 1034):
        sub = np.ascontiguousarray(X.reshape(-1, n)[r0:r0 + 7])
        xs = ane.ggml_tensor(ane.GgmlType.F32, [n, 7], dev(sub))
        ms = None
        if masked:
            ms = ane.ggml_tensor(ane.GgmlType.F32, [n, 7], dev(M[[r % T for r in range(r0, r0 + 7)]]))
        compute(ane, "SOFT_MAX", [n, 7], few, (xs, ms), (float(scale), 0.0))
        a, b = got[r0:r0 + 7], host(few)
        assert np.array_equal(np.isnan(a), np.isnan(b))
        same(np.nan_to_num(a), np.nan_to_num(b))


@pytest.mark.parametrize("op", ["ADD", "MUL"])
@pytest.mark.parametrize("shape,bshape", [((1, 3), (1, 3)), ((5, 7), (5, 7)), ((33, 2052), (33, 2052)),
                                          ((1, 4), (1, 4)), ((9, 4), (1, 4)), ((301, 1028), (1, 1028)),
                                          ((2, 6), (1, 6)), ((20000, 8), (1, 8))])
def test_elementwise_forms(ane, op, shape, bshape):
    A, B = rnd(shape, 1), rnd(bshape, 2)
    want = A + B if op == "ADD" else A * B
    t = ane.GgmlType.F32
    for off in (0, 1):  # 16-byte aligned, and one float past it (the row kernel)
        bufs = [dev(np.zeros(v.size + 8, F32)) for v in (A, B, A)]
        a, b, o = (buf[off:off + v.size] for buf, v in zip(bufs, (A, B, A)))
        a.copy_(dev(A.ravel()))
        b.copy_(dev(B.ravel()))
        at = ane.ggml_tensor(t, list(reversed(shape)), a)
        bt = ane.ggml_tensor(t, list(reversed(bshape)), b)
        compute(ane, op, list(reversed(shape)), o, (at, bt))
        same(host(o), want.ravel())
        assert not host(bufs[2])[off + A.size:].any()
        compute(ane, op, list(reversed(shape)), a, (at, bt))  # in place
        same(host(a), want.ravel())


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 4099])
def test_scale_and_silu_tails(ane, oracle, n):
    X = rnd((n,), n, 5.0)
    t = ane.GgmlType.F32
    for off in (0, 1):
        src, out = dev(np.zeros(n + 8, F32)), dev(np.zeros(n + 8, F32))
        src[off:off + n].copy_(dev(X))
        x = ane.ggml_tensor(t, [n], src[off:])
        compute(ane, "SCALE", [n], out[off:], (x,), (0.37, 0.0))
        same(host(out)[off:off + n], X * F32(0.37))
        compute(ane, "SILU", [n], out[off:], (x,))
        same(host(out)[off:off + n], oracle.silu_fp32(X))
        assert not host(out)[off + n:].any()


def test_silu_estimates(ane, oracle):
    """Every mantissa step of the reciprocal estimate (1 + e^-x over its 256
    table entries, several exponents) and the range's ends."""
    X = np.concatenate([np.linspace(-90, 90, 60001), np.linspace(-1, 1, 20001),
                        [0.0, -0.0, 1e-40, -1e-40, 3e38, -3e38, np.inf]]).astype(F32)
    out = dev(np.zeros(X.size, F32))
    compute(ane, "SILU", [X.size], out, (ane.ggml_tensor(ane.GgmlType.F32, [X.size], dev(X)),))
    got, want = host(out), oracle.silu_fp32(X)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    same(np.nan_to_num(got), np.nan_to_num(want))


@pytest.mark.parametrize("D,H,T", [(2, 1, 1), (6, 5, 1000), (100, 3, 67), (128, 9, 1000), (64, 41, 999)])
def test_rope_sweeps(ane, D, H, T):
    """More rows than one sweep (4096) included; each position against the
    one-position kernel."""
    import torch

    X, P = rnd((T, H, D), D), np.random.default_rng(T).integers(0, 3000, T).astype(np.int32)
    out = dev(np.zeros(X.shape, F32))
    x = ane.ggml_tensor(ane.GgmlType.F32, [D, H, T], dev(X))
    pos = ane.ggml_tensor(ane.GgmlType.I32, [T], dev(P))
    compute(ane, "ROPE", [D, H, T], out, (x, pos), (0, D, 0, 0, 0, 10000.0, 1.0, 0.0, 1.0, 0.0, 0.0))
    got = host(out)
    ref = torch.zeros((H, D), device="cuda")
    for t in {0, T // 3, T // 2, T - 2 if T > 1 else 0, T - 1}:
        ane.rope_fp32(H, D, int(P[t]), 10000.0, dev(X[t]), ref)
        same(got[t], host(ref))
