"""The work a user of ane_amd has it do, as timed cases.

Each case is one pass through the public entry points: the opcode records of
``stream_exec``, the kernel-level wrappers, a ggml backend node (or a short
run of them), or one decoded token.  ``listed`` names twelve of them,
``draw`` gives more of the same ranges, and ``exact`` restates each in 64
bits with plain torch.

Kinds and what they stand for:

mlp       the reference's MNIST program: two dense_fused_i8 records in one
          dispatch stream, a batch of images through both layers.
fused     one dense_fused_i8 layer on fp32 operands (quantize, contract,
          dequantize), workspace kept by the caller.
dense     the quantize-once pattern: dense_i8 / dense_u8s8 on an int8
          activation batch and weights packed beforehand.
convert   turning fp32 weights and activations into the int8 forms: per-tensor
          quantize, panel packing, per-row quantize, dequantize.
igemm     the strided integer GEMMs, signed, unsigned and mixed, transposed or
          not, with row strides that need not be aligned.
q8, q4    a ggml MUL_MAT node on Q8_0 / Q4_0 weights: one token (decode), a
          few (a batch of sequences) or a prompt (prefill).
kquant    a matrix-vector product in one of the other weight formats.
rows      the fp32 nodes around the products over a prompt: norm, weight,
          RoPE, masked softmax, SiLU, product, residual add.
token     one decoded token of a Llama-shaped model: embedding row, layers,
          final norm, output head.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import ane_amd
from ane_amd import GgmlOp, GgmlType

DEV = "cuda:0"
QVALS = {"q4_k": 256, "q2_k": 256, "q3_k": 256, "q5_k": 256, "q6_k": 256, "q4_0": 32}
FP16_AT = {"q4_k": (0, 2), "q2_k": (80, 82), "q3_k": (108,), "q5_k": (0, 2), "q6_k": (208,), "q4_0": (0,)}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: the MNIST layers of the reference's test program
        {"name": "mlp_mnist", "kind": "mlp", "batch": 50, "n_in": 784, "n_hidden": 128, "n_out": 10},
        # the headline benchmark
        {"name": "fused_4096", "kind": "fused", "M": 4096, "N": 4096, "K": 4096, "relu": True},
        # a layer whose sizes are multiples of nothing
        {"name": "fused_ragged", "kind": "fused", "M": 301, "N": 2003, "K": 1777, "relu": False},
        # a hidden layer over a large batch, weights packed once
        {"name": "dense_batch", "kind": "dense", "M": 2048, "N": 4096, "K": 4096, "unsigned": False, "relu": True},
        # preparing one layer's weights and a batch of its activations
        {"name": "convert_layer", "kind": "convert", "K": 4096, "N": 6144, "rows": 1024},
        # uint8 activations times int8 weights, both row-major
        {"name": "igemm_mixed", "kind": "igemm", "variant": "usgemm", "ta": False, "tb": False, "blas": False,
         "M": 1536, "N": 2048, "K": 2048, "pad": 0},
        # one token through a feed-forward projection
        {"name": "q8_token", "kind": "q8", "N": 4096, "K": 11008, "T": 1},
        # a prompt through a feed-forward projection
        {"name": "q8_prompt", "kind": "q8", "N": 14336, "K": 4096, "T": 512},
        # the same path with 4-bit weights
        {"name": "q4_prompt", "kind": "q4", "N": 4096, "K": 4096, "T": 128},
        # a K-quant matrix-vector product
        {"name": "q6k_token", "kind": "kquant", "fmt": "q6_k", "N": 14336, "K": 4096},
        # the steps around the products over a prompt
        {"name": "rows_prompt", "kind": "rows", "T": 512, "heads": 16, "ffn": 8192},
        # one token of a model: the latency a chat user sees
        {"name": "token_4layers", "kind": "token", "layers": 4, "kv_heads": 8, "ffn": 14336, "ctx": 4096,
         "pos": 3000, "vocab": 32768},
    ]


def draw(rng):
    def size(lo, hi, step=1):
        """Log-uniform in [lo, hi]; a multiple of step."""
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        return max(lo, min(hi, int(round(v / step)) * step))

    def ragged(lo, hi, step):
        """As size; a multiple of step half the time, any number otherwise."""
        return size(lo, hi, step if rng.random() < 0.5 else 1)

    kind = rng.choice(["mlp", "fused", "dense", "convert", "igemm", "q8", "q8", "q4", "kquant", "rows", "token"])
    c = {"kind": kind}
    if kind == "mlp":
        c.update(batch=size(1, 512), n_in=size(32, 1024), n_hidden=size(8, 512), n_out=size(2, 200))
    elif kind == "fused":
        c.update(M=ragged(1, 4096, 16), N=ragged(16, 4096, 64), K=ragged(32, 4096, 128), relu=rng.random() < 0.5)
    elif kind == "dense":
        c.update(M=ragged(1, 2048, 16), N=ragged(10, 4096, 64), K=ragged(32, 4096, 64),
                 unsigned=rng.random() < 0.4, relu=rng.random() < 0.5)
    elif kind == "convert":
        c.update(K=ragged(16, 4096, 64), N=ragged(10, 6144, 64), rows=size(1, 1024))
    elif kind == "igemm":
        c.update(variant=rng.choice(["igemm", "ugemm", "usgemm"]), ta=rng.random() < 0.25, tb=rng.random() < 0.5,
                 blas=rng.random() < 0.5, M=ragged(1, 1536, 16), N=ragged(8, 2048, 64), K=ragged(64, 2048, 64),
                 pad=rng.choice([0, 0, 16, 5]))
    elif kind in ("q8", "q4"):
        tmax = 512 if kind == "q8" else 128
        cap = (14336 * 4096 * 512) if kind == "q8" else (4096 * 4096 * 128)
        while True:
            c.update(N=ragged(64, 14336, 256), K=size(256, 14336, rng.choice([32, 256, 256, 512])),
                     T=rng.choice([1, size(2, 16), size(2, tmax), size(16, tmax)]))
            c["K"] = max(256, c["K"] // 32 * 32)
            if c["N"] * c["K"] * c["T"] <= cap:
                break
    elif kind == "kquant":
        c.update(fmt=rng.choice(sorted(QVALS)), N=ragged(64, 14336, 256), K=size(256, 4096, 256))
    elif kind == "rows":
        while True:
            c.update(T=size(1, 512), heads=rng.choice([1, 2, 3, 5, 8, 12, 16]), ffn=size(128, 8192, 32))
            if c["T"] * c["ffn"] >= 128:
                break
    else:
        ctx = size(64, 4096, 64)
        c.update(layers=rng.randint(1, 4), kv_heads=rng.choice([2, 4, 8]), ffn=size(256, 14336, 256), ctx=ctx,
                 pos=rng.randrange(ctx), vocab=size(256, 32768, 32))
    return c


# ----------------------------------------------------------------- the inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(0x5EED + 7919 * int(seed))
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)


def _q8_rows(g, n, k):
    """n rows of Q8_0 blocks quantized from N(0, 0.02) weights (uint8 bytes)."""
    out = torch.empty((n, k // 32, 34), dtype=torch.uint8, device=DEV)
    for r in range(0, n, 4096):  # bounded temporaries
        w = (_randn(g, min(4096, n - r), k // 32, 32) * 0.02)
        d = (w.abs().amax(dim=2) / 127.0).to(torch.float16)
        q = torch.clamp(torch.round(w / d.float().unsqueeze(2)), -127, 127).to(torch.int8)
        out[r:r + 4096, :, :2] = d.view(torch.uint8).view(-1, k // 32, 2)
        out[r:r + 4096, :, 2:] = q.view(torch.uint8)
    return out.view(n, -1)


def _q_rows(g, fmt, n, k):
    """n rows of a format's blocks: random quants and scales, fp16 super-scales |N(0, 0.01)|."""
    nbytes, nvals = ane_amd.QFORMATS[fmt]
    w = torch.randint(0, 256, (n, k // nvals, nbytes), generator=g, device=DEV, dtype=torch.uint8)
    for at in FP16_AT[fmt]:
        d = (_randn(g, n, k // nvals).abs() * 0.01).to(torch.float16)
        w[:, :, at:at + 2] = d.view(torch.uint8).view(n, -1, 2)
    return w.view(n, -1)


def _ceil(x, m):
    return (x + m - 1) // m * m


def _rows_inputs(case, g):
    T, H, F = case["T"], case["heads"], case["ffn"]
    D = 128
    return {
        "x": _randn(g, T, H * D), "w": 1.0 + 0.1 * _randn(g, H * D), "s": _randn(g, H, T, T) * 8.0,
        "mask": torch.triu(torch.full((T, T), float("-inf"), device=DEV), diagonal=1).contiguous(),
        "pos": torch.arange(T, dtype=torch.int32, device=DEV), "gate": _randn(g, T, F) * 2.0, "up": _randn(g, T, F),
    }


def _token_inputs(case, g):
    H, L = case["kv_heads"] * 4 * 128, case["layers"]
    kvd, ffn, ctx = case["kv_heads"] * 128, case["ffn"], case["ctx"]
    layers = []
    for _ in range(L):
        layers.append({
            "w_qkv": _q8_rows(g, H + 2 * kvd, H), "w_o": _q8_rows(g, H, H), "w_gate_up": _q8_rows(g, 2 * ffn, H),
            "w_down": _q8_rows(g, H, ffn), "attn_norm": 1.0 + 0.1 * _randn(g, H), "ffn_norm": 1.0 + 0.1 * _randn(g, H),
            "k": (_randn(g, case["kv_heads"], ctx, 128)).to(torch.float16),
            "v": (_randn(g, case["kv_heads"], ctx, 128)).to(torch.float16)})
    return {"layers": layers, "embed": _q8_rows(g, case["vocab"], H), "norm": 1.0 + 0.1 * _randn(g, H),
            "token": torch.randint(0, case["vocab"], (1,), generator=g, device=DEV, dtype=torch.int32),
            "rope": torch.from_numpy(ane_amd.rope_table(ctx)).to(DEV)}


def _inputs(case, seed):
    """The tensors a pass starts from, the same for run and exact."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "mlp":
        # pixels in [0, 1], four in five of them zero
        x = torch.rand((case["batch"], case["n_in"]), generator=g, device=DEV)
        x[torch.rand(x.shape, generator=g, device=DEV) < 0.8] = 0.0
        return {"x": x, "w1": 0.05 * _randn(g, case["n_in"], case["n_hidden"]),
                "w2": 0.05 * _randn(g, case["n_hidden"], case["n_out"])}
    if kind == "fused":
        return {"A": _randn(g, case["M"], case["K"]), "B": _randn(g, case["K"], case["N"])}
    if kind == "dense":
        M, N, K = case["M"], case["N"], case["K"]
        Mp, Kp = max(16, _ceil(M, 16)), _ceil(K, 64)
        A = torch.zeros((Mp, Kp), dtype=torch.uint8 if case["unsigned"] else torch.int8, device=DEV)
        a = _randn(g, M, K) * 30.0
        A[:M, :K] = (a.abs() if case["unsigned"] else a).round().clamp(-127, 127).to(A.dtype)
        B = torch.zeros((Kp, N), dtype=torch.int8, device=DEV)
        B[:K] = (_randn(g, K, N) * 30.0).round().clamp(-127, 127).to(torch.int8)
        return {"A": A, "B": B, "bias": _randn(g, N)}
    if kind == "convert":
        K, N, R = case["K"], case["N"], case["rows"]
        pad = max(16, _ceil(K, 16))
        x = torch.zeros((R, pad), device=DEV)
        x[:, :K] = _randn(g, R, K) * torch.exp(_randn(g, R, 1))  # rows of different scales
        w = torch.zeros(max(16, _ceil(K * N, 16)), device=DEV)
        w[:K * N] = (0.05 * _randn(g, K * N))
        return {"w": w, "x": x}
    if kind == "igemm":
        M, N, K, p = case["M"], case["N"], case["K"], case["pad"]
        # the handler's transA reads rows i%16 at offsets up to M, so it gets 16 rows of K + M bytes
        if case["ta"] and not case["blas"]:
            ash = (16, K + M + 16 + p)
        else:
            ash = (K, M + p) if case["ta"] else (M, K + p)
        bsh = (N, K + p) if case["tb"] else (K, N + p)
        A = torch.randint(0, 256, ash, generator=g, device=DEV, dtype=torch.uint8)
        B = torch.randint(0, 256, bsh, generator=g, device=DEV, dtype=torch.uint8)
        return {"A": A, "B": B}
    if kind == "q8":
        return {"W": _q8_rows(g, case["N"], case["K"]), "x": _randn(g, case["T"], case["K"])}
    if kind == "q4":
        return {"W": _q_rows(g, "q4_0", case["N"], case["K"]), "x": _randn(g, case["T"], case["K"])}
    if kind == "kquant":
        return {"W": _q_rows(g, case["fmt"], case["N"], case["K"]), "x": _randn(g, case["K"])}
    if kind == "rows":
        return _rows_inputs(case, g)
    return _token_inputs(case, g)


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    kind = case["kind"]
    f32 = dict(dtype=torch.float32, device=DEV)
    u8 = dict(dtype=torch.uint8, device=DEV)
    if kind == "mlp":
        s["h"] = torch.empty((case["batch"], case["n_hidden"]), **f32)
        s["y"] = torch.empty((case["batch"], case["n_out"]), **f32)
    elif kind == "fused":
        s["C"] = torch.empty((case["M"], case["N"]), **f32)
        s["ws"] = torch.empty(ane_amd.dense_fused_i8_workspace_size(case["M"], case["N"], case["K"]), **u8)
    elif kind == "dense":
        Kp, N = s["B"].shape
        s["Bp"] = torch.empty(ane_amd.packed_b_size(Kp, N), dtype=torch.int8, device=DEV)
        ane_amd.pack_b_i8(Kp, N, s["B"], s["Bp"])
        s["C"] = torch.empty((s["A"].shape[0], N), **f32)
        del s["B"]
    elif kind == "convert":
        K, N, R = case["K"], case["N"], case["rows"]
        s.update(qw=torch.empty(s["w"].numel(), dtype=torch.int8, device=DEV), sw=torch.empty(1, **f32),
                 Bp=torch.empty(ane_amd.packed_b_size(K, N), dtype=torch.int8, device=DEV),
                 qx=torch.empty(s["x"].shape, dtype=torch.int8, device=DEV), sx=torch.empty(R, **f32),
                 back=torch.empty(s["w"].numel(), **f32),
                 ws=torch.empty(ane_amd.lib().ane_hip_quantize_workspace_size(s["w"].numel()), **u8))
    elif kind == "igemm":
        s["C"] = torch.empty((case["M"], case["N"]), **f32)
        wsb = ane_amd.lib().ane_hip_cblas_igemm_workspace_size(case["M"], case["N"], case["K"])
        s["ws"] = torch.empty(wsb, **u8)
    elif kind in ("q8", "q4"):
        s["y"] = torch.empty((case["T"], case["N"]), **f32)
        s["be"] = ane_amd.GgmlBackend()
        wt = GgmlType.Q8_0 if kind == "q8" else GgmlType.Q4_0
        a = ane_amd.ggml_tensor(wt, [case["K"], case["N"]], s["W"])
        b = ane_amd.ggml_tensor(GgmlType.F32, [case["K"], case["T"]], s["x"])
        s["node"] = ane_amd.ggml_tensor(GgmlType.F32, [case["N"], case["T"]], s["y"], op=GgmlOp.MUL_MAT, src=(a, b))
    elif kind == "kquant":
        s["y"] = torch.empty(case["N"], **f32)
    elif kind == "rows":
        _rows_nodes(s)
    else:
        _token_state(s)
    return s


def _rows_nodes(s):
    """A prompt's nodes: q = rope(norm(x) * w), p = softmax(s / sqrt(128) + mask),
    h = silu(gate) * up, r = x + q."""
    case, F, O = s["case"], GgmlType.F32, GgmlOp
    T, H, ffn = case["T"], case["heads"], case["ffn"]
    D = H * 128
    t, par = ane_amd.ggml_tensor, ane_amd.ggml_op_params
    for name, shape in (("n", (T, D)), ("nw", (T, D)), ("q", (T, D)), ("p", (H, T, T)), ("g", (T, ffn)),
                        ("h", (T, ffn)), ("r", (T, D))):
        s[name] = torch.empty(shape, dtype=torch.float32, device=DEV)
    x, w = t(F, [D, T], s["x"]), t(F, [D], s["w"])
    n = t(F, [D, T], s["n"], op=O.RMS_NORM, src=(x,), op_params=par(1e-5))
    nw = t(F, [D, T], s["nw"], op=O.MUL, src=(n, w))
    nw3, pos = t(F, [128, H, T], s["nw"]), t(GgmlType.I32, [T], s["pos"])
    q = t(F, [128, H, T], s["q"], op=O.ROPE, src=(nw3, pos),
          op_params=par(0, 128, 0, 0, 0, 10000.0, 1.0, 0.0, 1.0, 0.0, 0.0))
    sc, mk = t(F, [T, T, H], s["s"]), t(F, [T, T], s["mask"])
    p = t(F, [T, T, H], s["p"], op=O.SOFT_MAX, src=(sc, mk), op_params=par(1.0 / math.sqrt(128.0), 0.0))
    ga, up = t(F, [ffn, T], s["gate"]), t(F, [ffn, T], s["up"])
    g = t(F, [ffn, T], s["g"], op=O.SILU, src=(ga,))
    h = t(F, [ffn, T], s["h"], op=O.MUL, src=(g, up))
    q2 = t(F, [D, T], s["q"])
    r = t(F, [D, T], s["r"], op=O.ADD, src=(x, q2))
    s["nodes"] = [n, nw, q, p, g, h, r]
    s["be"] = ane_amd.GgmlBackend()


def _token_state(s):
    case = s["case"]
    H = case["kv_heads"] * 4 * 128
    cfg = ane_amd.DecodeConfig(case["layers"], H, case["ffn"], case["kv_heads"] * 4, case["kv_heads"], 128,
                               case["ctx"], 1e-5)
    arr = (ane_amd.DecodeLayer * case["layers"])()
    for i, l in enumerate(s["layers"]):
        arr[i] = ane_amd.DecodeLayer(*[l[n].data_ptr() for n in ("w_qkv", "w_o", "w_gate_up", "w_down", "attn_norm",
                                                                  "ffn_norm", "k", "v")])
    s.update(cfg=cfg, arr=arr, x=torch.empty(H, dtype=torch.float32, device=DEV),
             xn=torch.empty(H, dtype=torch.float32, device=DEV),
             logits=torch.empty(case["vocab"], dtype=torch.float32, device=DEV),
             dws=ane_amd.decode_workspace(cfg, DEV),
             hws=torch.empty(ane_amd.q8_0_mul_mat_workspace_size(H, 1, case["vocab"]), dtype=torch.uint8, device=DEV))


# ------------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "mlp":
        b, i, h, o = case["batch"], case["n_in"], case["n_hidden"], case["n_out"]
        ane_amd.stream_exec([ane_amd.rec_dense_fused_i8(b, h, i, 1.0, True, s["x"], s["w1"], s["h"]),
                             ane_amd.rec_dense_fused_i8(b, o, h, 1.0, False, s["h"], s["w2"], s["y"])])
        return {"hidden": s["h"], "out": s["y"]}
    if kind == "fused":
        ane_amd.dense_fused_i8(case["M"], case["N"], case["K"], 1.0, case["relu"], s["A"], s["B"], s["C"],
                               workspace=s["ws"], check_wait=False)
        return s["C"]
    if kind == "dense":
        ane_amd.dense_i8(case["M"], case["N"], case["K"], 0.011, 0.0037, case["relu"], s["A"], s["Bp"], s["bias"],
                         s["C"], unsigned_a=case["unsigned"])
        return s["C"]
    if kind == "convert":
        K, N, R = case["K"], case["N"], case["rows"]
        L, st = ane_amd.lib(), torch.cuda.current_stream().cuda_stream
        ane_amd.quantize_fp32_i8(s["w"], s["qw"], s["sw"], count=K * N, workspace=s["ws"])
        ane_amd.pack_b_i8(K, N, s["qw"], s["Bp"])
        ane_amd.check(L.ane_hip_quantize_channelwise(R, K, s["x"].data_ptr(), s["qx"].data_ptr(),
                                                     s["sx"].data_ptr(), st))
        ane_amd.check(L.ane_hip_dequantize_i8_fp32(K * N, 0.0021, s["qw"].data_ptr(), s["back"].data_ptr(), st))
        return {"qw": s["qw"], "sw": s["sw"], "Bp": s["Bp"], "qx": s["qx"], "sx": s["sx"], "back": s["back"]}
    if kind == "igemm":
        flags = (1 if case["ta"] else 0) | (2 if case["tb"] else 0)
        ane_amd.cblas_igemm(case["variant"], flags, case["M"], case["N"], case["K"], s["A"].shape[1],
                            s["B"].shape[1], case["N"], 0.0123, 0.0, s["A"], s["B"], s["C"], blas=case["blas"],
                            workspace=s["ws"])
        return s["C"]
    if kind in ("q8", "q4"):
        s["be"].set_stream(None)
        s["be"].compute(s["node"])
        return s["y"]
    if kind == "kquant":
        ane_amd.q_gemv(case["fmt"], case["N"], case["K"], s["x"], s["W"], s["y"])
        return s["y"]
    if kind == "rows":
        s["be"].set_stream(None)
        for node in s["nodes"]:
            s["be"].compute(node)
        return {k: s[k] for k in ("n", "nw", "q", "p", "g", "h", "r")}
    H = s["x"].numel()
    ane_amd.get_rows("q8_0", 1, H, s["embed"], case["vocab"], s["token"], s["x"])
    ane_amd.decode_token(s["cfg"], s["arr"], s["rope"], case["pos"], s["x"], s["dws"])
    ane_amd.rms_norm(H, s["x"], s["norm"], 1e-5, s["xn"])
    ane_amd.q8_0_mul_mat(case["vocab"], H, 1, s["xn"], s["embed"], s["logits"], workspace=s["hws"])
    return {"hidden": s["x"], "logits": s["logits"], "k": [l["k"] for l in s["layers"]],
            "v": [l["v"] for l in s["layers"]]}


# ------------------------------------------------------- what a pass is worth
def work(case):
    kind = case["kind"]
    if kind == "mlp":
        b, i, h, o = case["batch"], case["n_in"], case["n_hidden"], case["n_out"]
        return {"bytes": 4 * (b * i + i * h + b * h + h * o + b * o), "flops": 2 * b * h * (i + o)}
    if kind in ("fused", "dense", "igemm"):
        M, N, K = case["M"], case["N"], case["K"]
        e = 4 if kind == "fused" else 1
        return {"bytes": e * (M * K + K * N) + 4 * M * N, "flops": 2 * M * N * K}
    if kind == "convert":
        K, N, R = case["K"], case["N"], case["rows"]
        # quantize, pack, per-row quantize, dequantize: the fp32 weights and the
        # int8 form once each, then the results
        return {"bytes": K * N * (4 + 1 + 1 + 4) + R * K * 5, "flops": 2 * (2 * K * N + R * K)}
    if kind in ("q8", "q4", "kquant"):
        N, K, T = case["N"], case["K"], case.get("T", 1)
        nbytes, vals = (34, 32) if kind == "q8" else ane_amd.QFORMATS["q4_0" if kind == "q4" else case["fmt"]]
        return {"bytes": N * (K // vals) * nbytes + 4 * T * (K + N), "flops": 2 * N * K * T}
    if kind == "rows":
        T, H, F = case["T"], case["heads"], case["ffn"]
        D = H * 128
        # norm, weight, RoPE, add: x read, four results; softmax: scores, mask, result; SiLU and product
        n = 5 * T * D + D + 2 * H * T * T + T * T + 4 * T * F
        return {"bytes": 4 * n, "flops": 12 * T * D + 12 * H * T * T + 12 * T * F}
    H, kvd = case["kv_heads"] * 512, case["kv_heads"] * 128
    weights = case["layers"] * (H * (H + 2 * kvd) + H * H + 3 * H * case["ffn"]) + case["vocab"] * H
    kv = case["layers"] * 2 * case["kv_heads"] * (case["pos"] + 1) * 128
    return {"bytes": weights * 34 // 32 + 2 * kv + 4 * (2 * H + case["vocab"]), "flops": 2 * weights + 8 * kv}


def tolerance(case):
    if case["kind"] == "token":
        # expf and the rounding of activations to int8 between layers: a value
        # that falls on the other side of a rounding step moves its block by one
        # quantum and travels through every later product
        return {"rel": 2e-2}
    # Integer sums are exact in any order, and the fp32 operations around them
    # have one defined order each: the results are pinned bit for bit.
    return "exact"


# ------------------------------------------------------------- 64-bit results
def _quant(x, amax):
    """The int8 form of x for a given max |x| (fp32 arithmetic, as defined) and its scale."""
    a = torch.where(amax == 0, torch.full_like(amax, 127.0), amax).double()
    scale, inv = (a / 127.0).float(), (127.0 / a).float()  # one rounding each: 53 bits hold the quotients' 24
    inv = torch.where(amax == 0, torch.full_like(inv, 127.0), inv)
    return torch.clamp(x * inv, -127.0, 127.0).round(), scale


def _fused64(A, B, relu):
    qa, sa = _quant(A, A.abs().amax())
    qb, sb = _quant(B, B.abs().amax())
    c = (qa.double() @ qb.double()) * (sa.double() * sb.double())
    return c.clamp(min=0.0) if relu else c


def _q8_values(W, n, k):
    b = W.view(n, k // 32, 34)
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    return (b[:, :, 2:].contiguous().view(torch.int8).double() * d).view(n, k)


def _q8_act(x):
    """x rounded to int8 per 32-value block, as values."""
    b = x.float().reshape(-1, 32)
    q, s = _quant(b, b.abs().amax(dim=1, keepdim=True))
    return (q.double() * s.double()).view(x.shape)


def _nib(b):
    return (b & 15), (b >> 4)


def _scale_min6(s):
    """The eight 6-bit (scale, min) pairs of 12 packed bytes (last axis)."""
    sc, mn = [], []
    for j in range(8):
        if j < 4:
            sc.append(s[..., j] & 63)
            mn.append(s[..., j + 4] & 63)
        else:
            sc.append((s[..., j + 4] & 15) | ((s[..., j - 4] >> 6) << 4))
            mn.append((s[..., j + 4] >> 4) | ((s[..., j] >> 6) << 4))
    return torch.stack(sc, -1), torch.stack(mn, -1)


def _bits(words, count, width):
    """Field l of each word (last axis): (word >> width*l) & mask, l < count."""
    sh = torch.arange(count, device=words.device, dtype=torch.int64) * width
    return (words.unsqueeze(-1) >> sh) & ((1 << width) - 1)


def _words(b):
    """Little-endian 32-bit words of bytes along the last axis."""
    b = b.long().view(*b.shape[:-1], -1, 4)
    return b[..., 0] | (b[..., 1] << 8) | (b[..., 2] << 16) | (b[..., 3] << 24)


def _values(fmt, W, n, k, x):
    """The weights of a format in the order its product visits them (float64, n x k)."""
    nbytes, vals = ane_amd.QFORMATS[fmt]
    raw = W.view(n, k // vals, nbytes)
    b = raw.long()

    def half(at):
        return raw[:, :, at:at + 2].contiguous().view(torch.float16).double()  # n, nb, 1

    if fmt == "q4_0":
        lo, hi = _nib(b[:, :, 2:18])
        return ((torch.cat([lo, hi], -1) - 8).double() * half(0)).view(n, k)
    if fmt in ("q4_k", "q5_k"):
        sc, mn = _scale_min6(b[:, :, 4:16])
        qs = b[:, :, 16:144] if fmt == "q4_k" else b[:, :, 48:176]
        lo, hi = _nib(qs.view(n, -1, 8, 16))
        if fmt == "q5_k":
            h = _bits(_words(b[:, :, 16:48]), 32, 1)  # n, nb, 8, 32
            lo, hi = lo | (h[..., :16] << 4), hi | (h[..., 16:] << 4)
        q = torch.cat([lo, hi], -1).double()
        return (q * (half(0) * sc).unsqueeze(-1) - (half(2) * mn).unsqueeze(-1)).view(n, k)
    if fmt == "q2_k":
        q = _bits(_words(b[:, :, 16:80]), 16, 2).double()  # n, nb, 16, 16
        sc, mn = _nib(b[:, :, :16])
        return (q * (half(80) * sc).unsqueeze(-1) - (half(82) * mn).unsqueeze(-1)).view(n, k)
    if fmt == "q6_k":
        lo, hi = _nib(b[:, :, :128].view(n, -1, 16, 8))
        nib = torch.stack([lo, hi], -1).view(n, -1, 16, 16)
        q = nib | (_bits(_words(b[:, :, 128:192]), 16, 2) << 4)
        sc = raw[:, :, 192:208].contiguous().view(torch.int8).double() * half(208)
        return ((q - 32).double() * sc.unsqueeze(-1)).view(n, k)
    # q3_k: the second half of each sub-block shifts its word by the bits of
    # the first half's input before taking its fields
    s = b[:, :, 96:108]
    sc = torch.stack([(s[..., j] & 63) if j < 4 else ((s[..., j + 4] & 15) | ((s[..., j - 4] >> 6) << 4))
                      for j in range(8)], -1)
    words, hm = _words(b[:, :, 32:96]).view(n, -1, 8, 2), _bits(_words(b[:, :, :32]), 32, 1)
    q0 = _bits(words[..., 0], 16, 2) | (hm[..., :16] << 2)
    xb = x.view(torch.int32).long().view(1, -1, 8, 32)[..., :16] & 0xFFFFFFFF
    w1 = torch.where(xb >= 32, torch.zeros_like(xb), words[..., 1].unsqueeze(-1) >> xb.clamp(max=31))
    q1 = ((w1 >> (2 * torch.arange(16, device=W.device))) & 3) | (hm[..., 16:] << 2)
    q = torch.cat([q0, q1], -1) - 4
    return (q.double() * (half(108) * (sc - 32)).unsqueeze(-1)).view(n, k)


def _exp_poly(x):
    """The handlers' exp: 2^floor times a degree-4 polynomial of the fraction."""
    c = [np.array(v, np.uint32).view(np.float32).item()
         for v in (0x3FB8AA3B, 0x3C1D955A, 0x3D635847, 0x3E75FDF0, 0x3F317218)]
    t = x * c[0]
    n = torch.floor(t)
    f = t - n
    return ((((c[1] * f + c[2]) * f + c[3]) * f + c[4]) * f + 1.0) * torch.exp2(n)


def _rows64(i, case):
    T, H = case["T"], case["heads"]
    x = i["x"].double()
    n = x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + 1e-5)
    nw = n * i["w"].double()
    v = i["s"].double() / math.sqrt(128.0) + i["mask"].double()
    d = v - v.amax(dim=2, keepdim=True)
    e = torch.where(torch.isinf(d), torch.zeros_like(d), _exp_poly(torch.where(torch.isinf(d), torch.zeros_like(d), d)))
    gate = i["gate"].double()
    g = gate / (1.0 + _exp_poly(-gate))
    # the rotation is a chain of fp32 products (angles grow with the position):
    # it has no 64-bit value of its own
    return {"n": n, "nw": nw, "q": None, "p": e / e.sum(dim=2, keepdim=True), "g": g, "h": g * i["up"].double(),
            "r": None}


def _token64(i, case):
    G, ffn, pos, V = case["kv_heads"], case["ffn"], case["pos"], case["vocab"]
    H, kvd = G * 512, G * 128

    def norm(x, w):
        return x / torch.sqrt((x * x).mean() + 1e-5) * w.double()

    def rope(q, h):
        a = i["rope"][pos].double()
        p = q.view(h, 64, 2)
        return torch.stack([p[..., 0] * a[:, 0] - p[..., 1] * a[:, 1], p[..., 0] * a[:, 1] + p[..., 1] * a[:, 0]],
                           -1).view(h, 128)

    x = _q8_values(i["embed"][int(i["token"])].view(1, -1), 1, H).view(-1)
    ks, vs = [], []
    for l in i["layers"]:
        qkv = _q8_values(l["w_qkv"], H + 2 * kvd, H) @ _q8_act(norm(x, l["attn_norm"]))
        k, v = l["k"].clone(), l["v"].clone()
        k[:, pos] = rope(qkv[H:H + kvd], G).half()
        v[:, pos] = qkv[H + kvd:].view(G, 128).half()
        q = rope(qkv[:H], 4 * G).view(G, 4, 128)
        p = torch.softmax(q @ k[:, :pos + 1].double().transpose(1, 2).contiguous() / math.sqrt(128.0), dim=-1)
        x = x + _q8_values(l["w_o"], H, H) @ _q8_act((p @ v[:, :pos + 1].double()).reshape(-1))
        gu = (_q8_values(l["w_gate_up"], 2 * ffn, H) @ _q8_act(norm(x, l["ffn_norm"]))).view(-1, 2, 32)
        g, u = gu[:, 0].reshape(-1), gu[:, 1].reshape(-1)
        x = x + _q8_values(l["w_down"], H, ffn) @ _q8_act(g / (1.0 + torch.exp(-g)) * u)
        ks.append(k.double())
        vs.append(v.double())
    logits = _q8_values(i["embed"], V, H) @ _q8_act(norm(x, i["norm"]))
    return {"hidden": x, "logits": logits, "k": ks, "v": vs}


def exact(case, seed):
    i = _inputs(case, seed)
    kind = case["kind"]
    if kind == "mlp":
        h = _fused64(i["x"], i["w1"], True)
        return {"hidden": h, "out": _fused64(h.float(), i["w2"], False)}
    if kind == "fused":
        return _fused64(i["A"], i["B"], case["relu"])
    if kind == "dense":
        s = float(np.float32(0.011) * np.float32(0.0037))
        c = (i["A"].double() @ i["B"].double()) * s + i["bias"].double()
        return c.clamp(min=0.0) if case["relu"] else c
    if kind == "convert":
        K, N = case["K"], case["N"]
        qw, sw = _quant(i["w"], i["w"].abs().amax())
        qx, sx = _quant(i["x"], i["x"].abs().amax(dim=1, keepdim=True))
        b = torch.zeros((_ceil(K, 4), _ceil(N, 16)), device=DEV)
        b[:K, :N] = qw[:K * N].view(K, N)
        panels = b.view(_ceil(K, 4) // 4, 4, _ceil(N, 16) // 16, 16).permute(2, 0, 3, 1).reshape(-1)
        back = qw.double() * float(np.float32(0.0021))
        return {"qw": qw.double(), "sw": sw.double().view(1), "Bp": panels.double(), "qx": qx.double(),
                "sx": sx.double().view(-1), "back": back}
    if kind == "igemm":
        M, N, K = case["M"], case["N"], case["K"] // 64 * 64
        if not K:
            return torch.zeros((M, N), dtype=torch.float64, device=DEV)
        A = (i["A"] if case["variant"] != "igemm" else i["A"].view(torch.int8)).double()
        B = (i["B"] if case["variant"] == "ugemm" else i["B"].view(torch.int8)).double()
        if case["ta"] and not case["blas"]:
            r = torch.arange(M, device=DEV)
            at = ((r % 16) * A.shape[1] + (r - r % 16)).unsqueeze(1) + torch.arange(K, device=DEV)
            A = A.reshape(-1)[at]
        else:
            A = (A.t() if case["ta"] else A)[:M, :K].contiguous()
        B = (B.t() if case["tb"] else B)[:K, :N].contiguous()
        return (A @ B) * float(np.float32(0.0123))
    if kind == "q8":
        return _q8_act(i["x"]) @ _q8_values(i["W"], case["N"], case["K"]).t().contiguous()
    if kind == "q4":
        return i["x"].double() @ _values("q4_0", i["W"], case["N"], case["K"], None).t().contiguous()
    if kind == "kquant":
        return _values(case["fmt"], i["W"], case["N"], case["K"], i["x"]) @ i["x"].double()
    if kind == "rows":
        return _rows64(i, case)
    return _token64(i, case)
