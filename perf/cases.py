"""Performance cases: the work that users of the framework run, through its public entry points.

Two kinds of entry point are called: the model binding (`kernix_amd.kernix.Model`: a .knx file loaded once, then
forwards on device or host buffers) and the kernel C ABI (`kernix_amd.hipabi`: single layers on device buffers the
caller owns).  A case is a dict of plain values; "kind" picks one of the families below, each standing for

    mlp        a small int8-quantized classifier answering one request or a small batch: launches and latency
    qlinear    one int8 Linear on fp32 activations (quantize, product, dequantize, bias, activation)
    i8gemm     the int8 matrix product alone, on rows that are already quantized
    linear     one fp32 Linear layer with its activation, or with the residual it is added to
    conv       one fp32 convolution layer (channels-last), dense or depthwise
    attention  the attention core on a fused Q|K|V projection
    recurrent  one LSTM / GRU / RNN layer over a batch of sequences
    rows       layer_norm, softmax, bias + GELU and elementwise addition
    encoder    a pre-LayerNorm Transformer encoder (int8 weights), called whole on device buffers
    cnn        a residual convolution net, called whole on host buffers, copies included

The framework runs forward passes only, so there is no backward direction to time.  Floating point is fp32, weights
fp32 or per-channel int8; `mode` "ref" multiplies int8 weights as the file format's runtime does (int8 arithmetic for
at most 2 rows, their fp32 values above), "i8" in int8 arithmetic at every size.
"""
import ctypes
import math
import os
import tempfile

import numpy as np
import torch

from kernix_amd import hipabi, knxfile
from kernix_amd.kernix import INT8_I8, INT8_REF, Model

ACT = {"none": -1, "relu": 0, "gelu": 1}
GATES = {"LSTM": 4, "GRU": 3, "RNN": 1}
FLOPS_MAX = 2.0 * 8192 * 4096 * 4096  # the largest listed case (linear_8192x4096x4096)
BYTES_MAX = 4.0 * (2 * 8192 * 4096 + 4096 * 4096)


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one request to a quantized classifier: three dependent layers of one row, nothing but latency
        {"name": "mlp_int8_1", "kind": "mlp", "batch": 1, "dims": "784-512-256-10", "mode": "ref"},
        # a few rows through a large quantized layer (a decode step of a small batch): the weights' bytes
        {"name": "qlinear_16x4096x4096", "kind": "qlinear", "M": 16, "N": 4096, "K": 4096, "act": "relu"},
        # the headline int8 product
        {"name": "i8gemm_4096", "kind": "i8gemm", "M": 4096, "N": 4096, "K": 4096, "act": "relu"},
        # a hidden layer of the large fp32 MLP at its full batch: the largest product
        {"name": "linear_8192x4096x4096", "kind": "linear", "M": 8192, "N": 4096, "K": 4096, "act": "relu", "res": False},
        # a classifier head over an ordinary batch, no size a multiple of a tile
        {"name": "linear_500x1000x2000", "kind": "linear", "M": 500, "N": 1000, "K": 2000, "act": "none", "res": False},
        # the inner convolution of a small image net at a large batch
        {"name": "conv_256x32x32_64to64", "kind": "conv", "B": 256, "hw": 32, "C": 64, "Co": 64, "k": 3, "stride": 1,
         "groups": 1, "act": "relu", "res": False},
        # a strided layer of a larger image net at a small batch: odd image, channels that fill no 32-wide tile
        {"name": "conv_16x57x57_24to80", "kind": "conv", "B": 16, "hw": 57, "C": 24, "Co": 80, "k": 3, "stride": 2,
         "groups": 1, "act": "relu", "res": False},
        # causal attention over a long, ragged sequence
        {"name": "attention_4x12x1000_causal", "kind": "attention", "B": 4, "H": 12, "S": 1000, "d": 64, "causal": True},
        # a recurrent layer over a batch of sequences, its last state
        {"name": "lstm_100x32_200", "kind": "recurrent", "cell": "LSTM", "B": 100, "T": 32, "F": 128, "u": 200,
         "dirs": 1, "seq": False, "int8": False, "mode": "ref"},
        # the normalization of a Transformer's rows: memory bandwidth
        {"name": "layernorm_8192x512", "kind": "rows", "op": "layernorm", "rows": 8192, "cols": 512},
        # a whole quantized Transformer encoder on device buffers
        {"name": "encoder_4x64x128x512", "kind": "encoder", "layers": 4, "B": 64, "S": 128, "d": 512, "heads": 8,
         "mode": "ref"},
        # a whole image classifier from host arrays, as a service calls it
        {"name": "cnn_64_host", "kind": "cnn", "B": 64, "hw": 32, "width": 64},
    ]


def _log(rng, lo, hi, step=1):
    """a size between lo and hi, spread over its logarithm, a multiple of step"""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(lo, min(hi, int(v) // step * step))


def _draw(rng):
    kind = rng.choice(["mlp", "qlinear", "i8gemm", "linear", "linear", "conv", "conv", "attention", "recurrent", "rows",
                       "encoder", "cnn"])
    act = rng.choice(["none", "relu", "gelu"])
    if kind == "mlp":
        dims = [_log(rng, 16, 1024) for _ in range(rng.randint(2, 4))] + [_log(rng, 2, 256)]
        return {"kind": kind, "batch": _log(rng, 1, 64), "dims": "-".join(map(str, dims)), "mode": rng.choice(["ref", "i8"])}
    if kind == "qlinear":
        return {"kind": kind, "M": _log(rng, 1, 4096), "N": _log(rng, 16, 4096), "K": _log(rng, 64, 4096), "act": act}
    if kind == "i8gemm":
        return {"kind": kind, "M": _log(rng, 1, 4096), "N": _log(rng, 16, 4096), "K": _log(rng, 64, 4096, 64), "act": act}
    if kind == "linear":
        res = rng.random() < 0.25
        return {"kind": kind, "M": _log(rng, 1, 8192), "N": _log(rng, 10, 4096), "K": _log(rng, 16, 4096),
                "act": "none" if res else act, "res": res}
    if kind == "conv":
        depthwise = rng.random() < 0.2
        c = _log(rng, 3, 256)
        res = rng.random() < 0.2
        return {"kind": kind, "B": _log(rng, 1, 256), "hw": _log(rng, 7, 64), "C": c, "Co": c if depthwise else _log(rng, 8, 256),
                "k": 3 if depthwise else rng.choice([1, 3, 3, 5]), "stride": rng.choice([1, 1, 2]),
                "groups": c if depthwise else 1, "act": "none" if res else rng.choice(["none", "relu"]), "res": res}
    if kind == "attention":
        return {"kind": kind, "B": _log(rng, 1, 64), "H": _log(rng, 1, 16), "S": _log(rng, 16, 2048),
                "d": rng.choice([16, 32, 48, 64, 64, 80, 96, 128]), "causal": rng.random() < 0.5}
    if kind == "recurrent":
        return {"kind": kind, "cell": rng.choice(["LSTM", "LSTM", "GRU", "RNN"]), "B": _log(rng, 1, 256),
                "T": _log(rng, 4, 32), "F": _log(rng, 8, 256), "u": _log(rng, 16, 256), "dirs": rng.choice([1, 1, 2]),
                "seq": rng.random() < 0.5, "int8": rng.random() < 0.4, "mode": rng.choice(["ref", "i8"])}
    if kind == "rows":
        return {"kind": kind, "op": rng.choice(["layernorm", "softmax", "gelu", "add"]), "rows": _log(rng, 1, 65536),
                "cols": _log(rng, 10, 4096)}
    if kind == "encoder":
        heads = rng.choice([2, 4, 8, 12])
        return {"kind": kind, "layers": rng.randint(1, 4), "B": _log(rng, 1, 64), "S": _log(rng, 8, 384),
                "d": heads * rng.choice([32, 64]), "heads": heads, "mode": rng.choice(["ref", "i8"])}
    return {"kind": kind, "B": _log(rng, 1, 256), "hw": rng.randint(12, 40), "width": rng.choice([16, 24, 32, 48, 64])}


def draw(rng):
    """one more case of the same families and ranges, no larger than the largest listed one"""
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= FLOPS_MAX and w["bytes"] <= BYTES_MAX:
            return case


# ---------------------------------------------------------------- inputs and weights, from the seed alone
def _gen(seed):
    return np.random.default_rng([seed, 20240])


def _normal(seed, stream, shape, std=1.0):
    """fp32 N(0, std) on the GPU"""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 64 + stream)
    return torch.randn(shape, generator=g, device="cuda") * std


def _int8(seed, stream, shape):
    """int8 rows as a quantizer leaves them: N(0, 42), clamped"""
    return (_normal(seed, stream, shape, 42.0)).round_().clamp_(-127, 127).to(torch.int8)


def _quantized(rng, k, n):
    """a quantized k×n weight: (q int8, scale fp32 per column), every column's largest entry ±127 so that the file's
    quantizer gives back these values"""
    q = np.clip(np.rint(rng.standard_normal((k, n), dtype=np.float32) * 42), -127, 127)
    q[rng.integers(0, k, n), np.arange(n)] = 127
    scale = (rng.uniform(0.9, 1.1, n) / (42 * math.sqrt(k))).astype(np.float32)
    return q.astype(np.int8), scale


def _values(w):
    """the real matrix of a (q, scale) weight, or the fp32 matrix itself"""
    return w[0].astype(np.float64) * w[1].astype(np.float64) if isinstance(w, tuple) else w


def _f32w(rng, k, n, gain=1.0):
    return rng.standard_normal((k, n), dtype=np.float32) * np.float32(gain / math.sqrt(k))


def _bias(rng, n):
    return (rng.standard_normal(n) * 0.01).astype(np.float32)


def _dims(case):
    return [int(v) for v in case["dims"].split("-")]


def _weights(case, seed):
    """the weights of a model family, in the order its graph uses them"""
    rng = _gen(seed)
    kind = case["kind"]
    if kind == "mlp":
        d = _dims(case)
        return [(_quantized(rng, a, b), _bias(rng, b)) for a, b in zip(d, d[1:])]
    if kind == "encoder":
        d, out = case["d"], []
        for _ in range(case["layers"]):
            norm = lambda: ((1 + 0.05 * rng.standard_normal(d)).astype(np.float32), (0.05 * rng.standard_normal(d)).astype(np.float32))  # noqa: E731
            out.append({"ln1": norm(), "ln2": norm(), "att": [(_quantized(rng, d, d), _bias(rng, d)) for _ in range(4)],
                        "up": (_quantized(rng, d, 4 * d), _bias(rng, 4 * d)),
                        "down": (_quantized(rng, 4 * d, d), _bias(rng, d))})
        return out
    if kind == "cnn":
        w = case["width"]
        convs = [(_f32w(rng, 9 * ci, co, math.sqrt(2)), _bias(rng, co)) for ci, co in ((3, w), (w, w), (w, 2 * w), (2 * w, 4 * w))]
        return convs + [(_f32w(rng, 4 * w, 10), _bias(rng, 10))]
    g, u, out = GATES[case["cell"]] * case["u"], case["u"], []
    for _ in range(case["dirs"]):
        wx = _f32w(rng, case["F"], g)
        wh = _quantized(rng, u, g) if case["int8"] else _f32w(rng, u, g)
        out.append((wx, wh, _bias(rng, 2 * g if case["cell"] == "GRU" else g)))
    return out


def _model(case, seed):
    """the case's weights saved as a .knx file and loaded"""
    w, kind = _weights(case, seed), case["kind"]
    if kind == "mlp":
        b = knxfile.ModelBuilder((_dims(case)[0],))
        h = b.input
        for i, (q, bias) in enumerate(w):
            h = b.linear(h, _values(q), bias, activation="relu" if i < len(w) - 1 else None, fmt="i8_col")
    elif kind == "encoder":
        b = knxfile.ModelBuilder((case["S"], case["d"]), int8=True)
        x = b.input
        for p in w:
            h = b.layer_norm(x, *p["ln1"], 1e-5)
            ws, bs = [_values(q) for q, _ in p["att"]], [v for _, v in p["att"]]
            x = b.add(x, b.attention(h, case["heads"], *ws, *bs))
            h = b.layer_norm(x, *p["ln2"], 1e-5)
            h = b.linear(h, _values(p["up"][0]), p["up"][1], activation="gelu")
            x = b.add(x, b.linear(h, _values(p["down"][0]), p["down"][1]))
    elif kind == "cnn":
        b = knxfile.ModelBuilder((case["hw"], case["hw"], 3), channels_first=True)
        conv = lambda x, p, s: b.conv(x, p[0], p[1], kernel=(3, 3), stride=(s, s), padding=(1, 1, 1, 1), activation="relu")  # noqa: E731
        h1 = conv(b.input, w[0], 1)
        h = b.add(h1, conv(h1, w[1], 1))
        h = b.global_pool(conv(conv(h, w[2], 2), w[3], 2), "avg")
        b.linear(h, w[4][0], w[4][1])
    else:
        b = knxfile.ModelBuilder((case["T"], case["F"]))
        b.recurrent(b.input, case["cell"], case["u"], [(wx, _values(wh), bias) for wx, wh, bias in w],
                    return_sequences=case["seq"], fmt_recurrent="i8_col" if case["int8"] else "f32")
    fd, path = tempfile.mkstemp(suffix=".knx")
    os.close(fd)
    try:
        b.save(path)
        m = Model(path)
    finally:
        os.unlink(path)
    m.set_int8_mode(INT8_I8 if case.get("mode") == "i8" else INT8_REF)
    return m


def _model_input(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        return _normal(seed, 1, (case["batch"], _dims(case)[0])).abs_().clamp_(0, 1)  # pixel values
    if kind == "encoder":
        return _normal(seed, 1, (case["B"], case["S"], case["d"]))
    if kind == "recurrent":
        return _normal(seed, 1, (case["B"], case["T"], case["F"]))
    return _gen(seed + 1).standard_normal((case["B"], 3, case["hw"], case["hw"]), dtype=np.float32)


def _tensors(case, seed):
    """the operands of a single-layer case"""
    kind = case["kind"]
    if kind in ("qlinear", "i8gemm"):
        M, N, K = case["M"], case["N"], case["K"]
        kp = -(-K // 64) * 64
        t = {"W": torch.zeros((N, kp), dtype=torch.int8, device="cuda"),
             "sw": _normal(seed, 2, (N,)).abs_().clamp_(0.2, 2).mul_(1 / (42 * math.sqrt(K))), "b": _normal(seed, 3, (N,), 0.1)}
        t["W"][:, :K] = _int8(seed, 1, (N, K))
        if kind == "qlinear":
            t["x"] = _normal(seed, 4, (M, K))
        else:
            t["A"], t["sa"] = _int8(seed, 4, (M, K)), _normal(seed, 5, (M,)).abs_().clamp_(0.2, 2).mul_(0.02)
        return t
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        t = {"x": _normal(seed, 1, (M, K)), "W": _normal(seed, 2, (N, K), math.sqrt(2 / K)), "b": _normal(seed, 3, (N,), 0.1)}
        if case["res"]:
            t["R"] = _normal(seed, 4, (M, N))
        return t
    if kind == "conv":
        B, hw, C, Co, k, ho = case["B"], case["hw"], case["C"], case["Co"], case["k"], _out_hw(case)
        kk = k * k * C // case["groups"]
        t = {"x": _normal(seed, 1, (B, hw, hw, C)), "W": _normal(seed, 2, (Co, kk), math.sqrt(2 / kk)), "b": _normal(seed, 3, (Co,), 0.1)}
        if case["res"]:
            t["R"] = _normal(seed, 4, (B, ho, ho, Co))
        return t
    if kind == "attention":
        return {"qkv": _normal(seed, 1, (case["B"] * case["S"], 3 * case["H"] * case["d"]))}
    r, c = case["rows"], case["cols"]
    t = {"x": _normal(seed, 1, (r, c), 2.0), "b": _normal(seed, 3, (c,), 0.1)}
    if case["op"] == "layernorm":
        t["g"] = 1 + _normal(seed, 2, (c,), 0.05)
    if case["op"] == "add":
        t["z"] = _normal(seed, 4, (r, c))
    return t


def _out_hw(case):
    return (case["hw"] + 2 * (case["k"] // 2) - case["k"]) // case["stride"] + 1


def _out_shape(case):
    kind = case["kind"]
    if kind in ("qlinear", "i8gemm", "linear"):
        return (case["M"], case["N"])
    if kind == "conv":
        return (case["B"], _out_hw(case), _out_hw(case), case["Co"])
    if kind == "attention":
        return (case["B"] * case["S"], case["H"] * case["d"])
    if kind == "mlp":
        return (case["batch"], _dims(case)[-1])
    if kind == "encoder":
        return (case["B"], case["S"], case["d"])
    if kind == "recurrent":
        return (case["B"], case["T"], case["u"] * case["dirs"]) if case["seq"] else (case["B"], case["u"] * case["dirs"])
    return (case["rows"], case["cols"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "cnn":
        return {"case": case, "model": _model(case, seed), "x": _model_input(case, seed)}
    st = {"case": case, "y": torch.empty(_out_shape(case), device="cuda")}
    if kind in ("mlp", "encoder", "recurrent"):
        st.update(model=_model(case, seed), x=_model_input(case, seed), stream=torch.cuda.Stream())
        st["rows"] = st["x"].numel() // st["x"].shape[-1]
        torch.cuda.synchronize()  # the model runs on a stream of its own
        return st
    st.update(_tensors(case, seed))
    if kind == "qlinear":
        kp = st["W"].shape[1]
        st["xq"] = torch.empty((case["M"], kp), dtype=torch.int8, device="cuda")
        st["sx"] = torch.empty((case["M"],), device="cuda")
    elif kind == "conv":
        k, hw, ho = case["k"], case["hw"], _out_hw(case)
        st["geom"] = hipabi.ConvGeom(case["B"], hw, hw, case["C"], ho, ho, case["Co"], k, k, case["stride"], case["stride"],
                                     1, 1, k // 2, k // 2, case["groups"])
    elif kind == "attention":
        n = case["B"] * case["H"] * case["S"]
        st["scores"] = torch.empty((n * case["S"],), device="cuda")
        st["vt"] = torch.empty((n * case["d"],), device="cuda")
    return st


def run(st):
    """one pass; enqueues on the state's (or torch's current) stream and returns the output buffer"""
    case = st["case"]
    kind = case["kind"]
    if kind == "cnn":
        return st["model"](st["x"])
    if "model" in st:
        st["model"].forward_device(st["x"].data_ptr(), st["rows"], st["y"].data_ptr(), st["stream"].cuda_stream)
        return st["y"]
    L, P, S, y = hipabi.lib(), hipabi.ptr, hipabi.stream(), st["y"]
    if kind == "qlinear":
        M, N, K, kp = case["M"], case["N"], case["K"], st["W"].shape[1]
        rc = L.knx_hip_qlinear(P(st["x"]), K, M, K, kp, P(st["xq"]), P(st["sx"]), P(st["W"]), kp, N, P(st["sw"]), P(st["b"]),
                               ACT[case["act"]], 0.0, 0, None, 0, P(y), N, S)
    elif kind == "i8gemm":
        M, N, K = case["M"], case["N"], case["K"]
        rc = L.knx_hip_i8gemm(M, N, K, P(st["A"]), K, P(st["sa"]), P(st["W"]), K, P(st["sw"]), P(st["b"]), ACT[case["act"]],
                              0.0, 0, P(y), N, None, 0, S)
    elif kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        if case["res"]:
            rc = L.knx_hip_sgemm_nt_ep_res(M, N, K, P(st["x"]), K, P(st["W"]), K, P(st["b"]), ACT[case["act"]], 0.0, P(st["R"]),
                                           N, P(y), N, S)
        else:
            rc = L.knx_hip_sgemm_nt_ep(M, N, K, P(st["x"]), K, P(st["W"]), K, P(st["b"]), ACT[case["act"]], 0.0, P(y), N, S)
    elif kind == "conv":
        g = ctypes.byref(st["geom"])
        if case["res"]:
            rc = L.knx_hip_conv_t_res(g, P(st["x"]), P(st["W"]), P(st["b"]), ACT[case["act"]], 0.0, P(st["R"]), P(y), S)
        else:
            rc = L.knx_hip_conv_t(g, P(st["x"]), P(st["W"]), P(st["b"]), ACT[case["act"]], 0.0, P(y), S)
    elif kind == "attention":
        H, d, s = case["H"], case["d"], case["S"]
        q = st["qkv"].data_ptr()
        at = lambda i: ctypes.c_void_p(q + 4 * i * H * d)  # noqa: E731
        rc = L.knx_hip_attention_core_ex(at(0), 3 * H * d, at(1), 3 * H * d, at(2), 3 * H * d, P(st["vt"]), P(y),
                                         P(st["scores"]), case["B"], H, s, s, d, d, 1 / math.sqrt(d), int(case["causal"]), S)
    else:
        r, c = case["rows"], case["cols"]
        if case["op"] == "layernorm":
            rc = L.knx_hip_layernorm(P(st["x"]), P(y), r, c, P(st["g"]), P(st["b"]), 1e-5, S)
        elif case["op"] == "softmax":
            rc = L.knx_hip_softmax(P(st["x"]), P(y), r, c, S)
        elif case["op"] == "gelu":
            rc = L.knx_hip_bias_act(P(st["x"]), P(y), r, c, P(st["b"]), ACT["gelu"], 0.0, S)
        else:
            rc = L.knx_hip_binary(knxfile.BINARY_OPS.index("add"), P(st["x"]), r, c, P(st["z"]), r, c, P(y), 1, r, c, S)
    hipabi.check(rc)
    return y


# ---------------------------------------------------------------- the work of one pass
def work(case):
    kind = case["kind"]
    if kind == "mlp":
        d, m = _dims(case), case["batch"]
        prod = sum(a * b for a, b in zip(d, d[1:]))
        return {"bytes": prod + 4 * m * (d[0] + d[-1]) + 8 * sum(d[1:]), "flops": 2.0 * m * prod}
    if kind in ("qlinear", "i8gemm", "linear"):
        M, N, K = case["M"], case["N"], case["K"]
        a, w = {"qlinear": (4, 1), "i8gemm": (1, 1), "linear": (4, 4)}[kind]
        return {"bytes": a * M * K + w * N * K + 4 * M * N * (2 if case.get("res") else 1) + 8 * N, "flops": 2.0 * M * N * K}
    if kind == "conv":
        B, C, Co, hw, ho = case["B"], case["C"], case["Co"], case["hw"], _out_hw(case)
        kk = case["k"] ** 2 * C // case["groups"]
        return {"bytes": 4.0 * (B * hw * hw * C + B * ho * ho * Co * (2 if case["res"] else 1) + kk * Co),
                "flops": 2.0 * B * ho * ho * Co * kk}
    if kind == "attention":
        B, H, S, d = case["B"], case["H"], case["S"], case["d"]
        pairs = S * (S + 1) / 2 if case["causal"] else S * S
        return {"bytes": 16.0 * B * H * S * d, "flops": 4.0 * B * H * pairs * d}
    if kind == "recurrent":
        B, T, F, u, n = case["B"], case["T"], case["F"], case["u"], case["dirs"]
        g = GATES[case["cell"]] * u
        w = n * g * (4 * F + (1 if case["int8"] else 4) * u)
        return {"bytes": 4.0 * B * T * F + w + 4.0 * B * u * n * (T if case["seq"] else 1), "flops": 2.0 * n * B * T * g * (F + u)}
    if kind == "rows":
        n = case["rows"] * case["cols"]
        return {"bytes": 4.0 * n * (3 if case["op"] == "add" else 2), "flops": n * {"layernorm": 8.0, "softmax": 5.0, "gelu": 20.0, "add": 1.0}[case["op"]]}
    if kind == "encoder":
        B, S, d, n = case["B"], case["S"], case["d"], case["layers"]
        return {"bytes": 8.0 * B * S * d + n * 12.0 * d * d, "flops": n * B * S * (24.0 * d * d + 4.0 * S * d)}
    B, hw, w = case["B"], case["hw"], case["width"]
    h2 = (hw + 1) // 2
    h4 = (h2 + 1) // 2
    per = hw * hw * 9 * w * (3 + w) + h2 * h2 * 18 * w * w + h4 * h4 * 72 * w * w + 40 * w
    return {"bytes": 4.0 * (3 * B * hw * hw + 10 * B + 9 * w * (3 + w) + 90 * w * w), "flops": 2.0 * B * per}


def tolerance(case):
    """fp32 sums in another order: about four times the distance to 64-bit arithmetic over the ranges"""
    kind = case["kind"]
    if kind in ("i8gemm", "qlinear"):
        return {"rel": 2e-6}  # exact integer sums; the fp32 epilogue, and GELU's 7.1.26 polynomial
    if kind == "mlp":
        # a last-bit difference in an activation can move one value across a rounding edge of the next quantization
        return {"rel": 5e-3}
    if kind == "encoder":
        return {"rel": 1e-2 if case["mode"] == "i8" or case["B"] * case["S"] <= 2 else 1e-5}
    if kind == "recurrent":
        return {"rel": 5e-3 if case["int8"] and (case["mode"] == "i8" or case["B"] <= 2) else 1e-5}
    return {"rel": 5e-6}


# ---------------------------------------------------------------- the same in 64 bits
def _erf_gelu(v):
    return 0.5 * v * (1 + torch.erf(v / math.sqrt(2)))


def _activate(v, act):
    return torch.relu(v) if act == "relu" else _erf_gelu(v) if act == "gelu" else v


def _quantize_rows(x):
    """the row quantization as it is defined, in fp32 steps: (integers as float64, scale fp32)"""
    x = x.float()
    peak = x.abs().amax(dim=-1, keepdim=True)
    sx = torch.where(peak > 0, peak / torch.full_like(peak, 127.0), torch.ones_like(peak))
    inv = torch.ones_like(sx) / sx
    return (x * inv).round().clamp(-127, 127).double(), sx


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _product(x, w, int8):
    """x·w in float64, w an fp32 matrix or (q, scale); int8: the rows of x quantized first"""
    if not isinstance(w, tuple):
        return x @ _dev(w).double()
    q, s = _dev(w[0]), _dev(w[1])
    if int8:
        xq, sx = _quantize_rows(x)
        return (xq @ q.double()) * sx.double() * s.double()
    return x @ (q.float() * s).double()


def _layer_norm(x, g, b, eps=1e-5):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + eps) * g + b


def _attention(q, k, v, causal):
    """per (batch, head): q, k, v are B × H × S × d, one head at a time to bound the scores' memory"""
    out = torch.empty_like(q)
    S = q.shape[2]
    mask = torch.ones((S, S), dtype=torch.bool, device=q.device).triu(1) if causal else None
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            s = (q[b, h] @ k[b, h].t().contiguous()) / math.sqrt(q.shape[3])
            if causal:
                s = s.masked_fill(mask, -math.inf)
            out[b, h] = torch.softmax(s, -1) @ v[b, h]
    return out


def _heads(x, B, S, H):
    return x.reshape(B, S, H, -1).permute(0, 2, 1, 3).contiguous()


def _conv64(x, w, k, stride, groups):
    """channels-last convolution, padding k // 2: a sum over taps; w is (ky, kx, ci) rows × co in float64"""
    B, hw, _, C = x.shape
    p = k // 2
    ho = (hw + 2 * p - k) // stride + 1
    xp = torch.zeros((B, hw + 2 * p, hw + 2 * p, C), dtype=torch.float64, device=x.device)
    xp[:, p:p + hw, p:p + hw] = x
    y = 0
    for t in range(k * k):
        part = xp[:, t // k:t // k + (ho - 1) * stride + 1:stride, t % k:t % k + (ho - 1) * stride + 1:stride]
        if groups == 1:
            y = y + (part.reshape(-1, C) @ w[t * C:(t + 1) * C]).reshape(B, ho, ho, -1)
        else:  # depthwise
            y = y + part * w[t]
    return y


def _recurrent64(case, x, weights):
    u, T = case["u"], case["T"]
    int8 = case["int8"] and (case["mode"] == "i8" or case["B"] <= 2)
    outs = []
    for back, (wx, wh, bias) in enumerate(weights):
        bias = _dev(bias).double()
        g = GATES[case["cell"]] * u
        zx = x @ _dev(wx).double() + bias[:g]
        h = torch.zeros((case["B"], u), dtype=torch.float64, device="cuda")
        c, seq = torch.zeros_like(h), [None] * T
        for t in (range(T - 1, -1, -1) if back else range(T)):
            rec = _product(h, wh, int8)
            z = zx[:, t]
            if case["cell"] == "LSTM":
                i, f, cc, o = (z + rec).split(u, 1)
                c = torch.sigmoid(f) * c + torch.sigmoid(i) * torch.tanh(cc)
                h = torch.tanh(c) * torch.sigmoid(o)
            elif case["cell"] == "GRU":
                rec = rec + bias[g:]
                zr = torch.sigmoid(z[:, :2 * u] + rec[:, :2 * u])
                hh = torch.tanh(zr[:, u:] * rec[:, 2 * u:] + z[:, 2 * u:])
                h = (h - hh) * zr[:, :u] + hh
            else:
                h = torch.tanh(z + rec)
            seq[t] = h
        outs.append(torch.stack(seq, 1) if case["seq"] else h)
    return torch.cat(outs, -1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mlp", "encoder", "recurrent", "cnn"):
        w = _weights(case, seed)
        x = _model_input(case, seed)
        if kind == "cnn":
            x = _dev(x).double().permute(0, 2, 3, 1).contiguous()
            conv = lambda v, p, s: torch.relu(_conv64(v, _dev(p[0]).double(), 3, s, 1) + _dev(p[1]).double())  # noqa: E731
            h1 = conv(x, w[0], 1)
            h = conv(conv(h1 + conv(h1, w[1], 1), w[2], 2), w[3], 2)
            return (h.mean((1, 2)) @ _dev(w[4][0]).double() + _dev(w[4][1]).double()).cpu().numpy()
        x = x.double()
        if kind == "recurrent":
            return _recurrent64(case, x, w)
        if kind == "mlp":
            int8 = case["mode"] == "i8" or case["batch"] <= 2
            for i, (q, bias) in enumerate(w):
                x = _product(x, q, int8) + _dev(bias).double()
                x = torch.relu(x) if i < len(w) - 1 else x
            return x
        B, S, d, H = case["B"], case["S"], case["d"], case["heads"]
        int8 = case["mode"] == "i8" or B * S <= 2
        x = x.reshape(B * S, d)
        for p in w:
            h = _layer_norm(x, *[_dev(v).double() for v in p["ln1"]])
            q, k, v = (_heads(_product(h, a, False) + _dev(b).double(), B, S, H) for a, b in p["att"][:3])
            ctx = _attention(q, k, v, False).permute(0, 2, 1, 3).reshape(B * S, d)
            x = x + _product(ctx, p["att"][3][0], False) + _dev(p["att"][3][1]).double()
            h = _layer_norm(x, *[_dev(v).double() for v in p["ln2"]])
            h = _erf_gelu(_product(h, p["up"][0], int8) + _dev(p["up"][1]).double())
            x = x + _product(h, p["down"][0], int8) + _dev(p["down"][1]).double()
        return x.reshape(B, S, d)
    t = {n: v for n, v in _tensors(case, seed).items()}
    if kind == "qlinear":
        xq, sx = _quantize_rows(t["x"])
        return _activate((xq @ t["W"][:, :case["K"]].double().t()) * sx.double() * t["sw"].double() + t["b"].double(), case["act"])
    if kind == "i8gemm":
        acc = t["A"].double() @ t["W"].double().t()
        return _activate(acc * t["sa"].double()[:, None] * t["sw"].double() + t["b"].double(), case["act"])
    if kind == "linear":
        y = _activate(t["x"].double() @ t["W"].double().t() + t["b"].double(), case["act"])
        return y + t["R"].double() if case["res"] else y
    if kind == "conv":
        wk = t["W"].double().t().contiguous()
        y = _activate(_conv64(t["x"].double(), wk, case["k"], case["stride"], case["groups"]) + t["b"].double(), case["act"])
        return y + t["R"].double() if case["res"] else y
    if kind == "attention":
        B, S, H, d = case["B"], case["S"], case["H"], case["d"]
        q, k, v = (_heads(p, B, S, H) for p in t["qkv"].double().split(H * d, 1))
        return _attention(q, k, v, case["causal"]).permute(0, 2, 1, 3).reshape(B * S, H * d)
    x, b = t["x"].double(), t["b"].double()
    if case["op"] == "layernorm":
        return _layer_norm(x, t["g"].double(), b)
    if case["op"] == "softmax":
        return torch.softmax(x, -1)
    if case["op"] == "gelu":
        return _erf_gelu(x + b)
    return x + t["z"].double()
