"""The work that users of this library have it do, as measurable cases.

Whole embedding calls (FastFace / fastface.h) over the range of batch sizes,
sources and pixel types, and single layers through the kernel-level ABI
(fastface_kernels.h): the tuned IResNet convolutions, convolutions of other
geometries, the FC head and the stand-alone elementwise ops.  Every result is
an int8 tensor or an embedding whose bits are specified (integer sums are
exact and each fp32 operation is one IEEE rounding), so results compare
exactly.
"""
import ctypes as C
import math
import os
import struct

import numpy as np
import torch

import fastface_amd as fa
from fastface_amd import synth

ROOT = synth.REPO_ROOT
FACE = fa.FASTFACE_INPUT_N
EMB = fa.FASTFACE_OUTPUT_N
FC_K = 25088
MODEL_SEED = 3
DEV = "cuda"

# The IResNet layer geometries (cin, cout, kernel, stride, input size).  A
# stage's 1x1 shortcut reads the compact block input, so it runs at stride 1.
LAYERS = (
    (64, 64, 3, 1, 112), (64, 64, 3, 2, 112), (64, 64, 1, 1, 56), (64, 64, 3, 1, 56),
    (64, 128, 3, 1, 56), (128, 128, 3, 2, 56), (64, 128, 1, 1, 28), (128, 128, 3, 1, 28),
    (128, 256, 3, 1, 28), (256, 256, 3, 2, 28), (128, 256, 1, 1, 14), (256, 256, 3, 1, 14),
    (256, 512, 3, 1, 14), (512, 512, 3, 2, 14), (256, 512, 1, 1, 7), (512, 512, 3, 1, 7),
)


def listed():
    return [
        # One face, host to host: the reference's headline latency (an
        # interactive verification call).
        {"name": "embed_1_host", "kind": "embed", "batch": 1, "source": "host_f32"},
        # The faces of one video frame, already on the GPU from a detector.
        {"name": "embed_8_device", "kind": "embed", "batch": 8, "source": "device_f32"},
        # A crowded frame's uint8 crops, an odd number of them.
        {"name": "embed_37_device_rgb8", "kind": "embed", "batch": 37, "source": "device_rgb8"},
        # A gallery import from decoded images in host memory.
        {"name": "embed_203_host_rgb8", "kind": "embed", "batch": 203, "source": "host_rgb8"},
        # Offline throughput: the benchmark's batch.
        {"name": "embed_1024_device", "kind": "embed", "batch": 1024, "source": "device_f32"},
        # The network's commonest layer (26 of 53 convs) at the batch the
        # benchmark quotes for it.
        {"name": "conv_256_14_n64", "kind": "conv", "cin": 256, "cout": 256, "k": 3, "stride": 1, "pad": 1,
         "hin": 14, "batch": 64, "epi": "prelu"},
        # An early layer with large images and few channels, large batch.
        {"name": "conv_64_56_n384", "kind": "conv", "cin": 64, "cout": 64, "k": 3, "stride": 1, "pad": 1,
         "hin": 56, "batch": 384, "epi": "add_bn"},
        # A late layer at a handful of faces: long reductions, few outputs.
        {"name": "conv_512_7_n5", "kind": "conv", "cin": 512, "cout": 512, "k": 3, "stride": 1, "pad": 1,
         "hin": 7, "batch": 5, "epi": "add_bn"},
        # The embedding head for the faces of one frame.
        {"name": "fc_n13", "kind": "fc", "batch": 13},
        # Convolutions of models other than IResNet at 112x112: a 5x5 layer
        # of the network's width, and a narrower layer at an odd image size.
        {"name": "conv_5x5_256_14_n256", "kind": "conv", "cin": 256, "cout": 256, "k": 5, "stride": 1, "pad": 2,
         "hin": 14, "batch": 256, "epi": "prelu"},
        {"name": "conv_3x3_96_45_n33", "kind": "conv", "cin": 96, "cout": 96, "k": 3, "stride": 1, "pad": 1,
         "hin": 45, "batch": 33, "epi": "prelu"},
        # A BN that no conv absorbs (the final BN of other networks).
        {"name": "bn_128_28_n300", "kind": "bn", "channels": 128, "pixels": 300 * 28 * 28},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["embed", "embed", "embed", "conv", "conv", "conv", "other", "other", "fc", "bn", "add"])
    if kind == "embed":
        return {"kind": "embed", "batch": _log_int(rng, 1, 1024),
                "source": rng.choice(["device_f32", "device_rgb8", "host_f32", "host_rgb8"])}
    if kind == "conv":
        cin, cout, k, stride, hin = rng.choice(LAYERS)
        return {"kind": "conv", "cin": cin, "cout": cout, "k": k, "stride": stride, "pad": k // 2, "hin": hin,
                "batch": _log_int(rng, 1, 1024), "epi": rng.choice(["prelu", "none", "prelu_bn", "add_bn"])}
    if kind == "other":
        k = rng.choice([1, 3, 5, 7])
        cin = rng.choice([16, 24, 32, 48, 80, 96, 160, 192, 256, 320])
        cout = 8 * rng.randint(2, 48)
        hin = rng.randint(max(k, 7), 80)
        most = 3e11 / (2.0 * cin * cout * k * k * hin * hin)
        return {"kind": "conv", "cin": cin, "cout": cout, "k": k, "stride": rng.choice([1, 1, 2]), "pad": k // 2,
                "hin": hin, "batch": max(1, min(256, int(most), _log_int(rng, 1, 256))),
                "epi": rng.choice(["prelu", "none", "add_bn"])}
    if kind == "fc":
        return {"kind": "fc", "batch": _log_int(rng, 1, 2048)}
    # stand-alone elementwise ops
    c = rng.choice([64, 128, 256, 512])
    return {"kind": kind, "channels": c, "pixels": _log_int(rng, 49, 1024 * 3136 * 64 // c)}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _activations(shape, g):
    """int8 activations as the network's requantized tensors hold them."""
    return torch.randn(shape, generator=g, device=DEV).mul_(40.0).round_().clamp_(-128, 127).to(torch.int8)


def _weights(shape, g):
    return torch.randint(-127, 128, shape, generator=g, device=DEV, dtype=torch.int8)


def _uniform(n, lo, hi, g):
    return torch.rand(n, generator=g, device=DEV) * (hi - lo) + lo


def _faces(case, seed):
    """fp32 faces in [-1, 1] or uint8 pixels, [B, 112, 112, 3], on the GPU."""
    shape = (case["batch"], 112, 112, 3)
    if case["source"].endswith("rgb8"):
        return torch.randint(0, 256, shape, generator=_gen(seed), device=DEV, dtype=torch.uint8)
    return torch.rand(shape, generator=_gen(seed), device=DEV) * 2.0 - 1.0


def _out_hw(case):
    return (case["hin"] + 2 * case["pad"] - case["k"]) // case["stride"] + 1


def _conv_inputs(case, seed):
    """Input, OIHW weights, [FFK_NPARAM][cout] parameters and the residual of
    a conv case, scaled as the network's layers are (outputs spread over the
    int8 range, residual and output of the same scale)."""
    g = _gen(seed)
    cin, cout, k, n, h = case["cin"], case["cout"], case["k"], case["batch"], case["hin"]
    ho = _out_hw(case)
    scale = _uniform(cout, 0.015, 0.03, g)
    P = torch.zeros((fa.FFK_NPARAM, cout), device=DEV)
    P[fa.FFK_P_WS] = scale * _uniform(cout, 0.5, 1.5, g) / (math.sqrt(cin * k * k) * 73.6)
    P[fa.FFK_P_BIAS] = torch.randn(cout, generator=g, device=DEV) * 0.05
    P[fa.FFK_P_SLOPE] = _uniform(cout, 0.0, 0.3, g)
    P[fa.FFK_P_ADDSCALE] = scale * 0.8
    P[fa.FFK_P_INV] = 1.0 / (scale + 1e-9)
    P[fa.FFK_P_BN_SIN] = scale
    P[fa.FFK_P_BN_S] = _uniform(cout, 0.5, 1.5, g)
    P[fa.FFK_P_BN_O] = torch.randn(cout, generator=g, device=DEV) * 0.05
    P[fa.FFK_P_BN_INV] = 1.0 / (scale + 1e-9)
    w = _weights((cout, cin, k, k), g)
    x = _activations((n, h, h, cin), g)
    add = _activations((n, ho, ho, cout), g) if case["epi"].startswith("add") else None
    return x, w, P, add


def _fc_inputs(case, seed):
    g = _gen(seed)
    w = _weights((EMB, FC_K), g)
    ws = _uniform(EMB, 0.5, 1.5, g) / (math.sqrt(FC_K) * 73.6 * 40.0)
    bias = torch.randn(EMB, generator=g, device=DEV) * 0.05
    return _activations((case["batch"], FC_K), g), w, ws, bias


def _bn_inputs(case, seed):
    g = _gen(seed)
    c = case["channels"]
    s_in = _uniform(c, 0.015, 0.03, g)
    rows = torch.stack([s_in, _uniform(c, 0.5, 1.5, g), torch.randn(c, generator=g, device=DEV) * 0.05,
                        1.0 / (s_in + 1e-9)])
    return _activations((case["pixels"], c), g), rows


_ADD_SCALES = (0.021, 0.017, 0.027)     # the op's per-tensor scales: a, b, output


def _add_inputs(case, seed):
    g = _gen(seed)
    shape = (case["pixels"], case["channels"])
    return _activations(shape, g), _activations(shape, g)


# ---------------------------------------------------------------- states

def _ok(rc):
    if rc != 0:
        raise RuntimeError("call failed (%d): %s" % (rc, fa.last_error()))


_model = None


def _face_model():
    """The context a server keeps for its life: one model, any batch size."""
    global _model
    if _model is None:
        _model = fa.FastFace(synth.synthetic_ffw4_path(MODEL_SEED), cwd=ROOT)
    return _model


def _prepare_embed(case, seed):
    x = _faces(case, seed)
    st = {"kind": case["source"], "ff": _face_model(), "lib": fa.load(), "batch": case["batch"]}
    if case["source"].startswith("host"):
        st["x"] = x.cpu().numpy()
    else:
        st["x"] = x
        st["out"] = torch.empty((case["batch"], EMB), device=DEV)
    return st


def _prepare_conv(case, seed):
    lib = fa.load()
    x, w, P, add = _conv_inputs(case, seed)
    n, ho, cout, epi = case["batch"], _out_hw(case), case["cout"], case["epi"]
    k, ktot = case["k"], case["k"] * case["k"] * case["cin"]
    w_host, P_host = w.cpu().contiguous(), P.cpu().contiguous()
    packed = torch.empty(lib.ffk_conv_packed_bytes(case["cin"], cout, k, k), dtype=torch.int8)
    _ok(lib.ffk_pack_conv_weights(w_host.data_ptr(), cout, case["cin"], k, k, packed.data_ptr()))
    # the epilogue forms the launch plan proves for these parameters
    flags = fa.FFK_EPI_BIAS
    flags |= fa.FFK_EPI_PRELU if epi.startswith("prelu") else 0
    flags |= fa.FFK_EPI_ADD if epi.startswith("add") else 0
    flags |= fa.FFK_EPI_BN if epi.endswith("bn") else 0
    if flags & fa.FFK_EPI_PRELU and lib.ffk_prelu_le1_ok(P_host.data_ptr(), cout, ktot, 0):
        flags |= fa.FFK_EPI_PRELU_LE1
    if lib.ffk_requant_in_range(P_host.data_ptr(), cout, ktot, flags):
        flags |= fa.FFK_EPI_IN_RANGE
        if lib.ffk_requant_fma_ok(P_host.data_ptr(), cout, ktot, flags):
            flags |= fa.FFK_EPI_FMA_TAIL
    keep = {"x": x, "w": packed.to(DEV), "P": P, "add": add,
            "out": torch.empty((n, ho, ho, cout), dtype=torch.int8, device=DEV)}
    d = fa.ffk_conv_desc()
    d.batch, d.cin, d.cout, d.kh, d.kw = n, case["cin"], cout, k, k
    d.stride, d.pad, d.hin, d.win = case["stride"], case["pad"], case["hin"], case["hin"]
    d.in_, d.w, d.params, d.out = x.data_ptr(), keep["w"].data_ptr(), P.data_ptr(), keep["out"].data_ptr()
    d.flags = flags
    if add is not None:
        d.add_src = add.data_ptr()
    outs = [keep["out"]]
    if flags & fa.FFK_EPI_BN:
        lut = torch.empty((cout, 256), dtype=torch.int8)
        _ok(lib.ffk_make_bn_lut(*(P_host[r].data_ptr() for r in (fa.FFK_P_BN_SIN, fa.FFK_P_BN_S, fa.FFK_P_BN_O,
                                                                 fa.FFK_P_BN_INV)), cout, lut.data_ptr()))
        keep["lut"], keep["out_bn"] = lut.to(DEV), torch.empty_like(keep["out"])
        d.bn_lut, d.out_bn = keep["lut"].data_ptr(), keep["out_bn"].data_ptr()
        outs.append(keep["out_bn"])
    need = lib.ffk_conv_workspace_bytes(C.byref(d))
    if need:
        keep["ws"] = torch.zeros(need, dtype=torch.int8, device=DEV)
        d.workspace, d.workspace_bytes = keep["ws"].data_ptr(), need
    return {"kind": "conv", "lib": lib, "desc": d, "keep": keep, "outs": outs}


def _prepare_fc(case, seed):
    lib = fa.load()
    a, w, ws, bias = _fc_inputs(case, seed)
    w_host = w.cpu().contiguous()
    packed = torch.empty(lib.ffk_fc_packed_bytes(EMB, FC_K), dtype=torch.int8)
    _ok(lib.ffk_pack_fc_weights(w_host.data_ptr(), EMB, FC_K, packed.data_ptr()))
    keep = {"a": a, "w": packed.to(DEV), "ws": ws, "bias": bias,
            "out": torch.empty((case["batch"], EMB), device=DEV)}
    d = fa.ffk_fc_desc()
    d.batch, d.n, d.k = case["batch"], EMB, FC_K
    d.a, d.w, d.ws, d.bias = a.data_ptr(), keep["w"].data_ptr(), ws.data_ptr(), bias.data_ptr()
    d.a_scale, d.out = 1.0, keep["out"].data_ptr()
    need = lib.ffk_fc_workspace_bytes(C.byref(d))
    if need:
        keep["wk"] = torch.zeros(need, dtype=torch.int8, device=DEV)
        d.workspace, d.workspace_bytes = keep["wk"].data_ptr(), need
    return {"kind": "fc", "lib": lib, "desc": d, "keep": keep}


def _prepare_bn(case, seed):
    lib = fa.load()
    x, rows = _bn_inputs(case, seed)
    r = rows.cpu().contiguous()
    lut = torch.empty((case["channels"], 256), dtype=torch.int8)
    _ok(lib.ffk_make_map_lut(r[0].data_ptr(), r[1].data_ptr(), r[2].data_ptr(), None, r[3].data_ptr(),
                             case["channels"], lut.data_ptr()))
    return {"kind": "bn", "lib": lib, "x": x, "lut": lut.to(DEV), "out": torch.empty_like(x)}


def _prepare_add(case, seed):
    lib = fa.load()
    a, b = _add_inputs(case, seed)
    lut = torch.empty(65536, dtype=torch.int8)
    _ok(lib.ffk_make_add_lut(*_ADD_SCALES, lut.data_ptr()))
    return {"kind": "add", "lib": lib, "a": a, "b": b, "lut": lut.to(DEV), "out": torch.empty_like(a)}


def prepare(case, seed):
    return {"embed": _prepare_embed, "conv": _prepare_conv, "fc": _prepare_fc, "bn": _prepare_bn,
            "add": _prepare_add}[case["kind"]](case, seed)


def run(st):
    kind = st["kind"]
    if kind == "host_f32":
        if st["batch"] == 1:
            return st["ff"].embed(st["x"][0])
        return st["ff"].embed_batch(st["x"])
    if kind == "host_rgb8":
        return st["ff"].embed_batch_rgb8(st["x"])
    lib = st["lib"]
    if kind == "device_f32":
        _ok(lib.fastface_embed_batch_device(st["ff"].ff, st["x"].data_ptr(), st["batch"], st["out"].data_ptr(), None))
        return st["out"]
    if kind == "device_rgb8":
        _ok(lib.fastface_embed_batch_rgb8_device(st["ff"].ff, st["x"].data_ptr(), st["batch"], st["out"].data_ptr(),
                                                 None))
        return st["out"]
    if kind == "conv":
        _ok(lib.ffk_conv(C.byref(st["desc"]), None))
        return st["outs"]
    if kind == "fc":
        _ok(lib.ffk_fc(C.byref(st["desc"]), None))
        return st["keep"]["out"]
    if kind == "bn":
        n, c = st["x"].shape
        _ok(lib.ffk_map_i8(st["x"].data_ptr(), st["out"].data_ptr(), n, c, st["lut"].data_ptr(), None))
        return st["out"]
    _ok(lib.ffk_add_i8(st["a"].data_ptr(), st["b"].data_ptr(), st["out"].data_ptr(), st["a"].numel(),
                       st["lut"].data_ptr(), None))
    return st["out"]


def work(case):
    kind = case["kind"]
    if kind == "embed":
        b = case["batch"]
        px = 1 if case["source"].endswith("rgb8") else 4
        macs, weights = 0, 0
        hw, cin = 112, 3
        for op in synth.iresnet_schedule():
            if op["type"] == synth.OP_CONV:
                shortcut = op["k"] == 1
                h_out = hw if shortcut or op["s"] == 1 else hw // 2     # (the shortcut follows the strided conv)
                macs += h_out * h_out * op["Cout"] * op["Cin"] * op["k"] ** 2
                weights += op["Cout"] * op["Cin"] * op["k"] ** 2
                hw = h_out
            elif op["type"] == synth.OP_GEMM:
                macs += op["N"] * op["K"]
                weights += op["N"] * op["K"]
        return {"bytes": b * (FACE * px + EMB * 4) + weights, "flops": 2.0 * macs * b}
    if kind == "conv":
        n, ho, cin, cout, k, h = case["batch"], _out_hw(case), case["cin"], case["cout"], case["k"], case["hin"]
        outs = n * ho * ho * cout
        epi = case["epi"]
        streams = 1 + epi.startswith("add") + epi.endswith("bn")
        # a 1x1 stride-2 conv reads a quarter of the pixels
        read = n * (ho * ho if k == 1 else h * h) * cin
        return {"bytes": read + streams * outs + cout * cin * k * k, "flops": 2.0 * outs * cin * k * k}
    if kind == "fc":
        return {"bytes": EMB * FC_K + case["batch"] * (FC_K + EMB * 4), "flops": 2.0 * case["batch"] * EMB * FC_K}
    n = case["pixels"] * case["channels"]
    return {"bytes": n * (2 if kind == "bn" else 3), "flops": 0}


def tolerance(case):
    """Integer sums are exact and every later operation is one specified
    rounding: all results are the same bits."""
    return "exact"


# ---------------------------------------------------------------- 64-bit results

def _half_away(t):
    return torch.sign(t) * torch.floor(t.abs() + 0.5)


def _i8(t):
    return t.clamp(-128, 127)


def _acc64(x, w, stride, pad):
    """Integer sums of a convolution of NHWC integers with OIHW weights, in
    float64 (exact), as [pixels, cout]."""
    n, h, _, cin = x.shape
    cout, _, k, _ = w.shape
    ho = (h + 2 * pad - k) // stride + 1
    wm = w.to(DEV).permute(2, 3, 1, 0).reshape(-1, cout).double()
    out = torch.empty((n, ho * ho, cout), dtype=torch.float64, device=DEV)
    step = max(1, int(2e8 // (ho * ho * k * k * cin)))
    for i in range(0, n, step):
        xp = torch.nn.functional.pad(x[i:i + step].double(), (0, 0, pad, pad, pad, pad))
        span = (ho - 1) * stride + 1
        cols = torch.cat([xp[:, r:r + span:stride, s:s + span:stride] for r in range(k) for s in range(k)], dim=-1)
        out[i:i + step] = (cols.reshape(-1, cols.shape[-1]) @ wm).reshape(-1, ho * ho, cout)
    return out.reshape(n, ho, ho, cout)


def _bn64(x, s_in, scale, offset, inv):
    return _i8(_half_away((x * s_in * scale + offset) * inv))


def _exact_conv(case, seed):
    x, w, P, add = _conv_inputs(case, seed)
    P = P.double()
    outs = ([], [])
    step = max(1, int(3e8 // (_out_hw(case) ** 2 * case["cout"])))
    for i in range(0, case["batch"], step):
        f = _acc64(x[i:i + step], w, case["stride"], case["pad"]) * P[fa.FFK_P_WS] + P[fa.FFK_P_BIAS]
        if add is not None:
            f = f + add[i:i + step].double() * P[fa.FFK_P_ADDSCALE]
        if case["epi"].startswith("prelu"):
            f = torch.where(f < 0, f * P[fa.FFK_P_SLOPE], f)
        q = _i8(_half_away(f * P[fa.FFK_P_INV]))
        outs[0].append(q.to(torch.int8))
        if case["epi"].endswith("bn"):
            outs[1].append(_bn64(q, P[fa.FFK_P_BN_SIN], P[fa.FFK_P_BN_S], P[fa.FFK_P_BN_O],
                                 P[fa.FFK_P_BN_INV]).to(torch.int8))
    return [torch.cat(o) for o in outs if o]


def _read_model():
    """The model file's ops: conv / GEMM weights with their scales and
    biases, BN and PReLU rows."""
    with open(synth.synthetic_ffw4_path(MODEL_SEED), "rb") as f:
        d = f.read()
    pos = 8

    def arr(dtype, n):
        nonlocal pos
        a = np.frombuffer(d, dtype, n, pos)
        pos += a.nbytes
        return torch.from_numpy(a.copy()).to(DEV)

    ops = []
    for _ in range(struct.unpack_from("<I", d, 4)[0]):
        op = {"type": d[pos]}
        pos += 1
        if op["type"] == synth.OP_CONV:
            cin, cout, kh, kw, op["s"], op["p"] = struct.unpack_from("<6H", d, pos)
            pos += 12
            op["w"] = arr(np.int8, cout * cin * kh * kw).reshape(cout, cin, kh, kw)
            op["ws"], op["bias"] = arr(np.float32, cout).double(), arr(np.float32, cout).double()
        elif op["type"] in (synth.OP_BN, synth.OP_PRELU):
            n = struct.unpack_from("<H", d, pos)[0]
            pos += 2
            op["a"] = arr(np.float32, n).double()
            if op["type"] == synth.OP_BN:
                op["b"] = arr(np.float32, n).double()
        elif op["type"] == synth.OP_GEMM:
            n, k = struct.unpack_from("<II", d, pos)
            pos += 8
            op["w"] = arr(np.int8, n * k).reshape(n, k)
            op["ws"], op["bias"] = arr(np.float32, n).double(), arr(np.float32, n).double()
        ops.append(op)
    return ops


def _read_scales():
    """(input scales, per-op output scales or None) of the per-channel scale file."""
    with open(os.path.join(ROOT, "models", "op_scales_v2.bin"), "rb") as f:
        d = f.read()
    n_ops, n_in = struct.unpack_from("<II", d, 5)
    pos = 13
    rows = []
    for n in [n_in] + [None] * n_ops:
        if n is None:
            n = struct.unpack_from("<I", d, pos)[0]
            pos += 4
        rows.append(torch.from_numpy(np.frombuffer(d, np.float32, n, pos).copy()).to(DEV).double() if n else None)
        pos += 4 * n
    return rows[0], rows[1:]


def _forward64(x, ops, in_scale, scales):
    """The int8 network in float64 on fp32 faces [B, 112, 112, 3]."""
    inv = lambda s: 1.0 / (s + 1e-9)
    A = _i8(torch.round(x.double() * inv(in_scale)))
    cur = in_scale
    saved = block = None
    i = 0
    while i < len(ops):
        op = ops[i]
        t = op["type"]
        if t == synth.OP_CONV:
            shortcut = ops[i - 1]["type"] == synth.OP_SAVE_ID and i > 0
            f = _acc64(block if shortcut else A, op["w"], op["s"], op["p"]) * op["ws"] + op["bias"]
            nxt = ops[i + 1]["type"]
            if nxt == synth.OP_PRELU:
                f = torch.where(f < 0, f * ops[i + 1]["a"], f)
            elif nxt == synth.OP_ADD:
                f = f + saved[0] * saved[1]
            if nxt in (synth.OP_PRELU, synth.OP_ADD):
                i += 1
            A = _i8(_half_away(f * inv(scales[i])))
            cur = scales[i]
        elif t == synth.OP_BN:
            A = _bn64(A, cur, op["a"], op["b"], inv(scales[i]))
            cur = scales[i]
        elif t == synth.OP_BLOCK_START:
            block = A
        elif t == synth.OP_SAVE_ID:
            saved = (A, cur)
        elif t == synth.OP_FLATTEN:
            A = A.permute(0, 3, 1, 2).reshape(A.shape[0], -1)
        elif t == synth.OP_GEMM:
            A = (A @ op["w"].double().t()) * op["ws"] + op["bias"]
        i += 1
    return A


def _exact_embed(case, seed):
    ops = _read_model()
    in_scale, scales = _read_scales()
    x = _faces(case, seed)
    if x.dtype == torch.uint8:
        x = (x.double() - 127.5) / 127.5
    out = torch.cat([_forward64(x[i:i + 64], ops, in_scale, scales) for i in range(0, case["batch"], 64)])
    if case["source"].startswith("host"):
        out = out.cpu().numpy()
        return out[0] if case["batch"] == 1 and case["source"] == "host_f32" else out
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "embed":
        return _exact_embed(case, seed)
    if kind == "conv":
        return _exact_conv(case, seed)
    if kind == "fc":
        a, w, ws, bias = _fc_inputs(case, seed)
        return (a.double() @ w.double().t()) * ws.double() + bias.double()
    if kind == "bn":
        x, rows = _bn_inputs(case, seed)
        r = rows.double()
        step = max(1, (1 << 27) // case["channels"])
        return torch.cat([_bn64(x[i:i + step].double(), *r).to(torch.int8) for i in range(0, case["pixels"], step)])
    a, b = _add_inputs(case, seed)
    sa, sb, so = _ADD_SCALES
    step = max(1, (1 << 27) // case["channels"])
    return torch.cat([_i8(torch.round((a[i:i + step].double() * sa + b[i:i + step].double() * sb) / (so + 1e-9)))
                      .to(torch.int8) for i in range(0, case["pixels"], step)])
