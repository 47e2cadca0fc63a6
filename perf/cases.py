"""The work that users of this runtime have it do, as cases that can be timed.

A compiled int8 model makes one C call per quantized op on tensors that stay in
GPU memory; :class:`om_mi355x.PreparedCall` is that call, so most cases bind
their calls once and a pass makes them.  Model weights are declared constant, as
a compiled model declares them.  One kind of case (``host``) hands host arrays
to the Python entry point instead, the way a program without GPU memory of its
own uses the runtime.

Kinds of cases and the ranges they stand for
  layer      one dynamically quantized linear layer, f32 in, f32 out:
             1 .. 4096 rows, K and N from 256 to 11008
  encoder    the four projections of a transformer encoder layer (QKV, output,
             feed-forward up with Gelu, feed-forward down) with biases:
             16 .. 4096 tokens, hidden sizes 256 .. 1024
  integer    MatMulInteger with weights, int32 results, both zero points
  qlinear    QLinearMatMul with weights, 8-bit results
  attention  MatMulInteger of two activations, batched over heads: scores
             (Q times K transposed) or context (probabilities times V)
  qdq        QuantizeLinear, then DequantizeLinear of its result: per tensor,
             per channel on the last axis or on an inner one
  dynamic    DynamicQuantizeLinear of one tensor
  host       a dynamically quantized layer on host arrays
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "onnx-mlir_amd"))
import om_mi355x as om  # noqa: E402

# The largest listed matrix product and the largest listed tensor: what a drawn
# case may cost at most.
MAX_MACS = 2048 * 4096 * 11008
MAX_ELEMENTS = 8192 * 32768


def listed():
    return [
        # A 7B-sized model generating text: one token, and sixteen sequences at
        # once, through a feed-forward layer.  Bound by reading the weights.
        {"name": "decode_1_up", "kind": "layer", "M": 1, "K": 4096, "N": 11008, "act": 0, "bias": False},
        {"name": "decode_16_down", "kind": "layer", "M": 16, "K": 11008, "N": 4096, "act": 0, "bias": False},
        # The same model reading a prompt of 2048 tokens.
        {"name": "prefill_up", "kind": "layer", "M": 2048, "K": 4096, "N": 11008, "act": 0, "bias": False},
        {"name": "prefill_down", "kind": "layer", "M": 2048, "K": 11008, "N": 4096, "act": 0, "bias": False},
        # BERT-base at batch 32 x sequence 128: the projections of one encoder layer.
        {"name": "encoder_4096", "kind": "encoder", "M": 4096, "hidden": 768, "inner": 3072},
        # One sentence of 128 tokens through a hidden-sized layer: a single
        # launch of a few microseconds.
        {"name": "layer_128", "kind": "layer", "M": 128, "K": 768, "N": 768, "act": 0, "bias": False},
        # Static quantization, uint8 weights with a zero point, uint8 results.
        {"name": "qlinear_512", "kind": "qlinear", "M": 512, "K": 1024, "N": 4096, "b_unsigned": True, "saturate": False},
        # A product none of whose sizes is a multiple of anything.
        {"name": "integer_ragged", "kind": "integer", "M": 4099, "K": 777, "N": 1001, "b_unsigned": True, "per_column": True},
        # Attention scores of that BERT layer: 32 sentences x 12 heads of 64.
        {"name": "attention_scores", "kind": "attention", "batch": 32, "heads": 12, "M": 128, "K": 64, "N": 128},
        # A large activation tensor with a scale per channel.
        {"name": "qdq_per_channel", "kind": "qdq", "shape": "8192x32768", "axis": 1, "signed": False},
        # A large activation tensor quantized by its own range.
        {"name": "dynamic_large", "kind": "dynamic", "shape": "8192x32768"},
        # The feed-forward layer of one BERT sentence on host arrays.
        {"name": "host_layer", "kind": "host", "M": 128, "K": 768, "N": 3072},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo=256, hi=11008):
    """A layer width: mostly a multiple of 64 as models have them, sometimes of
    16, sometimes any number."""
    n, r = _log(rng, lo, hi), rng.random()
    step = 64 if r < 0.6 else 16 if r < 0.75 else 1
    return max(lo, n // step * step)


def _fit(rng, lo=1, hi=4096):
    while True:
        M, K, N = _log(rng, lo, hi), _width(rng), _width(rng)
        if M * K * N <= MAX_MACS:
            return M, K, N


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "encoder", "integer", "integer", "qlinear", "attention",
                       "qdq", "qdq", "dynamic", "host"])
    if kind == "layer":
        M, K, N = _fit(rng)
        return {"kind": kind, "M": M, "K": K, "N": N, "act": rng.choice([0, 0, 1, 2]), "bias": rng.random() < 0.5}
    if kind == "encoder":
        hidden = rng.choice([256, 384, 512, 768, 1024])
        return {"kind": kind, "M": _log(rng, 16, 4096), "hidden": hidden, "inner": 4 * hidden}
    if kind == "integer":
        M, K, N = _fit(rng)
        return {"kind": kind, "M": M, "K": K, "N": N, "b_unsigned": rng.random() < 0.5, "per_column": rng.random() < 0.5}
    if kind == "qlinear":
        M, K, N = _fit(rng)
        return {"kind": kind, "M": M, "K": K, "N": N, "b_unsigned": rng.random() < 0.5, "saturate": rng.random() < 0.5}
    if kind == "attention":
        while True:
            seq, dim = _log(rng, 8, 512), rng.choice([32, 64, 64, 80, 128])
            c = {"kind": kind, "batch": _log(rng, 1, 64), "heads": rng.choice([4, 8, 12, 16]), "M": seq}
            c["K"], c["N"] = (dim, seq) if rng.random() < 0.5 else (seq, dim)
            n = c["batch"] * c["heads"]
            if n * seq * seq * dim <= MAX_MACS // 16 and n * seq * max(seq, dim) <= MAX_ELEMENTS // 4:
                return c
    if kind == "qdq":
        n, form = _log(rng, 1 << 14, MAX_ELEMENTS), rng.choice(["tensor", "last", "last", "inner"])
        signed = rng.random() < 0.5
        if form == "inner":
            h = rng.choice([7, 14, 28, 56, 57])
            c = rng.choice([64, 256, 512])
            return {"kind": kind, "shape": "%dx%dx%dx%d" % (max(1, n // (c * h * h)), c, h, h), "axis": 1, "signed": signed}
        cols = _width(rng, 64, 32768)
        return {"kind": kind, "shape": "%dx%d" % (max(1, n // cols), cols), "axis": 1 if form == "last" else -1, "signed": signed}
    if kind == "dynamic":
        cols = _width(rng, 64, 32768)
        return {"kind": kind, "shape": "%dx%d" % (max(1, _log(rng, 1 << 12, MAX_ELEMENTS) // cols), cols)}
    return {"kind": kind, "M": _log(rng, 1, 512), "K": rng.choice([256, 512, 768, 1024]), "N": _width(rng, 256, 4096)}


class _Window:
    """GPU memory of the runtime as torch sees it; keeps the array alive."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": array.dtype.str,
                                         "data": (array.ptr, False), "strides": None, "version": 2}


class State:
    """What a program keeps: the tensors, the bound calls, the declared constants."""

    def __init__(self, seed):
        self.rng = torch.Generator(device="cuda").manual_seed(seed)
        self.calls, self.constants, self.outputs, self.program = [], [], [], None

    # -- tensors in the runtime's GPU memory
    def put(self, values):
        array = om.DeviceArray(tuple(values.shape), str(values.dtype).split(".")[1])
        torch.as_tensor(_Window(array), device="cuda").copy_(values)
        return array

    def empty(self, shape, dtype):
        """An output: the array, and the tensor that a pass returns for it."""
        array = om.DeviceArray(shape, dtype)
        self.outputs.append(torch.as_tensor(_Window(array), device="cuda"))
        return array

    def normal(self, shape, sigma=1.0):
        return self.put(torch.randn(shape, device="cuda", generator=self.rng).mul_(sigma))

    def uniform(self, shape, lo, hi):
        return self.put(torch.rand(shape, device="cuda", generator=self.rng).mul_(hi - lo).add_(lo))

    def whole(self, shape, lo, hi, dtype):
        return self.put(torch.randint(lo, hi + 1, shape, device="cuda", generator=self.rng, dtype=dtype))

    def scalar(self, value, dtype):
        return self.put(torch.tensor(value, device="cuda", dtype=dtype))

    def constant(self, array):
        om.mark_constant(array)
        self.constants.append(array)
        return array

    def call(self, entry, *operands):
        self.calls.append(om.PreparedCall(entry, *operands))

    def layer(self, x, M, K, N, act, bias):
        """A dynamically quantized linear layer; its result."""
        w = self.constant(self.whole((K, N), -127, 127, torch.int8))
        scale = self.constant(self.uniform((N,), 1e-3, 5e-3))
        b = self.constant(self.normal((N,), 0.1)) if bias else None
        y = self.empty((M, N), np.float32)
        self.call("om_mi355x_DynQuantMatMulDequant", y, x, w, None, scale, b, act)
        return y

    def __del__(self):
        for c in self.calls:
            c.close()
        for a in self.constants:
            om.unmark_constant(a)


def _shape(case):
    return tuple(int(n) for n in case["shape"].split("x"))


def prepare(case, seed):
    s, kind = State(seed), case["kind"]
    if kind == "layer":
        M, K, N = case["M"], case["K"], case["N"]
        s.layer(s.normal((M, K)), M, K, N, case["act"], case["bias"])
    elif kind == "encoder":
        M, H, F = case["M"], case["hidden"], case["inner"]
        s.layer(s.normal((M, H)), M, H, 3 * H, 0, True)
        s.layer(s.normal((M, H)), M, H, H, 0, True)
        up = s.layer(s.normal((M, H)), M, H, F, om.ACTIVATION_GELU, True)
        s.layer(up, M, F, H, 0, True)
    elif kind == "integer":
        M, K, N = case["M"], case["K"], case["N"]
        a = s.whole((M, K), 0, 255, torch.uint8)
        zps = (N,) if case["per_column"] else ()
        if case["b_unsigned"]:
            b, bz = s.whole((K, N), 0, 255, torch.uint8), s.whole(zps, 96, 160, torch.uint8)
        else:
            b, bz = s.whole((K, N), -127, 127, torch.int8), s.whole(zps, -8, 8, torch.int8)
        s.constant(b)
        s.constant(bz)
        s.call("om_mi355x_MatMulInteger", s.empty((M, N), np.int32), a, b, s.whole((), 96, 160, torch.uint8), bz)
    elif kind == "qlinear":
        M, K, N = case["M"], case["K"], case["N"]
        a = s.whole((M, K), 0, 255, torch.uint8)
        if case["b_unsigned"]:
            b, bz = s.whole((K, N), 0, 255, torch.uint8), s.scalar(120, torch.uint8)
        else:  # symmetric weights, the usual case
            b, bz = s.whole((K, N), -127, 127, torch.int8), s.scalar(0, torch.int8)
        # results spread over the 8-bit range: the products' deviation is about 74 * 74 * sqrt(K)
        y_scale = 74.0 * 74.0 * math.sqrt(K) * 0.01 * 0.005 / 50.0
        consts = [s.constant(c) for c in (b, bz, s.scalar(0.01, torch.float32), s.scalar(128, torch.uint8),
                                          s.scalar(0.005, torch.float32), s.scalar(y_scale, torch.float32),
                                          s.scalar(128, torch.uint8))]
        b, bz, a_s, a_z, b_s, y_s, y_z = consts
        s.call("om_mi355x_QLinearMatMul", s.empty((M, N), np.uint8), a, a_s, a_z, b, b_s, bz, y_s, y_z,
               om.SATURATE if case["saturate"] else om.WRAP)
    elif kind == "attention":
        lead, M, K, N = (case["batch"], case["heads"]), case["M"], case["K"], case["N"]
        a, b = s.whole(lead + (M, K), 0, 255, torch.uint8), s.whole(lead + (K, N), 0, 255, torch.uint8)
        s.call("om_mi355x_MatMulInteger", s.empty(lead + (M, N), np.int32), a, b,
               s.whole((), 96, 160, torch.uint8), s.whole((), 96, 160, torch.uint8))
    elif kind == "qdq":
        shape, axis = _shape(case), case["axis"]
        channels = () if axis < 0 else (shape[axis],)
        x = s.normal(shape, 2.0)
        scale = s.constant(s.uniform(channels, 0.005, 0.05))
        zp = s.constant(s.whole(channels, -128, 127, torch.int8) if case["signed"] else s.whole(channels, 0, 255, torch.uint8))
        q, d = s.empty(shape, zp.dtype), s.empty(shape, np.float32)
        s.call("om_mi355x_QuantizeLinear", q, x, scale, zp, max(axis, 0), 1)
        s.call("om_mi355x_DequantizeLinear", d, q, scale, zp, max(axis, 0))
    elif kind == "dynamic":
        shape = _shape(case)
        s.call("om_mi355x_DynamicQuantizeLinear", s.empty(shape, np.uint8), s.empty((), np.float32), s.empty((), np.uint8),
               s.normal(shape, 2.0))
    elif kind == "host":
        rng = np.random.default_rng(seed)
        M, K, N = case["M"], case["K"], case["N"]
        x = rng.standard_normal((M, K), dtype=np.float32)
        w = rng.integers(-127, 128, (K, N), dtype=np.int8)
        scale = rng.uniform(1e-3, 5e-3, N).astype(np.float32)
        y = np.empty((M, N), np.float32)
        s.constant(w)
        s.constant(scale)
        s.program = lambda: om.DynQuantMatMulDequant(x, w, None, scale, out=y)
    else:
        raise ValueError(kind)
    return s


def run(state):
    if state.program is not None:
        return state.program()
    for call in state.calls:
        call()
    return state.outputs


def _product(M, K, N, a_bytes, y_bytes, per_column=4):
    return {"bytes": M * K * a_bytes + K * N + per_column * N + M * N * y_bytes, "flops": 2.0 * M * K * N}


def work(case):
    kind = case["kind"]
    if kind in ("layer", "host"):
        return _product(case["M"], case["K"], case["N"], 4, 4)
    if kind == "encoder":
        M, H, F = case["M"], case["hidden"], case["inner"]
        parts = [_product(M, H, 3 * H, 4, 4, 8), _product(M, H, H, 4, 4, 8), _product(M, H, F, 4, 4, 8), _product(M, F, H, 4, 4, 8)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    if kind == "integer":
        return _product(case["M"], case["K"], case["N"], 1, 4, 1)
    if kind == "qlinear":
        return _product(case["M"], case["K"], case["N"], 1, 1, 0)
    if kind == "attention":
        n, M, K, N = case["batch"] * case["heads"], case["M"], case["K"], case["N"]
        return {"bytes": n * (M * K + K * N + 4 * M * N), "flops": 2.0 * n * M * K * N}
    n = math.prod(_shape(case))
    # f32 in, 8 bits out; then 8 bits in, f32 out
    return {"bytes": 10 * n if kind == "qdq" else 5 * n, "flops": 4.0 * n}


def tolerance(case):
    # Every op but Gelu is a fixed sequence of correctly rounded operations (the
    # products are sums of integers), so its result has only one value.  Gelu's
    # erf is an approximation: against the same layer in 64 bits the results are
    # off by 5e-8.  In the encoder the next layer quantizes Gelu's results again,
    # and an ulp in their largest moves the scale and with it some values to the
    # neighbouring 8-bit step: measured 4e-5, and 0.005 for a single value.
    if case["kind"] == "encoder":
        return {"rel": 2e-4, "max": 0.02}
    if case["kind"] == "layer" and case["act"] == 2:
        return {"rel": 2e-7, "max": 8e-6}
    return "exact"
