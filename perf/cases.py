"""Timing cases: what a program that uses this framework has it do.

A case is a dict of plain values; ``kind`` names the path:

  linear   ``QuantLinear.forward`` in W4A4 (the activations quantized, packed and
           multiplied with the packed weight);
  mlp      ``QuantMLP.forward``, the SiLU-gated block over three of them;
  fake     ``QuantLinear.forward`` at other bit widths (fake quantization around
           a dense product: how a model is evaluated at 8, 6 or 3 bits);
  pack     ``w4a4.pack_weight``: a checkpoint's weight made ready when it is loaded;
  export   ``weight_codes``, ``pack_int4`` and ``unpack_int4``: the packed form
           written to a file and read back.

``graph`` (a few tokens, as a decode loop calls the layer): the forward is
captured once in a HIP graph and a pass replays it; the others call the module.
Activations are N(0, 1) with 1% of the channels scaled by 50, weights N(0, 0.02).
"""
import math

import torch
from torch import nn

from dscquant_amd import w4a4
from dscquant_amd.core import quantization as q
from dscquant_amd.core.linear import QuantLinear
from dscquant_amd.core.mlp import QuantMLP

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


class _Bits:
    """The model configuration's part that the layers read."""

    def __init__(self, bits):
        self.weight_bits = self.activation_bits = bits


# ------------------------------------------------------------------ the cases

def _linear(M, K, N, dtype, rotate=128, bias=False, clip=1.0, graph=False):
    return {"kind": "linear", "M": M, "K": K, "N": N, "dtype": dtype, "rotate": rotate,
            "bias": bias, "clip": clip, "graph": graph}


def _mlp(M, K, N, dtype, rotate=128, graph=False):
    return {"kind": "mlp", "M": M, "K": K, "N": N, "dtype": dtype, "rotate": rotate,
            "graph": graph}


def _fake(M, K, N, dtype, bits):
    return {"kind": "fake", "M": M, "K": K, "N": N, "dtype": dtype, "bits": bits}


def _pack(N, K, dtype, rotate):
    return {"kind": "pack", "N": N, "K": K, "dtype": dtype, "rotate": rotate}


def _export(N, K, dtype):
    return {"kind": "export", "N": N, "K": K, "dtype": dtype}


def listed():
    return [
        # One generated token through one projection, called eagerly: the
        # smallest call, where launches and the host path count.
        dict(_linear(1, 4096, 4096, "fp16"), name="decode_linear"),
        # The MLP block of a 7B-shaped layer for four sequences, in the decode
        # loop's captured graph.
        dict(_mlp(4, 4096, 11008, "fp16", graph=True), name="decode_mlp_graph"),
        # Sixteen sequences through the up projection, captured likewise.
        dict(_linear(16, 4096, 11008, "fp16", graph=True), name="batch16_linear_graph"),
        # A model kept in bf16: a few dozen tokens (speculative decoding, a
        # short prompt) through the MLP block.
        dict(_mlp(48, 4096, 11008, "bf16"), name="small_mlp_bf16"),
        # A prompt of 2048 tokens through one attention projection.
        dict(_linear(2048, 4096, 4096, "fp16"), name="prefill_linear"),
        # 512 tokens through the MLP block.
        dict(_mlp(512, 4096, 11008, "fp16"), name="prefill_mlp"),
        # A prompt of no round length through a 70B-shaped projection with a
        # bias, in bf16.
        dict(_linear(3001, 8192, 8192, "bf16", bias=True), name="prefill_linear_bf16"),
        # The largest product: a 70B-shaped down projection of 4096 tokens.
        dict(_linear(4096, 28672, 8192, "fp16"), name="large_down"),
        # Odd sizes throughout (a pruned layer, an extended vocabulary), a bias
        # and a calibrated clip.
        dict(_linear(333, 4100, 10007, "fp16", rotate=0, bias=True, clip=0.9),
             name="ragged_linear"),
        # A weight packed at load time.
        dict(_pack(11008, 4096, "fp16", 128), name="pack_weight"),
        # The same weight in fp32, written to a file's packed form and read back.
        dict(_export(11008, 4096, "fp32"), name="export_codes"),
        # Evaluation at 8 bits: fake quantization of both operands on each call.
        dict(_fake(512, 4096, 4096, "bf16", 8), name="fake_quant_linear"),
    ]


def _size(rng, lo, hi, step=1):
    """A size spread evenly over its logarithm, a multiple of ``step``."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "mlp", "fake", "pack", "export"])
    if kind == "linear":
        M = _size(rng, 1, 4096)
        K = _size(rng, 1024, 11008, rng.choice([128, 128, 8, 1]))
        N = _size(rng, 1024, 16384, rng.choice([128, 8, 1]))
        return _linear(M, K, N, rng.choice(["fp16", "fp16", "bf16", "fp32"]),
                       rotate=rng.choice([0, 128]) if K % 128 == 0 else 0,
                       bias=rng.random() < 0.5, clip=rng.choice([1.0, 1.0, 0.9]),
                       graph=M <= 16 and rng.random() < 0.5)
    if kind == "mlp":
        M = _size(rng, 1, 2048)
        return _mlp(M, _size(rng, 1024, 8192, 128), _size(rng, 2048, 14336, 128),
                    rng.choice(["fp16", "fp16", "bf16"]), rotate=rng.choice([0, 128]),
                    graph=M <= 16 and rng.random() < 0.5)
    if kind == "fake":
        return _fake(_size(rng, 1, 4096), _size(rng, 1024, 8192, rng.choice([8, 1])),
                     _size(rng, 1024, 8192, rng.choice([8, 1])),
                     rng.choice(["fp16", "bf16"]), rng.choice([8, 6, 3]))
    N = _size(rng, 1024, 14336, rng.choice([8, 1]))
    K = _size(rng, 1024, 11008, rng.choice([128, 8, 1]))
    if kind == "pack":
        return _pack(N, K, rng.choice(["fp16", "bf16", "fp32"]),
                     rng.choice([0, 128]) if K % 128 == 0 else 0)
    return _export(N, K, rng.choice(["fp16", "fp32"]))


# ------------------------------------------------------------------ inputs

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed, n):
    return torch.Generator(device=_device()).manual_seed(1000 * seed + n)


def _activations(case, seed):
    g = _gen(seed, 0)
    x = torch.randn(case["M"], case["K"], generator=g, device=_device())
    top = torch.randperm(case["K"], generator=g, device=_device())[:max(1, case["K"] // 100)]
    x[:, top] *= 50
    return x.to(DTYPES[case["dtype"]])


def _weight(N, K, dtype, seed, n):
    w = torch.randn(N, K, generator=_gen(seed, n), device=_device()) * 0.02
    return w.to(DTYPES[dtype])


def _bias(N, dtype, seed):
    return torch.randn(N, generator=_gen(seed, 9), device=_device()).to(DTYPES[dtype])


def _layer(w, bias=None, bits=4, rotate=0, clip=1.0):
    base = nn.Linear(w.shape[1], w.shape[0], bias=bias is not None, device="meta")
    base.weight = nn.Parameter(w, requires_grad=False)
    if bias is not None:
        base.bias = nn.Parameter(bias, requires_grad=False)
    lin = QuantLinear(base, _Bits(bits))
    lin.enabled, lin.rotate_block = True, rotate
    with torch.no_grad():
        lin.activation_clip.fill_(clip)
    return lin


def _mlp_weights(case, seed):
    N, K, d = case["N"], case["K"], case["dtype"]
    return _weight(N, K, d, seed, 1), _weight(N, K, d, seed, 2), _weight(K, N, d, seed, 3)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("pack", "export"):
        return {"case": case, "w": _weight(case["N"], case["K"], case["dtype"], seed, 1)}
    x = _activations(case, seed)
    if kind == "mlp":
        gate, up, down = _mlp_weights(case, seed)
        # The rotation is the down projection's: its input has the outliers.
        module = QuantMLP(_layer(gate), _layer(up), _layer(down, rotate=case["rotate"]))
        module.packed()
    else:
        w = _weight(case["N"], case["K"], case["dtype"], seed, 1)
        b = _bias(case["N"], case["dtype"], seed) if case.get("bias") else None
        module = _layer(w, b, case.get("bits", 4), case.get("rotate", 0), case.get("clip", 1.0))
        if kind == "linear":
            module.packed_weight()
    state = {"case": case, "x": x, "module": module}
    if case.get("graph"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            module(x)
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = module(x)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "pack":
        return w4a4.pack_weight(state["w"], 1.0, case["rotate"])
    if case["kind"] == "export":
        codes, scale = q.weight_codes(state["w"], 4)
        packed = q.pack_int4(codes)
        return scale, packed, q.unpack_int4(packed, case["K"])
    if case.get("graph"):
        state["graph"].replay()
        return state["out"]
    return state["module"](state["x"])


# ------------------------------------------------------------------ what a pass needs

def _esize(case):
    return DTYPES[case["dtype"]].itemsize


def work(case):
    e, N, K = _esize(case), case["N"], case["K"]
    if case["kind"] == "pack":
        fwht = 7 * N * K if case["rotate"] else 0
        return {"bytes": N * K * e + N * K / 2 + 8 * N, "flops": fwht}
    if case["kind"] == "export":
        # The weight in; scales, packed nibbles and the codes read back out.
        return {"bytes": N * K * e + 4 * N + N * K / 2 + N * K, "flops": 0}
    M = case["M"]
    if case["kind"] == "mlp":
        return {"bytes": 2 * M * K * e + 3 * (N * K / 2) + 8 * (2 * N + K), "flops": 6 * M * N * K}
    if case["kind"] == "fake":
        return {"bytes": (M * K + N * K + M * N) * e, "flops": 2 * M * N * K}
    return {"bytes": (M * K + M * N) * e + N * K / 2 + 8 * N, "flops": 2 * M * N * K}


# About four times the largest error against exact() over the listed and ninety drawn
# cases: the output's rounding (fp16 2.1e-4, bf16 1.66e-3, fp32 4.4e-8), for an fp32
# rotation a code here and there that its rounding decides (1.3e-4), and in the MLP
# block the same for codes of the rounded SiLU (fp16 1.0e-3, bf16 5.3e-3).
def tolerance(case):
    if case["kind"] in ("pack", "export"):
        return "exact"
    if case["kind"] == "mlp":
        return {"rel": {"fp16": 4e-3, "bf16": 2e-2}[case["dtype"]]}
    if case["dtype"] == "fp32":
        return {"rel": 6e-4 if case["rotate"] else 1e-6}
    return {"rel": {"fp16": 9e-4, "bf16": 7e-3}[case["dtype"]]}


# ------------------------------------------------------------------ in 64 bits

def _hadamard(n=128):
    h = torch.ones(1, 1, dtype=torch.float64, device=_device())
    while h.shape[0] < n:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h


def _rotated(x, rotate, scale=1.0):
    x = x.double()
    if not rotate:
        return x
    return (x.reshape(-1, rotate) @ (_hadamard(rotate) * scale)).reshape(x.shape)


# Codes are whole numbers that the format defines by fp32 arithmetic (scale, quotient,
# sum, then round half to even); in 16-bit inputs exact ties are common, and only that
# arithmetic decides them. They are taken by it here, from values computed in 64 bits;
# everything after them stays in 64 bits.

def _over(t, number):
    # By a tensor: torch multiplies by a number's rounded reciprocal instead.
    return t / torch.full_like(t, number)


def _act(x, bits, clip):
    """(code - zero, scale) of a matrix's rows."""
    x, top = x.float(), 2 ** bits - 1
    lo = x.amin(1, keepdim=True).clamp(max=0) * clip
    hi = x.amax(1, keepdim=True).clamp(min=0) * clip
    scale = _over(hi - lo, top).clamp(min=1e-8)
    zero = (-lo / scale).round().clamp(0, top)
    return ((x / scale + zero).round().clamp(0, top) - zero).double(), scale.double()


def _wgt(w, bits):
    w, top = w.float(), 2 ** (bits - 1) - 1
    scale = _over(w.abs().amax(1, keepdim=True), top).clamp(min=1e-8)
    return (w / scale).round().clamp(-top, top).double(), scale.double()


def _product(x, w, rotate=0, clip=1.0, bias=None):
    cx, sx = _act(_rotated(x, rotate), 4, clip)
    cw, sw = _wgt(_rotated(w, rotate, 1 / 128), 4)
    y = (cx @ cw.t()) * sx * sw.t()
    return y if bias is None else y + bias.double()


def exact(case, seed):
    N, K, kind = case["N"], case["K"], case["kind"]
    if kind == "pack":
        # Packed bytes and code sums are whole numbers; the scales are computed.
        w = _rotated(_weight(N, K, case["dtype"], seed, 1), case["rotate"], 1 / 128)
        pad = torch.zeros(-N % 8, dtype=torch.float64, device=w.device)
        return [None, torch.cat([(w.abs().amax(1) / 7).clamp(min=1e-8), pad]), None]
    if kind == "export":
        w = _weight(N, K, case["dtype"], seed, 1).double()
        return (w.abs().amax(1, keepdim=True) / 7).clamp(min=1e-8), None, None
    dtype = DTYPES[case["dtype"]]
    x = _activations(case, seed)
    if kind == "mlp":
        # Between the projections the model's own dtype, as its modules hand
        # their results on.
        gate, up, down = _mlp_weights(case, seed)
        g, u = _product(x, gate).to(dtype).double(), _product(x, up).to(dtype).double()
        act = (g / (1 + torch.exp(-g))).to(dtype).double()
        return _product((act * u).to(dtype), down, case["rotate"])
    w = _weight(N, K, case["dtype"], seed, 1)
    if kind == "fake":
        cx, sx = _act(x.double(), case["bits"], 1.0)
        cw, sw = _wgt(w.double(), case["bits"])
        # Both fake-quantized operands are of the model's dtype.
        return (cx * sx).to(dtype).double() @ (cw * sw).to(dtype).double().t()
    b = _bias(N, case["dtype"], seed) if case["bias"] else None
    return _product(x, w, case["rotate"], case["clip"], b)
