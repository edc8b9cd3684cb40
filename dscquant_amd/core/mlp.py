"""SiLU-gated MLP block on the W4A4 path: down(act_fn(gate(x)) * up(x)).

The reference quantizes each projection of a Llama MLP through its own
QuantLinear (core/linear.py:48-52; core/model_ops.py drives the model) and
runs the activation in between unquantized in torch.  ``QuantMLP`` keeps the
three QuantLinear modules (their weights, clips, folds and rotations) and
runs the block in up to four launches:

    quantize(x)                                  -> packed x        (HIP)
    matmul_silu_mul(packed x, gate/up weights)   -> h [M, N]        (HIP)
    quantize(h)                                  -> packed h        (HIP)
    matmul(packed h, down weights)               -> out             (HIP)

gate and up read the same quantized x, so they run as one GEMM against the
packed weights interleaved in 64-row blocks, whose epilogue computes
h = fp16(fp16(silu(g)) * u) (an fp16 model's roundings) from the two halves
of each output tile.  When N is not a multiple of 64 the gate|up GEMM writes
[M, 2N] against the row-concatenated weights instead, and one kernel applies
the SiLU, the product and the down projection's input quantization
(silu_mul_quantize); both give the same h and the same packed h.  The
block computes h with an fp16 model's roundings for fp16 inputs and with a bf16
model's for bf16 ones (N a multiple of 64); with the gated GEMM its launches are one
call of the library, in x's dtype, and for a few tokens fewer of them (a product then
quantizes its rows itself); other inputs run the composition through the three
modules (each on the integer path), as the reference would.
"""
from __future__ import annotations

import torch
from torch import nn

from .. import w4a4
from .linear import QuantLinear

_MAX_ROWS = 65528


def _state(*tensors):
    """What tells that a module's packed tensors were written in place since, or None for
    ones made under torch.inference_mode: those carry no version, and their module hands
    out new ones when its sources change."""
    if any(t.is_inference() for t in tensors):
        return None
    return [v for t in tensors for v in (t._version, t.data_ptr())]


_CALLED = ("__call__", "forward", "_forward_w4a4")


def _plain(m) -> bool:
    """Whether calling ``m`` is QuantLinear's own forward and nothing more."""
    t, own = type(m), m.__dict__
    return ((t is QuantLinear
             or (issubclass(t, QuantLinear)
                 and all(getattr(t, n) is getattr(QuantLinear, n) for n in _CALLED)))
            and not (own["_forward_hooks"] or own["_forward_pre_hooks"]
                     or "forward" in own or "_forward_w4a4" in own))


class QuantMLP(nn.Module):
    """Fused W4A4 form of ``down(silu(gate(x)) * up(x))`` over three QuantLinear."""

    def __init__(self, gate: QuantLinear, up: QuantLinear, down: QuantLinear):
        super().__init__()
        self.gate, self.up, self.down = gate, up, down
        self._packed = None  # (the modules' packed weights, their state, gated, gate|up and down)
        self._gu_bias = {}   # dtype -> (gate's and up's bias, their state, gated, gate|up bias, has one)

    def _fusable(self, x) -> bool:
        """The fused block computes h with the roundings of an fp16 or (gated GEMM only)
        a bf16 model; other dtypes run the three modules in turn."""
        gate, up, down = self.gate, self.up, self.down
        return ((x.dtype == torch.float16
                 or (x.dtype == torch.bfloat16 and self._one_call(x.shape[-1])))
                and gate.enabled and up.enabled and down.enabled
                and gate._is_w4a4() and up._is_w4a4() and down._is_w4a4()
                and gate.rotate_block == up.rotate_block
                and gate.clip_value("activation_clip") == up.clip_value("activation_clip")
                and gate.base.weight.shape[0] % 8 == 0)

    def _one_call(self, K: int) -> bool:
        """Whether the block can stand for its three modules in one call: the shapes fit
        together and the gated GEMM, and calling the modules would do nothing more
        (QuantLinear's own forward, no hooks)."""
        return (_plain(self.gate) and _plain(self.up) and _plain(self.down)
                and self._fits_one_call(K)
                and not nn.modules.module._has_any_global_hook())

    def _fits_one_call(self, K: int) -> bool:
        """Whether the shapes fit together and the gated GEMM (``w4a4.gated_mlp``)."""
        shape = self.gate.base.weight.shape
        N = shape[0]
        return (N % 64 == 0 and shape[1] == K and self.up.base.weight.shape == shape
                and self.down.base.weight.shape[1] == N
                and K <= 65536 and N * w4a4.padded(K, 64) < 1 << 32)

    def packed(self, dtype=torch.float16):
        """(gate|up packed, sw, sums, gate|up bias in ``dtype`` or None, down packed, sw,
        sums).

        Built from the three modules' own packed weights and cached while those
        are the same objects (each module re-packs when its weight, fold, clip or
        rotation changes, and then hands out new tensors)."""
        pgu, swgu, sgu, pd, swd, sd = self._joined_weights()
        bias, some = self._joined_bias(dtype)
        return pgu, swgu, sgu, bias if some else None, pd, swd, sd

    def _joined_weights(self):
        parts = (self.gate.packed_weight(), self.up.packed_weight(), self.down.packed_weight())
        gated, hit = self._gated_gemm(), self._packed
        if (hit is None or hit[2] != gated or any(p is not q for p, q in zip(hit[0], parts))
                or (hit[1] is not None
                    and hit[1] != [v for p in parts for t in p for v in (t._version, t.data_ptr())])):
            (pg, swg, sg), (pu, swu, su), down = parts
            join = self._join
            hit = self._packed = (parts, _state(*(t for p in parts for t in p)), gated,
                                  (join(pg, pu), join(swg, swu), join(sg, su), *down))
        return hit[3]

    def _join(self, a, b):
        """gate and up rows interleaved in 64-row blocks for matmul_silu_mul, else
        concatenated for the [M, 2N] GEMM + silu_mul_quantize."""
        return w4a4.interleave_gate_up(a, b) if self._gated_gemm() else torch.cat([a, b])

    def _joined_bias(self, dtype):
        """(the gate|up bias in ``dtype`` and the weights' row order, whether there is one:
        empty if neither has)."""
        bg, bu = self.gate.packed_bias(dtype), self.up.packed_bias(dtype)
        gated, hit = self._gated_gemm(), self._gu_bias.get(dtype)
        if (hit is None or hit[0] is not bg or hit[1] is not bu or hit[3] != gated
                or (hit[2] is not None and hit[2] != [bg._version, bg.data_ptr(), bu._version,
                                                      bu.data_ptr()])):
            bias, some = bg, bool(bg.numel() or bu.numel())
            if some:
                N = self.gate.base.weight.shape[0]
                zero = torch.zeros(N, dtype=dtype, device=bg.device)
                bias = self._join(*(b if b.numel() else zero for b in (bg, bu)))
            hit = self._gu_bias[dtype] = (bg, bu, _state(bg, bu), gated, bias, some)
        return hit[4], hit[5]

    def _gated_gemm(self) -> bool:
        """Whether gate and up run as one GEMM with the SiLU-gated epilogue."""
        return self.gate.base.weight.shape[0] % 64 == 0

    def forward(self, x):
        if not self._fusable(x):
            from torch.nn import functional as F
            return self.down(F.silu(self.gate(x)) * self.up(x))
        if x.requires_grad and torch.is_grad_enabled():
            raise RuntimeError("the W4A4 HIP path is inference-only (codes carry no gradient)")
        bias_dtype = torch.float16 if x.dtype == torch.float16 else torch.float32
        gate, down = self.gate, self.down
        pgu, swgu, sgu, pd, swd, sd = self._joined_weights()
        bgu, _ = self._joined_bias(bias_dtype)
        N = gate.base.weight.shape[0]
        NO = down.base.weight.shape[0]
        K = x.shape[-1]
        lead = x.shape[:-1]
        xr = x.reshape(-1, K).contiguous()
        bdown = down.packed_bias(bias_dtype)
        aclip = gate.clip_value("activation_clip")
        dclip = down.clip_value("activation_clip")
        rot_in, rot_down = int(gate.rotate_block), int(down.rotate_block)
        M = xr.shape[0]
        one_call = x.dtype == torch.bfloat16 or self._fits_one_call(K)

        def block(part):
            if one_call:
                return w4a4.gated_mlp(part, aclip, rot_in, pgu, swgu, sgu, bgu, N, dclip, rot_down,
                                      pd, swd, sd, bdown, NO)
            m = part.shape[0]
            pa, sx, zx = w4a4.quantize(part, aclip, True, rot_in)
            if self._gated_gemm():
                h = w4a4.matmul_silu_mul(pa, pgu, sx, zx, swgu, sgu, bgu, m, N)
                ph, sh, zh = w4a4.quantize(h, dclip, True, rot_down)
            else:
                gu, _ = w4a4.matmul(pa, pgu, sx, zx, swgu, sgu, bgu, m, 2 * N, True, False, False)
                ph, sh, zh = w4a4.silu_mul_quantize(gu, dclip, rot_down)
            return w4a4.matmul(ph, pd, sh, zh, swd, sd, bdown, m, NO, True, False, False)[0]

        if 0 < M <= _MAX_ROWS:
            return block(xr).reshape(*lead, NO)
        out = torch.empty((M, NO), dtype=x.dtype, device=x.device)
        for r0 in range(0, M, _MAX_ROWS):
            out[r0:r0 + _MAX_ROWS] = block(xr[r0:r0 + _MAX_ROWS])
        return out.reshape(*lead, NO)
