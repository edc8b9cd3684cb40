"""QuantMLP's one-call block on the host: which modules it stands for, and under
torch.inference_mode, where a module's packed tensors carry no version counter.  The
library calls are replaced by recorders, so no GPU is needed.
"""
import pytest
import torch
import torch.nn.functional as F
from torch import nn

from dscquant_amd import w4a4
from dscquant_amd.core.linear import QuantLinear
from dscquant_amd.core.mlp import QuantMLP

K, N = 64, 128


class _W4A4:
    weight_bits = activation_bits = 4


def _quant(rows, cols, bias=False):
    base = nn.Linear(cols, rows, bias=bias)
    lin = QuantLinear(base, _W4A4())
    lin.enabled = True
    return lin


@pytest.fixture
def packs(monkeypatch):
    """pack_weight by plain torch, gated_mlp and linear as recorders."""
    seen = {"pack": 0, "block": [], "linear": 0}

    def pack(w, clip=1.0, rotate=0, return_codes=False):
        seen["pack"] += 1
        n, kb = w4a4.padded(w.shape[0], 8), w4a4.padded(w.shape[1], 64) // 2
        return [torch.zeros(n, kb, dtype=torch.uint8) + seen["pack"], torch.ones(n),
                torch.zeros(n, dtype=torch.int32)]

    def block(x, clip, rot, b_gu, sw_gu, sums_gu, bias_gu, n, *rest):
        seen["block"].append((b_gu, bias_gu))
        return x.new_zeros(x.shape[0], rest[-1])

    def linear(x, clip, rot, b, sw, sums, bias, n):
        seen["linear"] += 1
        return x.new_zeros(x.shape[0], n)

    monkeypatch.setattr(w4a4, "pack_weight", pack)
    monkeypatch.setattr(w4a4, "gated_mlp", block)
    monkeypatch.setattr(w4a4, "linear", linear)
    monkeypatch.setattr(w4a4, "linear_decode_supported", lambda m, k: False)
    return seen


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_block_under_inference_mode(packs, dtype):
    """First call, repeated calls, a changed weight, and back outside the mode."""
    mlp = QuantMLP(_quant(N, K, True), _quant(N, K), _quant(K, N))
    x = torch.randn(3, K).to(dtype)
    with torch.inference_mode():
        assert mlp(x).shape == (3, K)
        mlp(x)
    assert packs["pack"] == 3 and len(packs["block"]) == 2
    assert packs["block"][1][0] is packs["block"][0][0]   # packed and joined once
    assert packs["block"][1][1] is packs["block"][0][1]
    with torch.no_grad():
        mlp(x)
        assert packs["pack"] == 3 and packs["block"][2][0] is packs["block"][0][0]
        mlp.up.base.weight.mul_(2)
    with torch.inference_mode():
        mlp(x)
    assert packs["pack"] == 4 and packs["block"][3][0] is not packs["block"][0][0]


class _Scaled(nn.Module):
    """A wrapper without the attributes of a QuantLinear."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, x):
        return self.inner(x) * 2


class _Other(QuantLinear):
    def _forward_w4a4(self, x):
        return super()._forward_w4a4(x) + 1


@pytest.mark.parametrize("which", ["gate", "up", "down"])
@pytest.mark.parametrize("kind", ["linear", "wrapper", "subclass", "instance"])
def test_other_modules_keep_the_composition(packs, which, kind):
    """bf16 inputs ran the composition with any three modules before the block took
    them; it stands for QuantLinear's own forward only."""
    mods = {"gate": _quant(N, K), "up": _quant(N, K), "down": _quant(K, N)}
    shape = (K, N) if which == "down" else (N, K)
    if kind == "linear":
        mods[which] = nn.Linear(shape[1], shape[0]).bfloat16()
    elif kind == "wrapper":
        mods[which] = _Scaled(mods[which])
    elif kind == "subclass":
        mods[which] = _Other(mods[which].base, _W4A4())
        mods[which].enabled = True
    else:
        plain = mods[which]._forward_w4a4
        mods[which]._forward_w4a4 = lambda t: plain(t) + 1
    mlp = QuantMLP(**mods)
    x = torch.randn(3, K).bfloat16()
    with torch.no_grad():
        y = mlp(x)
        assert not packs["block"] and packs["linear"] == (2 if kind == "linear" else 3)
        assert torch.equal(y, mlp.down(F.silu(mlp.gate(x)) * mlp.up(x)))
