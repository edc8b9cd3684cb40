"""The SiLU-gated block in bf16 (dscq_gated_mlp): equal to the three modules and
torch's silu and product in bf16, through the skinny, pipelined and wide gated
kernels; the fp16 form equal to the four calls; and the cases that keep the
composition (hooks, shapes, other N).
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F
from torch import nn

from dscquant_amd import _lib, w4a4
from dscquant_amd.core.linear import QuantLinear
from dscquant_amd.core.mlp import QuantMLP
from tests.conftest import activations, weights
from tests.test_gpu_wide import gemm_kernel

pytestmark = pytest.mark.gpu


class Cfg:
    weight_bits = activation_bits = 4


def _module(N, K, seed, gpu, bias, dtype, rot=0, scale=1.0):
    base = nn.Linear(K, N, bias=bias, device=gpu, dtype=dtype)
    with torch.no_grad():
        base.weight.copy_(torch.from_numpy(weights(N, K, seed=seed, dtype=np.float32)) * scale)
        if bias:
            base.bias.copy_(torch.randn(N, generator=torch.Generator().manual_seed(seed)))
    m = QuantLinear(base, Cfg())
    m.enabled, m.rotate_block = True, rot
    return m


def _mlp(K, N, gpu, bias=False, dtype=torch.bfloat16, scale=1.0):
    return QuantMLP(_module(N, K, 1, gpu, bias, dtype, scale=scale),
                    _module(N, K, 2, gpu, bias, dtype),
                    _module(K, N, 3, gpu, bias, dtype, rot=128 if N % 128 == 0 else 0))


# (M, K, N, bias, gemm kernel): skinny (one and several row groups), 64- / 128- / 256-
# row pipelined tiles, wide tiles forced, K that ends inside a slice.
CASES = [(1, 512, 128, False, 0), (16, 1024, 704, True, 0), (33, 768, 1088, False, 0),
         (40, 512, 8192, True, 0), (64, 320, 256, True, 0), (130, 512, 1024, False, 0),
         (512, 1024, 2816, True, 2), (700, 1000, 1024, False, 2), (300, 512, 1024, True, 3),
         (257, 1088, 192, False, 3)]


@pytest.mark.parametrize("M,K,N,bias,kernel", CASES)
def test_bf16_block_equals_its_modules(gpu, monkeypatch, M, K, N, bias, kernel):
    print(f"mlp bf16 M{M} K{K} N{N} bias{bias} kernel{kernel}", flush=True)
    calls = []
    real = w4a4.gated_mlp
    monkeypatch.setattr(w4a4, "gated_mlp", lambda *a: calls.append(1) or real(*a))
    mlp = _mlp(K, N, gpu, bias)
    x = torch.from_numpy(activations(M, K, seed=M, dtype=np.float32)).to(gpu).bfloat16()
    with torch.no_grad(), gemm_kernel(kernel):
        y = mlp(x)
        ref = mlp.down(F.silu(mlp.gate(x)) * mlp.up(x))
    # h equals torch's to the last bit save where torch's exp differs in its last place
    # across a bf16 tie (none seen); one such code would move outputs of that row.
    assert len(calls) == 1 and y.dtype == torch.bfloat16 and torch.equal(y, ref)


def test_silu_over_the_whole_bf16_range(gpu):
    """h for every finite bf16 gate value, through a layer that passes it on: one input
    channel at code 15 and a weight of one code make g = scale * bias-free; the gate
    comes from the bias instead, so g is exactly the bias."""
    vals = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    vals = vals[torch.isfinite(vals.float())]
    N = (vals.numel() + 63) // 64 * 64
    gate = torch.zeros(N, dtype=torch.float32)
    gate[:vals.numel()] = vals.float()
    up = torch.where(torch.arange(N) % 3 == 0, 1.0, 0.7265625)
    K = 64
    zero = w4a4.pack_weight(torch.zeros(2 * N, K, device=gpu))
    bias = w4a4.interleave_gate_up(gate, up).to(gpu)
    # The down projection's quantization would hide h: take the gated GEMM alone.
    need = _lib.lib().dscq_gated_mlp_workspace_bytes(1, K, N, 8)
    ws = torch.zeros(need, dtype=torch.uint8, device=gpu)
    down = w4a4.pack_weight(torch.zeros(8, N, device=gpu))
    y = torch.empty(1, 8, dtype=torch.bfloat16, device=gpu)
    x = torch.zeros(1, K, dtype=torch.bfloat16, device=gpu)
    _lib.call("dscq_gated_mlp", x.data_ptr(), 2, 1, K, 1.0, 0, zero[0].data_ptr(),
              zero[1].data_ptr(), zero[2].data_ptr(), bias.data_ptr(), N, 1.0, 0,
              down[0].data_ptr(), down[1].data_ptr(), down[2].data_ptr(), None, 8, y.data_ptr(),
              ws.data_ptr(), need, _lib.stream(gpu))
    torch.cuda.synchronize()
    # h sits behind the quantized input: packed [8, K / 2], scales and zero points.
    at = 3 * 256
    h = ws[at:at + 2 * N].view(torch.bfloat16)
    g = gate.to(gpu).bfloat16()
    ref = F.silu(g) * up.to(gpu).bfloat16()
    same = (h == ref) | (torch.isnan(h.float()) & torch.isnan(ref.float()))
    assert bool(same.all()), (g[~same][:8], h[~same][:8], ref[~same][:8])


def test_fp16_call_equals_the_four(gpu):
    for M, K, N in ((5, 512, 192), (48, 1024, 704), (600, 512, 1024)):
        mlp = _mlp(K, N, gpu, True, torch.float16)
        x = torch.from_numpy(activations(M, K, seed=M)).to(gpu)
        with torch.no_grad():
            ref = mlp(x)
            pgu, swgu, sgu, bgu, pd, swd, sd = mlp.packed()
            rot = int(mlp.down.rotate_block)
            y = w4a4.gated_mlp(x, 1.0, 0, pgu, swgu, sgu, bgu, N, 1.0, rot, pd, swd, sd,
                               mlp.down.packed_bias(torch.float16), K)
        assert torch.equal(y, ref)


# Rows quantized inside the products: each form of the gated kernel (v_dot8 up to two
# rows, MFMA beyond; one and two passes of 32 blocks, quads), K that ends inside a block,
# the last shape that fits and the first that does not (rows, K past 4096), and a down
# projection that fits or not.
FEW = [(1, 64, 64), (1, 4096, 192), (2, 4096, 704), (2, 1000, 1088), (3, 1344, 128),
       (4, 2048, 11008), (4, 4096, 4096), (5, 4096, 128), (8, 2048, 256), (9, 512, 128),
       (1, 4104, 256), (1, 1024, 12288), (1, 1024, 12352)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", FEW)
def test_few_rows_equal_the_separate_launches(gpu, dtype, M, K, N):
    """One call against quantize, gated GEMM, quantize, GEMM (fp16) or the modules (bf16),
    finite rows and rows with an infinity or a NaN, off a 16-byte boundary as well."""
    print(f"few rows M{M} K{K} N{N} {dtype}", flush=True)
    mlp = _mlp(K, N, gpu, True, dtype)
    if K % 128 == 0:
        mlp.gate.rotate_block = mlp.up.rotate_block = 128
    rot_in, rot = int(mlp.gate.rotate_block), int(mlp.down.rotate_block)
    base = torch.from_numpy(activations(M, K, seed=M + K, dtype=np.float32)).to(gpu).to(dtype)
    bad = base.clone()
    bad[0, 3], bad[-1, K - 1] = float("inf"), float("nan")
    off = torch.empty(M * K + 1, dtype=dtype, device=gpu)[1:].view(M, K).copy_(base)
    with torch.no_grad():
        for x in (base, off, bad):
            y = mlp(x)
            if dtype == torch.float16:
                pgu, swgu, sgu, bgu, pd, swd, sd = mlp.packed()
                pa, sx, zx = w4a4.quantize(x.contiguous(), 1.0, True, rot_in)
                h = w4a4.matmul_silu_mul(pa, pgu, sx, zx, swgu, sgu, bgu, M, N)
                ph, sh, zh = w4a4.quantize(h, 1.0, True, rot)
                ref = w4a4.matmul(ph, pd, sh, zh, swd, sd, mlp.down.packed_bias(dtype), M, K,
                                  True, False, False)[0]
            else:
                ref = mlp.down(F.silu(mlp.gate(x)) * mlp.up(x))
            assert torch.equal(y.isnan(), ref.isnan())
            assert torch.equal(y.nan_to_num(), ref.nan_to_num())


def test_what_keeps_the_composition(gpu, monkeypatch):
    monkeypatch.setattr(w4a4, "gated_mlp", lambda *a: pytest.fail("one call"))
    x = torch.from_numpy(activations(6, 512, seed=2, dtype=np.float32)).to(gpu).bfloat16()
    with torch.no_grad():
        mlp = _mlp(512, 1000, gpu)          # N % 64 != 0
        assert torch.equal(mlp(x), mlp.down(F.silu(mlp.gate(x)) * mlp.up(x)))
        mlp = _mlp(512, 1024, gpu)
        seen = []
        hook = mlp.up.register_forward_hook(lambda m, a, o: seen.append(o))
        mlp(x)
        assert len(seen) == 1
        hook.remove()
        with pytest.raises(RuntimeError, match="mat1 and mat2"):
            mlp(x[:, :500].contiguous())
    monkeypatch.undo()
    with torch.no_grad():
        assert mlp(x[:0]).shape == (0, 512) and mlp(x.view(2, 3, 512)).shape == (2, 3, 512)
