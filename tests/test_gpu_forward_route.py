"""QuantLinear and QuantMLP forwards, each one call of the library, against the calls
they stand for (quantize, matmul, matmul_silu_mul), bit for bit: the sizes where the
kernel behind them changes, input rows off a 16-byte boundary, and sources that change
between two calls.
"""
import pytest
import torch
from torch import nn

from dscquant_amd import w4a4
from dscquant_amd.core.linear import QuantLinear, _mark, _unchanged
from dscquant_amd.core.mlp import QuantMLP


class _Cfg:
    weight_bits = activation_bits = 4


def _layer(N, K, seed, device, dtype=torch.float16, bias=True, rot=0):
    g = torch.Generator().manual_seed(seed)
    lin = nn.Linear(K, N, bias=bias)
    with torch.no_grad():
        for p in lin.parameters():
            p.copy_(torch.randn(p.shape, generator=g) * 0.05)
    q = QuantLinear(lin.to(dtype).to(device), _Cfg())
    q.enabled, q.rotate_block = True, rot
    return q


def _rows(M, K, dtype, device, offset):
    store = torch.zeros(M * K + offset, dtype=dtype, device=device)
    x = store[offset:].view(M, K)
    x.copy_(torch.randn(M, K, generator=torch.Generator().manual_seed(M + K)))
    return x


def _two_calls(q, x):
    pw, sw, sums = q.packed_weight()
    fp32 = x.dtype == torch.float32
    pa, sx, zx = w4a4.quantize(x.clone(), 1.0, True, q.rotate_block)
    return w4a4.matmul(pa, pw, sx, zx, sw, sums, q.packed_bias(x.dtype), x.shape[0],
                       q.base.weight.shape[0], True, False, fp32)[0]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,K,N,rot", [(1, 1024, 520, 128), (4, 1024, 520, 0), (3, 1030, 77, 0),
                                       (9, 4096, 256, 128), (40, 1024, 4096, 0),
                                       (257, 1100, 515, 0)])
def test_linear_equals_its_two_calls(gpu, M, K, N, rot, dtype):
    q = _layer(N, K, 1, gpu, dtype, rot=rot)
    with torch.no_grad():
        for offset in (0, 1, 3):
            x = _rows(M, K, dtype, gpu, offset)
            assert torch.equal(q(x), _two_calls(q, x)), (M, K, N, offset)


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,K,N", [(1, 256, 128), (7, 256, 192), (17, 512, 1024), (130, 320, 448)])
def test_fp16_block_equals_its_four_calls(gpu, M, K, N, bias):
    mlp = QuantMLP(_layer(N, K, 1, gpu, bias=bias), _layer(N, K, 2, gpu, bias=bias and M != 7),
                   _layer(K, N, 3, gpu, bias=bias, rot=128 if N % 128 == 0 else 0))
    with torch.no_grad():
        pgu, swgu, sgu, bgu, _, _, _ = mlp.packed()
        assert (bgu is None) == (not bias)
        none = torch.empty(0, dtype=torch.float16, device=gpu)
        for offset in (0, 1):
            x = _rows(M, K, torch.float16, gpu, offset)
            pa, sx, zx = w4a4.quantize(x.clone(), 1.0)
            h = w4a4.matmul_silu_mul(pa, pgu, sx, zx, swgu, sgu, none if bgu is None else bgu, M, N)
            assert torch.equal(mlp(x), _two_calls(mlp.down, h)), (M, K, N, offset)
        before = mlp(x)
        mlp.up.base.weight.mul_(1.5)        # seen by its version
        mlp.down.base.weight.data = mlp.down.base.weight.data * 2  # and by its storage
        pgu, swgu, sgu, bgu, _, _, _ = mlp.packed()
        h = w4a4.matmul_silu_mul(pa, pgu, sx, zx, swgu, sgu, none if bgu is None else bgu, M, N)
        after = mlp(x)
        assert torch.equal(after, _two_calls(mlp.down, h)) and not torch.equal(after, before)


def test_marks_see_every_change():
    t = nn.Parameter(torch.ones(4), requires_grad=False)
    mark = _mark(t)
    assert _unchanged(mark, t) and _unchanged(_mark(None), None)
    assert not _unchanged(mark, None) and not _unchanged(None, t)
    assert not _unchanged(mark, nn.Parameter(torch.ones(4)))
    t.add_(1)
    assert not _unchanged(mark, t)
    mark = _mark(t)
    t.data = t.data.clone()
    assert not _unchanged(mark, t)
    mark = _mark(t)
    t.data = t.data.view(torch.int32)
    assert not _unchanged(mark, t)
