"""The wide-tile GEMM's 192-row and 192-column tiles (chosen where they take fewer
rounds of 256 CUs): identical to the pipelined kernel, which the other tests hold
against the oracle, at ragged rows and columns, K that ends inside a slice, one slice,
and outputs off a 16-byte boundary; the gated form at outputs that end inside a tile.
"""
import pytest
import torch

from dscquant_amd import w4a4
from tests.test_gpu_wide import gemm_kernel

pytestmark = pytest.mark.gpu


def _operands(M, N, K, gpu, seed):
    g = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=gpu)
    w = torch.randn(N, K, generator=g, device=gpu)
    pa, sx, zx = w4a4.quantize(x, 1.0)
    pw, sw, sums = w4a4.pack_weight(w)
    return pa, pw, sx, zx, sw, sums


# 192 x 256: 700 x 16384, 2301 x 4099 (ragged), 1536 x 8192 (whole); 256 x 192: 1023 x
# 11003 (ragged), 1024 x 12288 (whole).
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M,N,K", [(700, 16384, 128), (2301, 4099, 200), (1536, 8192, 768),
                                   (1023, 11003, 330), (1024, 12288, 512)])
def test_tiles_equal_the_pipelined_kernel(gpu, M, N, K, bias):
    print(f"192 tiles M{M} N{N} K{K} bias{bias}", flush=True)
    ops = _operands(M, N, K, gpu, M + K)
    b = torch.randn(N if bias else 0, device=gpu).half()
    out = w4a4.matmul(*ops, b, M, N)[0]
    with gemm_kernel(2):
        assert torch.equal(out, w4a4.matmul(*ops, b, M, N)[0])


@pytest.mark.parametrize("M,N,K", [(700, 16384, 128), (2301, 4099, 200), (1023, 11003, 330)])
def test_bf16_layer(gpu, M, N, K):
    print(f"192 tiles bf16 M{M} N{N} K{K}", flush=True)
    _, pw, _, _, sw, sums = _operands(8, N, K, gpu, K)
    x = torch.randn(M, K, device=gpu).bfloat16()
    b = torch.randn(N, device=gpu)
    out = w4a4.linear(x, 0.9, 0, pw, sw, sums, b, N)
    with gemm_kernel(2):
        assert torch.equal(out, w4a4.linear(x, 0.9, 0, pw, sw, sums, b, N))


@pytest.mark.parametrize("M,N,K,bias", [(512, 11008, 128, True), (300, 11008, 200, False),
                                        (768, 11008, 320, True), (385, 10944, 64, False)])
def test_gated_tiles_equal_the_pipelined_kernel(gpu, M, N, K, bias):
    print(f"192 tiles gated M{M} N{N} K{K}", flush=True)
    pa, pw, sx, zx, sw, sums = _operands(M, 2 * N, K, gpu, N + K)
    b = torch.randn(2 * N if bias else 0, device=gpu).half()
    h = w4a4.matmul_silu_mul(pa, pw, sx, zx, sw, sums, b, M, N)
    with gemm_kernel(2):
        assert torch.equal(h, w4a4.matmul_silu_mul(pa, pw, sx, zx, sw, sums, b, M, N))


def test_bf16_block(gpu):
    M, K, N = 512, 256, 11008
    args = []
    for rows, cols, seed in ((2 * N, K, 1), (K, N, 2)):
        _, pw, _, _, sw, sums = _operands(8, rows, cols, gpu, seed)
        args.append((pw, sw, sums, torch.randn(rows, device=gpu)))
    x = torch.randn(M, K, device=gpu).bfloat16()
    run = lambda: w4a4.gated_mlp(x, 1.0, 0, *args[0], N, 1.0, 0, *args[1], K)
    out = run()
    with gemm_kernel(2):
        assert torch.equal(out, run())
