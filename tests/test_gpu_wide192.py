"""The wide-tile GEMM's 192-row and 192-column tiles (chosen where they take fewer
rounds of 256 CUs): identical to the pipelined kernel, which the other tests hold
against the oracle, at ragged rows and columns, K that ends inside a slice,
and outputs off a 16-byte boundary; the gated form at outputs that end inside a tile.
Every case states the tile, and the library is asked that its automatic choice takes it.
"""
import pytest
import torch

from dscquant_amd import _lib, w4a4
from tests.test_gpu_wide import gemm_kernel

pytestmark = pytest.mark.gpu

TILE = "w4a4_gemm_wide_kernel<%s>"


def _takes(tile, M, N, K, gated=0, dtype=0):
    name = _lib.lib().dscq_matmul_kernel(M, N, w4a4.padded(K, 64), gated, 0, dtype, None, None,
                                         None, 0).decode()
    assert name == TILE % tile, f"{name} for M{M} N{N} K{K}: the case tests another kernel"


def _operands(M, N, K, gpu, seed):
    g = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.randn(M, K, generator=g, device=gpu)
    w = torch.randn(N, K, generator=g, device=gpu)
    pa, sx, zx = w4a4.quantize(x, 1.0)
    pw, sw, sums = w4a4.pack_weight(w)
    return pa, pw, sx, zx, sw, sums


# Rows and columns that end a whole tile, one past it, inside it and one short; of the
# 192 columns also around the 96 of a wave; K of whole slices and with a quarter, a half
# and three quarters of one.
CASES = [("192x256", 700, 16384, 2048), ("192x256", 577, 16129, 2112),
         ("192x256", 767, 16383, 2176), ("192x256", 768, 16384, 2240),
         ("192x256", 2301, 4099, 2000), ("192x256", 1536, 8192, 2048),
         ("192x256", 1345, 8001, 6150),
         ("256x192", 1023, 11003, 2112), ("256x192", 1024, 12288, 2048),
         ("256x192", 961, 10945, 2176), ("256x192", 1024, 11040, 2240),
         ("256x192", 1000, 11041, 2112), ("256x192", 1024, 11135, 4100),
         ("256x192", 1023, 11001, 6150)]


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("tile,M,N,K", CASES)
def test_tiles_equal_the_pipelined_kernel(gpu, tile, M, N, K, bias):
    print(f"192 tiles {tile} M{M} N{N} K{K} bias{bias}", flush=True)
    _takes(tile, M, N, K)
    pa, pw, sx, zx, sw, sums = _operands(M, N, K, gpu, M + K)
    b = torch.randn(N if bias else 0, device=gpu).half()
    with gemm_kernel(2):
        ref = w4a4.matmul(pa, pw, sx, zx, sw, sums, b, M, N)[0]
    for offset in (0, 1):  # a guard around an output on and off a 16-byte boundary
        buf = torch.full((M * N + 80,), 77, dtype=torch.float16, device=gpu)
        _lib.call("dscq_matmul", pa.data_ptr(), pw.data_ptr(), sx.data_ptr(), zx.data_ptr(),
                  sw.data_ptr(), sums.data_ptr(), _lib.ptr(b), M, N, w4a4.padded(K, 64), 1, 0, 0,
                  buf[40 + offset:].data_ptr(), None, _lib.stream(gpu))
        s = 40 + offset
        assert torch.equal(buf[s:s + M * N].view(M, N), ref)
        assert bool((buf[:s] == 77).all()) and bool((buf[s + M * N:] == 77).all())


@pytest.mark.parametrize("tile,M,N,K", [("192x256", 700, 16384, 2048), ("192x256", 2301, 4099, 2000),
                                        ("256x192", 1023, 11003, 2112)])
def test_bf16_layer(gpu, tile, M, N, K):
    print(f"192 tiles bf16 {tile} M{M} N{N} K{K}", flush=True)
    _takes(tile, M, N, K, dtype=2)
    _, pw, _, _, sw, sums = _operands(8, N, K, gpu, K)
    x = torch.randn(M, K, device=gpu).bfloat16()
    b = torch.randn(N, device=gpu)
    out = w4a4.linear(x, 0.9, 0, pw, sw, sums, b, N)
    with gemm_kernel(2):
        assert torch.equal(out, w4a4.linear(x, 0.9, 0, pw, sw, sums, b, N))


# 96 outputs a tile: the last one whole, two thirds and one third full; rows one past a tile.
@pytest.mark.parametrize("M,N,K,bias", [(512, 11008, 2048, True), (300, 11008, 2112, False),
                                        (257, 11072, 2176, True), (385, 10944, 2240, False),
                                        (768, 11008, 3200, True), (511, 11072, 6144, False)])
def test_gated_tiles_equal_the_pipelined_kernel(gpu, M, N, K, bias):
    print(f"192 tiles gated M{M} N{N} K{K}", flush=True)
    _takes("256x192", M, N, K, gated=1)
    pa, pw, sx, zx, sw, sums = _operands(M, 2 * N, K, gpu, N + K)
    b = torch.randn(2 * N if bias else 0, device=gpu).half()
    h = w4a4.matmul_silu_mul(pa, pw, sx, zx, sw, sums, b, M, N)
    with gemm_kernel(2):
        assert torch.equal(h, w4a4.matmul_silu_mul(pa, pw, sx, zx, sw, sums, b, M, N))


def test_bf16_block(gpu):
    M, K, N = 512, 2112, 11008
    _takes("256x192", M, N, K, gated=1, dtype=2)
    args = []
    for rows, cols, seed in ((2 * N, K, 1), (K, N, 2)):
        _, pw, _, _, sw, sums = _operands(8, rows, cols, gpu, seed)
        args.append((pw, sw, sums, torch.randn(rows, device=gpu)))
    x = torch.randn(M, K, device=gpu).bfloat16()
    run = lambda: w4a4.gated_mlp(x, 1.0, 0, *args[0], N, 1.0, 0, *args[1], K)
    out = run()
    with gemm_kernel(2):
        assert torch.equal(out, run())
