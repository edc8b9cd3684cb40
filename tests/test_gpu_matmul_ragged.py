"""GEMM outputs whose rows are not whole groups of eight columns, or do not start on a
16-byte boundary, through every tile shape of the pipelined and wide-tile kernels:
bit for bit against the oracle, and nothing written outside the [M, N] output.
"""
import numpy as np
import pytest
import torch

from dscquant_amd import _lib, w4a4
from oracle import native
from tests.test_gpu_matmul import _operands, _oracle_raw
from tests.test_gpu_wide import gemm_kernel

pytestmark = pytest.mark.gpu

GUARD = 40


def _call(o, M, N, KP, bias, raw, dtype, offset, gpu, ws=None):
    """dscq_matmul (with a workspace dscq_matmul_ws) into buffers with guards around,
    `offset` elements off alignment."""
    def guarded(dt):
        t = torch.full((M * N + 2 * GUARD,), 77, dtype=dt, device=gpu)
        return t, t[GUARD + offset:].data_ptr()

    out, pout = guarded(dtype)
    rawt, praw = guarded(torch.int32) if raw else (None, None)
    _lib.call("dscq_matmul" if ws is None else "dscq_matmul_ws", *(t.data_ptr() for t in o),
              _lib.ptr(bias), M, N, KP, 0 if raw else 1, 0, 1 if dtype == torch.float32 else 0,
              pout, praw, *(() if ws is None else (ws.data_ptr(), ws.numel())),
              _lib.stream(gpu))
    torch.cuda.synchronize()
    got = []
    for t in (out, rawt):
        if t is None:
            continue
        s = GUARD + offset
        assert bool((t[:s] == 77).all()) and bool((t[s + M * N:] == 77).all()), "write outside"
        got.append(t[s:s + M * N].view(M, N).cpu().numpy())
    return got


@pytest.mark.parametrize("M,N,K", [(17, 8064, 8512), (32, 4096, 16448), (33, 4096, 6144),
                                   (48, 4096, 11008), (63, 2056, 12352), (33, 4096, 512),
                                   (48, 4088, 4096)])
def test_mid_rows_match_oracle(gpu, M, N, K):
    """16 < M < 64 on both sides of the K split's line, with and without a workspace,
    and the skinny kernel's two- and three-tile grids."""
    ops = _operands(M, N, K, seed=M + N)
    o = [torch.from_numpy(v).to(gpu) for v in ops]
    a, b, sx, zx, sw, sums = ops
    raw_ref = _oracle_raw(a, b, M, N)
    for dtype in (np.float16, np.float32):
        print(f"mid rows M{M} N{N} K{K} {np.dtype(dtype).name}", flush=True)
        td = torch.float32 if dtype == np.float32 else torch.float16
        ref = native.restore(raw_ref, sx, zx, sw, sums, None, out_dtype=dtype)
        none = torch.empty(0, dtype=td, device=gpu)
        out, raw = w4a4.matmul(*o, none, M, N, False, False, td == torch.float32)
        np.testing.assert_array_equal(out.cpu().numpy(), ref)
        np.testing.assert_array_equal(raw.cpu().numpy(), raw_ref)
        got = _call(o, M, N, a.shape[1] * 2, None, False, td, 0, gpu)
        np.testing.assert_array_equal(got[0], ref)


# (M, N, K, gemm kernel): 64 x 128 tiles of eight and four waves, 128 x 128 of
# eight and four, 256 x 128, the wide kernel's two widths; N around a tile and a
# group of eight columns, K with and without a partial slice, the rows left alone
# in their tile, and the former rule's largest shapes.
CASES = [(64, 5001, 512, 2), (65, 8071, 320, 2), (100, 129, 4096, 2), (512, 11003, 320, 2),
         (130, 16385, 256, 2), (384, 8191, 576, 2), (1030, 4099, 512, 2), (300, 8002, 1088, 2),
         (2048, 4097, 256, 2), (40, 8067, 512, 0), (17, 8193, 4100, 0), (256, 257, 256, 3),
         (300, 1023, 512, 3), (70, 519, 768, 3), (300, 1023, 512, 4), (257, 129, 256, 4),
         (4096, 4093, 256, 0),
         # the wide kernel where rows end inside a slice (one to three quarters of
         # it, alone or after whole slices)
         (256, 256, 64, 3), (64, 300, 128, 3), (130, 261, 192, 3), (300, 520, 320, 3),
         (70, 519, 1088, 3), (1000, 1032, 4100, 3), (257, 264, 448, 4), (300, 515, 4032, 4),
         (4096, 4096, 320, 0)]


@pytest.mark.parametrize("M,N,K,kernel", CASES)
def test_ragged_outputs_match_oracle(gpu, M, N, K, kernel):
    ops = _operands(M, N, K, seed=M + 3 * N + K)
    a, b, sx, zx, sw, sums = ops
    o = [torch.from_numpy(v).to(gpu) for v in ops]
    raw_ref = _oracle_raw(a, b, M, N)
    rng = np.random.default_rng(N)
    for dtype, raw, use_bias, offset in ((np.float16, False, True, 0), (np.float16, False, False, 1),
                                         (np.float16, True, False, 0), (np.float32, False, True, 1),
                                         (np.float32, True, False, 0)):
        print(f"ragged M{M} N{N} K{K} kernel{kernel} {np.dtype(dtype).name} raw{raw} "
              f"bias{use_bias} offset{offset}", flush=True)
        bias = rng.standard_normal(N).astype(dtype) if use_bias else None
        tb = torch.from_numpy(bias).to(gpu) if use_bias else None
        with gemm_kernel(kernel):
            got = _call(o, M, N, a.shape[1] * 2, tb, raw, torch.from_numpy(np.zeros(1, dtype)).dtype,
                        offset, gpu)
        np.testing.assert_array_equal(got[0], native.restore(raw_ref, sx, zx, sw, sums, bias,
                                                             out_dtype=dtype))
        if raw:
            np.testing.assert_array_equal(got[1], raw_ref)


# fp32 rows of whole 64-byte pieces (stores past the caches), and those that miss the
# boundary by the output's address (GUARD + offset elements of 4 bytes), by N, and by N with
# a row end inside four columns; every tile shape of the pipelined kernel and the wide one.
@pytest.mark.parametrize("offset", [8, 0])
@pytest.mark.parametrize("M,N,K,kernel", [(300, 528, 320, 2), (300, 524, 320, 2), (300, 523, 320, 2),
                                          (700, 8208, 256, 2), (1030, 8196, 192, 2),
                                          (2050, 4112, 256, 2), (300, 528, 320, 3),
                                          (261, 524, 512, 3), (300, 523, 320, 3)])
def test_fp32_rows_on_and_off_cache_lines(gpu, M, N, K, kernel, offset):
    print(f"fp32 rows M{M} N{N} K{K} kernel{kernel} offset{offset}", flush=True)
    ops = _operands(M, N, K, seed=M + N)
    o = [torch.from_numpy(v).to(gpu) for v in ops]
    a, b, sx, zx, sw, sums = ops
    ref = native.restore(_oracle_raw(a, b, M, N), sx, zx, sw, sums, None, out_dtype=np.float32)
    with gemm_kernel(kernel):
        got = _call(o, M, N, a.shape[1] * 2, None, False, torch.float32, offset, gpu)
    np.testing.assert_array_equal(got[0], ref)


# Shapes that split K in a workspace but for N % 8 or the output's address (GUARD
# elements of 2 or 4 bytes put the first one off a 16-byte boundary): the second pass
# would take four columns across a row's end, or off its alignment.
@pytest.mark.parametrize("M,N,offset", [(128, 4100, 8), (48, 4100, 8), (128, 4096, 1),
                                        (48, 4096, 1), (128, 4096, 8), (48, 4096, 8)])
def test_outputs_that_do_not_split(gpu, M, N, offset):
    K = 11008
    splits = N % 8 == 0 and offset == 8
    ops = _operands(M, N, K, seed=M + N)
    a, b, sx, zx, sw, sums = ops
    o = [torch.from_numpy(v).to(gpu) for v in ops]
    raw_ref = _oracle_raw(a, b, M, N)
    ws = torch.full((4 * 8 * M * (N + 8),), 77, dtype=torch.uint8, device=gpu)
    for dtype, raw in ((np.float16, False), (np.float32, False), (np.float16, True)):
        print(f"workspace M{M} N{N} offset{offset} {np.dtype(dtype).name} raw{raw}", flush=True)
        bias = np.random.default_rng(M).standard_normal(N).astype(dtype)
        got = _call(o, M, N, a.shape[1] * 2, torch.from_numpy(bias).to(gpu), raw,
                    torch.from_numpy(np.zeros(1, dtype)).dtype, offset, gpu, ws)
        np.testing.assert_array_equal(got[0], native.restore(raw_ref, sx, zx, sw, sums, bias,
                                                             out_dtype=dtype))
        if raw:
            np.testing.assert_array_equal(got[1], raw_ref)
        assert bool((ws == 77).all()) != splits
        ws.fill_(77)
