"""w4a4.linear (dscq_linear): bf16 activations and results through every kernel that
reads or writes them, and the fp16 / fp32 forms, against the oracle's fp32 result
rounded once (small shapes) and against quantize + matmul in fp32 (the larger
ones, themselves held to the oracle elsewhere).  Bit for bit.
"""
import numpy as np
import pytest
import torch

from dscquant_amd import _lib, w4a4
from oracle import native
from tests.conftest import activations, weights
from tests.test_gpu_wide import gemm_kernel

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def _setup(M, K, N, rot, bias, gpu, dtype=BF16, offset=0):
    x = torch.from_numpy(activations(M, K, seed=M + K, dtype=np.float32)).to(dtype)
    store = torch.zeros(M * K + offset, dtype=dtype, device=gpu)
    xg = store[offset:].view(M, K)
    xg.copy_(x)
    w = torch.from_numpy(weights(N, K, seed=N, dtype=np.float32)).to(dtype).to(gpu)
    bd = torch.float16 if dtype == torch.float16 else torch.float32
    b = torch.randn(N, generator=torch.Generator().manual_seed(N)).to(bd).to(gpu) if bias else \
        torch.empty(0, dtype=bd, device=gpu)
    return xg, w, w4a4.pack_weight(w, 1.0, rot), b


# Fused decode: v_dot8 (1-2 rows; 4, 8, 12 pieces), MFMA (3-4 rows), the quad layout;
# skinny-M with one to three tiles; the tile shapes of the pipelined kernel, odd N,
# rows that end inside a chunk or a slice, rows at odd addresses, KP > 65536.
SMALL = [(1, 4096, 72, 128, True, 0), (2, 4096, 1000, 0, False, 0), (1, 11008, 40, 128, False, 0),
         (1, 8192, 33, 0, True, 1), (3, 4096, 130, 128, True, 0), (8, 1024, 64, 0, False, 3),
         (4, 4096, 4100, 128, False, 0), (7, 1000, 77, 0, True, 0), (16, 1031, 515, 0, True, 1),
         (33, 512, 9000, 128, False, 0), (40, 512, 8200, 128, True, 0), (65, 300, 1111, 0, True, 0),
         (128, 640, 2050, 128, False, 0), (320, 256, 4104, 0, True, 0), (513, 515, 1030, 0, False, 0),
         (64, 66000, 40, 0, True, 0), (2, 7, 24, 0, True, 0)]


@pytest.mark.parametrize("M,K,N,rot,bias,offset", SMALL)
def test_bf16_matches_oracle(gpu, M, K, N, rot, bias, offset):
    print(f"linear bf16 M{M} K{K} N{N} rot{rot} bias{bias} offset{offset}", flush=True)
    x, w, (pw, sw, sums), b = _setup(M, K, N, rot, bias, gpu, offset=offset)
    out = w4a4.linear(x, 1.0, rot, pw, sw, sums, b, N)
    ref, *_ = native.linear_w4a4(x.float().cpu().numpy(), w.float().cpu().numpy(),
                                 b.cpu().numpy() if bias else None, rotate_block=rot,
                                 out_dtype=np.float32)
    assert out.dtype == BF16 and torch.equal(out.cpu(), torch.from_numpy(ref).to(BF16))
    p_ref, sw_ref, sums_ref = native.pack_weight(w.float().cpu().numpy(), 1.0, rot)
    np.testing.assert_array_equal(pw.cpu().numpy(), p_ref)
    np.testing.assert_array_equal(sw.cpu().numpy(), sw_ref)
    np.testing.assert_array_equal(sums.cpu().numpy(), sums_ref)


LARGE = [(2048, 4096, 2048, 128, True, 0), (128, 11008, 4096, 0, True, 0),  # one row a wg; K split
         (2100, 2048, 4096, 0, False, 0), (600, 12288, 1024, 128, False, 0),
         (3001, 4096, 4096, 128, True, 0), (4096, 1024, 4100, 0, True, 0),
         (300, 4224, 1000, 128, True, 3), (700, 1088, 777, 0, True, 3)]      # wide, K tails


@pytest.mark.parametrize("M,K,N,rot,bias,kernel", LARGE)
@pytest.mark.parametrize("dtype", [torch.float16, BF16, torch.float32])
def test_linear_matches_quantize_and_matmul(gpu, M, K, N, rot, bias, kernel, dtype):
    print(f"linear {dtype} M{M} K{K} N{N} rot{rot} bias{bias} kernel{kernel}", flush=True)
    x, _, (pw, sw, sums), b = _setup(M, K, N, rot, bias, gpu, dtype)
    wide = dtype == BF16
    with gemm_kernel(kernel):
        out = w4a4.linear(x, 0.9, rot, pw, sw, sums, b, N)
    pa, sx, zx = w4a4.quantize(x.float() if wide else x, 0.9, True, rot)
    ref, _ = w4a4.matmul(pa, pw, sx, zx, sw, sums, b, M, N, True, False, dtype != torch.float16)
    assert out.dtype == dtype and torch.equal(out, ref.to(dtype))


def test_rejects_bad_arguments(gpu):
    x, _, (pw, sw, sums), b = _setup(16, 256, 64, 0, False, gpu)
    for bad in (lambda: w4a4.linear(x.double(), 1.0, 0, pw, sw, sums, b, 64),
                lambda: w4a4.linear(x[:, :128].contiguous(), 1.0, 0, pw, sw, sums, b, 64),
                lambda: w4a4.linear(x, 0.4, 0, pw, sw, sums, b, 64),
                lambda: w4a4.linear(x, 1.0, 0, pw, sw, sums, b.half().new_zeros(64), 64),
                lambda: w4a4.linear(x, 1.0, 0, pw, sw, sums, b, 65)):
        with pytest.raises(RuntimeError):
            bad()
    L = _lib.lib()
    need = L.dscq_linear_workspace_bytes(16, 256, 64)
    assert need > 0 and L.dscq_linear_workspace_bytes(1, 4096, 64) == 0
    out = torch.empty(16, 64, dtype=BF16, device=gpu)
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)
    for p, n in ((None, need), (ws.data_ptr(), need - 1), (ws.data_ptr() + 8, need)):
        assert L.dscq_linear(x.data_ptr(), 2, 16, 256, 1.0, 0, pw.data_ptr(), sw.data_ptr(),
                             sums.data_ptr(), None, 64, out.data_ptr(), p, n, None) == -1
    # The entry points that took fp16 and fp32 only still do.
    assert L.dscq_quantize(x.data_ptr(), 2, 16, 256, 1.0, 1, 0, ws.data_ptr(), ws.data_ptr(),
                           ws.data_ptr(), None, None) == -1
