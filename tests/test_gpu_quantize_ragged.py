"""Rows that end inside a chunk of eight elements, or start at an odd address, through
every row kernel (few rows, one to four waves a row, one row per workgroup,
streaming, rows below a chunk): bit for bit against the oracle.
"""
import numpy as np
import pytest
import torch

from dscquant_amd import w4a4
from oracle import native
from tests.conftest import activations, weights

pytestmark = pytest.mark.gpu


def _at(x, gpu, offset):
    """x on the GPU, `offset` elements into its storage (which ends with it)."""
    store = torch.zeros(x.size + offset, dtype=torch.from_numpy(x).dtype, device=gpu)
    t = store[offset:].view(*x.shape)
    t.copy_(torch.from_numpy(x))
    return t


# (M, K): the few-row kernel in 1-3 passes, the register kernel's waves-per-row x
# blocks shapes above 512 rows, one row per workgroup (2048+ rows), streaming, and
# K around one chunk.
SHAPES = [(3, 1), (2, 7), (5, 8), (3, 9), (7, 15), (16, 1001), (9, 4097), (4, 9003), (2, 12287),
          (513, 129), (520, 2047), (515, 2051), (700, 8190), (514, 8193), (600, 16381),
          (2050, 4090), (2049, 2053), (3, 32765), (2, 32770), (2, 40001)]


@pytest.mark.parametrize("M,K", SHAPES)
@pytest.mark.parametrize("dtype", [np.float16, np.float32])
def test_quantize_ragged_rows(gpu, M, K, dtype):
    x = activations(M, K, seed=M + K, dtype=dtype)
    for offset, clip in ((0, 1.0), (1, 0.8)):
        print(f"quantize ragged M{M} K{K} {np.dtype(dtype).name} offset{offset}", flush=True)
        p, s, z = w4a4.quantize(_at(x, gpu, offset), clip, True)
        p_ref, s_ref, z_ref = native.quantize_rows(x.astype(np.float32), clip, 0)
        np.testing.assert_array_equal(s.cpu().numpy(), s_ref)
        np.testing.assert_array_equal(z.cpu().numpy(), z_ref)
        np.testing.assert_array_equal(p.cpu().numpy(), p_ref)


@pytest.mark.parametrize("M,K,offset", [(5, 512, 1), (5, 4096, 3), (600, 2048, 1), (2048, 4096, 5),
                                        (3, 11008, 7), (530, 33024, 1)])
def test_rotated_rows_at_odd_addresses(gpu, M, K, offset):
    x = activations(M, K, seed=K)
    print(f"quantize rotated M{M} K{K} offset{offset}", flush=True)
    p, s, z = w4a4.quantize(_at(x, gpu, offset), 1.0, True, 128)
    p_ref, s_ref, z_ref = native.quantize_rows(x.astype(np.float32), 1.0, 128)
    np.testing.assert_array_equal(s.cpu().numpy(), s_ref)
    np.testing.assert_array_equal(p.cpu().numpy(), p_ref)


@pytest.mark.parametrize("N,K", [(5, 3), (9, 9), (13, 1003), (10, 2049), (7, 8191), (3, 20005),
                                 (2, 32771)])
def test_pack_weight_ragged_rows(gpu, N, K):
    w = weights(N, K, seed=N + K)
    for offset in (0, 1):
        print(f"pack_weight ragged N{N} K{K} offset{offset}", flush=True)
        p, sw, sums = w4a4.pack_weight(_at(w, gpu, offset), 0.9, 0)
        p_ref, sw_ref, sums_ref = native.pack_weight(w.astype(np.float32), 0.9, 0)
        np.testing.assert_array_equal(sw.cpu().numpy(), sw_ref)
        np.testing.assert_array_equal(sums.cpu().numpy(), sums_ref)
        np.testing.assert_array_equal(p.cpu().numpy(), p_ref)
