"""pack_weight where its reciprocal form has to fall back to division: weights on
exact ties (before and after the rotation), scales without a normal reciprocal and
at the floor; bit for bit against the oracle, over the row shapes of the kernels.
"""
import numpy as np
import pytest
import torch

from dscquant_amd import w4a4
from oracle import native, numpy_ref

pytestmark = pytest.mark.gpu


def _check(w, dtype, rot, gpu):
    w = w.astype(dtype)
    got = w4a4.pack_weight(torch.from_numpy(w).to(gpu), 1.0, rot, return_codes=True)
    p, sw, sums = native.pack_weight(w.astype(np.float32), 1.0, rot)
    np.testing.assert_array_equal(got[1].cpu().numpy(), sw)
    np.testing.assert_array_equal(got[2].cpu().numpy(), sums)
    np.testing.assert_array_equal(got[0].cpu().numpy(), p)
    np.testing.assert_array_equal(got[3].cpu().numpy(), native.unpack_int4(p, 2 * p.shape[1]))


@pytest.mark.parametrize("K", [128, 2048, 2176, 4096, 8192, 11008, 33024])
@pytest.mark.parametrize("rot", [0, 128])
def test_ties(gpu, K, rot):
    """Quotients (j + 1/2): scale 1/8 from a maximum of 7/8; with the rotation the
    weights whose transform, over 128, is that grid."""
    print(f"pack_weight ties K{K} rot{rot}", flush=True)
    rng = np.random.default_rng(K)
    w = (rng.integers(-7, 7, size=(9, K)) + 0.5) / 8
    w[:, 5] = 0.875
    if rot:
        w = (w.reshape(9, K // 128, 128) @ numpy_ref.sylvester(128)).reshape(9, K)
        _check(w, np.float32, rot, gpu)   # whole sixteenths up to 2^7: exact in fp32
    else:
        _check(w, np.float16, rot, gpu)
        _check(w, np.float32, rot, gpu)


@pytest.mark.parametrize("rot", [0, 128])
def test_scale_limits(gpu, rot):
    w = np.random.default_rng(3).standard_normal((8, 512)).astype(np.float32)
    # Rows 0 and 1 past 2^118 in scale without the rotation, near its overflow with it.
    w *= np.float32([2e36 if rot else 2e37, 1e36, 1e-9, 1e-20, 1e-36, 0.0, 1.0, 6e-8])[:, None]
    _check(w, np.float32, rot, gpu)
