"""Float codes and fake quantization (dscq_float_codes, dscq_fake_quant) against
the oracle, bit for bit: every row length where the kernel changes its shape
(one wave or four per row, 1 to 8 chunks per lane, rows walked twice, a last chunk
of 1 to 8 elements, rows below a chunk), rows at element alignment, the three
element types, and values on exact ties.
"""
import numpy as np
import pytest
import torch

from dscquant_amd.core import quantization as Q
from oracle import native

pytestmark = pytest.mark.gpu

LENGTHS = [1, 7, 8, 9, 511, 512, 513, 1024, 1031, 2048, 2049, 4095, 4104, 8192, 8201, 16384,
           16385, 20483]
TYPES = [torch.float16, torch.bfloat16, torch.float32]


def _rows(M, K, dtype, gpu, seed, offset):
    """[M, K] with outliers and a tie row, starting `offset` elements into its storage."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g)
    x[:, torch.randint(K, (max(1, K // 64),), generator=g)] *= 40
    # Row 0 on the grid of half steps: quotients at exact ties for several widths.
    x[0] = torch.randint(-30, 31, (K,), generator=g) * 0.5
    if M > 2:
        x[2] = 0
    store = torch.zeros(M * K + offset, dtype=dtype, device=gpu)
    rows = store[offset:].view(M, K)
    rows.copy_(x.to(dtype))
    return rows, rows.float().cpu().numpy()


@pytest.mark.parametrize("dtype", TYPES, ids=["fp16", "bf16", "fp32"])
@pytest.mark.parametrize("K", LENGTHS)
def test_rows_match_oracle(gpu, K, dtype):
    for M, bits, clip, offset in ((5, 8, 1.0, 0), (4, 4, 0.75, 1), (1, 3, 1.0, 3), (3, 2, 0.9, 0)):
        print(f"fake quant M{M} K{K} {dtype} bits{bits} clip{clip} offset{offset}", flush=True)
        x, ref = _rows(M, K, dtype, gpu, K + bits, offset)
        c_ref, s_ref, z_ref = native.activation_codes(ref, bits, clip)
        code, scale, zero = Q.activation_codes(x, bits, clip)
        np.testing.assert_array_equal(code.cpu().numpy(), c_ref.astype(np.float32))
        np.testing.assert_array_equal(scale.cpu().numpy()[:, 0], s_ref)
        np.testing.assert_array_equal(zero.cpu().numpy()[:, 0], z_ref)
        deq = (c_ref.astype(np.float32) - z_ref[:, None]) * s_ref[:, None]
        assert torch.equal(Q.quantize_activation(x, bits, clip).cpu(),
                           torch.from_numpy(deq).to(dtype))
        wc_ref, ws_ref = native.weight_codes(ref, bits, clip)
        code, scale = Q.weight_codes(x, bits, clip)
        np.testing.assert_array_equal(code.cpu().numpy(), wc_ref.astype(np.float32))
        np.testing.assert_array_equal(scale.cpu().numpy()[:, 0], ws_ref)
        deq = wc_ref.astype(np.float32) * ws_ref[:, None]
        assert torch.equal(Q.quantize_weight(x, bits, clip).cpu(), torch.from_numpy(deq).to(dtype))


def test_scales_outside_the_reciprocals_range(gpu):
    """fp32 rows whose scale has no normal reciprocal, and rows at the scale floor."""
    w = torch.randn(6, 300, generator=torch.Generator().manual_seed(1))
    w = w * torch.tensor([1e38, 4e37, 1e-12, 1e-30, 0.0, 1.0])[:, None]
    for bits in (2, 4, 8):
        c_ref, s_ref = native.weight_codes(w.numpy(), bits, 1.0)
        code, scale = Q.weight_codes(w.to(gpu), bits)
        np.testing.assert_array_equal(code.cpu().numpy(), c_ref.astype(np.float32))
        np.testing.assert_array_equal(scale.cpu().numpy()[:, 0], s_ref)


def test_shapes_and_other_dtypes(gpu):
    x = torch.randn(2, 3, 40, generator=torch.Generator().manual_seed(2)).to(gpu)
    for t in (x, x.double(), x.transpose(0, 1), x[..., ::2]):
        y = Q.quantize_activation(t, 8)
        assert y.shape == t.shape and y.dtype == t.dtype
        rows = t.float().reshape(-1, t.shape[-1]).cpu().numpy()
        c, s, z = native.activation_codes(rows, 8, 1.0)
        ref = (c.astype(np.float32) - z[:, None]) * s[:, None]
        np.testing.assert_array_equal(y.float().cpu().numpy().reshape(rows.shape), ref)
    assert Q.quantize_activation(x[:0], 8).shape == (0, 3, 40)
    with pytest.raises(RuntimeError, match="bits must be"):
        Q.quantize_weight(x[0], 9)
    with pytest.raises(RuntimeError, match="clip"):
        Q.quantize_activation(x, 8, 1.5)


def test_more_rows_than_one_grid_holds(gpu):
    """Past 2^26 rows of up to 2048 elements a grid would have 2^32 threads."""
    M, K = (1 << 26) + 5, 3
    x = torch.randn(1 << 20, K, generator=torch.Generator().manual_seed(3)).to(gpu).half()
    x = torch.cat([x.repeat(64, 1), x[:5] * 3])
    assert x.shape[0] == M
    code, scale, zero = Q.activation_codes(x, 4)
    y = Q.quantize_activation(x, 4)
    for r in (0, (1 << 25) - 2, M - 1000):  # the first rows, a launch's last and first, the end
        part = x[r:r + 1000]
        c, s, z = Q.activation_codes(part, 4)
        assert torch.equal(code[r:r + 1000], c) and torch.equal(scale[r:r + 1000], s)
        assert torch.equal(zero[r:r + 1000], z)
        assert torch.equal(y[r:r + 1000], Q.quantize_activation(part, 4))
    assert torch.equal(y[:1 << 20], y[1 << 25:(1 << 25) + (1 << 20)])  # whole launches alike
