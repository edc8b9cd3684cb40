"""pack_int4 / unpack_int4 at the edges of the kernels' pieces of 16 codes: joined
rows (even width) and rows cut by themselves (odd width, or a width below the
packed one), the range check, fp32 codes, and views at odd addresses.
"""
import numpy as np
import pytest
import torch

from dscquant_amd import _lib
from dscquant_amd.core import quantization as Q
from oracle import native

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (3, 2), (1, 15), (2, 16), (5, 17), (7, 31), (4, 32), (3, 33), (9, 48), (1, 4096),
          (257, 1003), (130, 514)]


@pytest.mark.parametrize("R,C", SHAPES)
def test_pack_and_unpack_match_oracle(gpu, R, C):
    rng = np.random.default_rng(R * 1000 + C)
    c = rng.integers(-8, 8, size=(R, C)).astype(np.int8)
    ref = native.pack_int4(c)
    for dtype in (torch.int8, torch.float32, torch.int64, torch.bfloat16):
        for offset in (0, 1):
            print(f"codec R{R} C{C} {dtype} offset{offset}", flush=True)
            store = torch.zeros(R * C + offset, dtype=dtype, device=gpu)
            t = store[offset:].view(R, C)
            t.copy_(torch.from_numpy(c))
            np.testing.assert_array_equal(Q.pack_int4(t).cpu().numpy(), ref)
    store = torch.zeros(ref.size + 1, dtype=torch.uint8, device=gpu)
    for p in (torch.from_numpy(ref).to(gpu), store[1:].view(ref.shape)):
        p.copy_(torch.from_numpy(ref))
        for width in sorted({C, max(1, C - 1), max(1, C // 2), 1, 2 * ref.shape[1] + 4}):
            u = Q.unpack_int4(p, width)
            np.testing.assert_array_equal(
                u.cpu().numpy(), native.unpack_int4(ref, min(width, 2 * ref.shape[1])))


@pytest.mark.parametrize("C", [16, 33, 40])
@pytest.mark.parametrize("dtype", [torch.int8, torch.float32, torch.int32])
def test_one_code_out_of_range_raises(gpu, C, dtype):
    for where in (0, 15, C - 1, 3 * C - 1):
        for value in (8, -9, 100, -128, 127):
            c = torch.zeros(3, C, dtype=dtype, device=gpu)
            c.view(-1)[where] = value
            with pytest.raises(ValueError, match="Signed INT4 code out of range."):
                Q.pack_int4(c)


def test_fp32_codes_convert_as_to_int8_does(gpu):
    """Fractions truncate; values outside int8 do what .to(torch.int8) does with them."""
    base = torch.tensor([[0.9, -0.9, 7.99, -8.5, 3.0, -3.0, 1e-30, -0.0]] * 4, device=gpu)
    assert torch.equal(Q.pack_int4(base), Q.pack_int4(base.to(torch.int8)))
    for value in (256.0, 259.0, -300.0, 1e10, float("nan"), float("inf")):
        c = base.clone()
        c[1, 3] = value
        try:
            ref = Q.pack_int4(c.to(torch.int8))
        except ValueError:
            with pytest.raises(ValueError):
                Q.pack_int4(c)
        else:
            assert torch.equal(Q.pack_int4(c), ref)


def test_empty(gpu):
    assert Q.pack_int4(torch.zeros(0, 6, dtype=torch.int8, device=gpu)).shape == (0, 3)
    assert Q.pack_int4(torch.zeros(4, 0, device=gpu)).shape == (4, 0)
    assert Q.unpack_int4(torch.zeros(0, 3, dtype=torch.uint8, device=gpu), 6).shape == (0, 6)


@pytest.mark.parametrize("R", [1, 2, 37])
@pytest.mark.parametrize("C", list(range(1, 20)) + [31, 33, 47])
def test_nothing_written_outside_and_the_next_row_left_out(gpu, R, C):
    """Every remainder of a row's last piece: buffers with guards around, the next row's
    codes (and a code past the matrix) out of range, which a row's own must not see."""
    rng = np.random.default_rng(R * 100 + C)
    for f32 in (0, 1):
        c = rng.integers(-8, 8, size=(R, C)).astype(np.int8)
        ref = native.pack_int4(c)
        src = torch.full((R * C + 80,), 99, dtype=torch.float32 if f32 else torch.int8, device=gpu)
        src[40:40 + R * C] = torch.from_numpy(c.reshape(-1)).to(gpu)
        out = torch.full((ref.size + 80,), 77, dtype=torch.uint8, device=gpu)
        bad = torch.zeros(1, dtype=torch.int32, device=gpu)
        _lib.call("dscq_pack_int4_checked", src[40:].data_ptr(), f32, R, C, out[40:].data_ptr(),
                  bad.data_ptr(), _lib.stream(gpu))
        got = out.cpu().numpy()
        np.testing.assert_array_equal(got[40:40 + ref.size].reshape(ref.shape), ref)
        assert (got[:40] == 77).all() and (got[40 + ref.size:] == 77).all() and not bool(bad)
        for r in range(min(R, 3)):  # a row's last code out of range is seen
            src[40 + (r + 1) * C - 1] = 9
            bad.zero_()
            _lib.call("dscq_pack_int4_checked", src[40:].data_ptr(), f32, R, C, out[40:].data_ptr(),
                      bad.data_ptr(), _lib.stream(gpu))
            assert bool(bad)
            src[40 + (r + 1) * C - 1] = float(c[r, -1]) if f32 else int(c[r, -1])
    packed = torch.from_numpy(ref).to(gpu)
    CB = ref.shape[1]
    for width in {C, 2 * CB, max(1, C - 1)}:
        out = torch.full((R * width + 80,), 77, dtype=torch.int8, device=gpu)
        _lib.call("dscq_unpack_int4", packed.data_ptr(), R, CB, width, out[40:].data_ptr(),
                  _lib.stream(gpu))
        got = out.cpu().numpy()
        np.testing.assert_array_equal(got[40:40 + R * width].reshape(R, width),
                                      native.unpack_int4(ref, width))
        assert (got[:40] == 77).all() and (got[40 + R * width:] == 77).all()
