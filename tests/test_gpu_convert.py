"""Index-side conversions at the edges of their kernels' shapes, bit for bit against the oracle."""

import numpy as np
import pytest

import oracle
from helpers import normalized

pytestmark = pytest.mark.gpu


def _shifted(capi, x, shift):
    """x on the device, starting `shift` floats into its allocation."""
    flat = np.concatenate([np.zeros(shift, np.float32), x.ravel()])
    d = capi.DeviceArray.from_host(flat)
    return d, d.ptr + 4 * shift


# 16, 32 and 64 lanes a row at their first and last widths, one to four vectors a lane; widths that
# are no multiple of 4 (and an unaligned source), in registers up to 1024 and read twice beyond
@pytest.mark.parametrize("rows,dim,shift", [
    (1, 4, 0), (37, 64, 0), (18, 68, 0), (33, 256, 0), (9, 260, 0), (21, 512, 0), (5, 516, 0), (7, 1024, 0),
    (5, 1028, 0), (3, 2052, 0), (13, 1, 0), (6, 1023, 0), (4, 1025, 0), (11, 768, 1),
])
def test_quantize_rows_shapes(gpu, rows, dim, shift):
    capi = gpu
    x = normalized(rows, dim, 1000 + dim)
    x[0] = 0.0  # an all-zero row has scale 1
    codes, scales = oracle.quantize_rows_i8(x)
    d_x, address = _shifted(capi, x, shift)
    d_codes, d_scales = capi.DeviceArray((rows, dim), np.int8), capi.DeviceArray(rows, np.float32)
    capi.launch_quantize_rows_i8(address, rows, dim, d_codes, d_scales)
    capi.synchronize()
    assert np.array_equal(d_codes.to_host(), codes) and np.array_equal(d_scales.to_host(), scales)


# rows of one piece and less, of whole pieces, with a last piece of one word and of a part of a
# word; more and fewer pieces than one wavefront's step
@pytest.mark.parametrize("rows,dim", [(1, 1), (3, 31), (40, 32), (17, 33), (9, 64), (1003, 96), (5, 100), (77, 1024)])
def test_pack_binary_shapes(gpu, rows, dim):
    capi = gpu
    x = normalized(rows, dim, 2000 + dim)
    x[:, ::5] = 0.0
    x[:, 3::7] = -0.0
    d_x = capi.DeviceArray.from_host(x)
    out = capi.DeviceArray((rows, (dim + 31) // 32), np.uint32)
    capi.launch_pack_binary(d_x, out, rows, dim)
    capi.synchronize()
    assert np.array_equal(out.to_host(), oracle.pack_binary(x))


# fewer elements than a group, a remainder past the last group, more than one block, an unaligned source
@pytest.mark.parametrize("count,shift", [(1, 0), (3, 0), (4, 0), (4099, 0), (70_001, 0), (4099, 1)])
def test_elementwise_shapes(gpu, count, shift):
    capi = gpu
    x = np.random.default_rng(count).standard_normal((1, count)).astype(np.float32)
    x[0, 0] = 1e6  # beyond both types' ranges
    d_x, address = _shifted(capi, x, shift)
    half, code = capi.DeviceArray((1, count), np.float16), capi.DeviceArray((1, count), np.int8)
    capi.launch_convert_f32_to_f16(address, half, count)
    capi.launch_convert_f32_to_i8(address, code, count, 0.01)
    capi.synchronize()
    assert np.array_equal(half.to_host().view(np.uint16), oracle.f32_to_f16(x).view(np.uint16))
    assert np.array_equal(code.to_host(), oracle.quantize_i8(x, 0.01))
