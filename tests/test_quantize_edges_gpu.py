"""The MXFP4 and fp8 weight quantizers at the edges of their lane layouts and
of their arithmetic, code for code against the encoders of l2c_formats.h built
for the CPU and numpy's fp32 division."""
import ctypes
import os

import numpy as np
import pytest

from conftest import PKG
from test_formats_host import SIGNIFICANDS, fp8_midpoint_rows

pytestmark = pytest.mark.gpu


def encode(fmt, v):
    lib = ctypes.CDLL(os.path.join(PKG, "lib", "libl2c_formats_host.so"))
    v = np.ascontiguousarray(v, np.float32)
    out = np.empty(v.size, np.uint8)
    lib.l2cf_encode_array(ctypes.c_int(fmt), v.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(v.size),
                          out.ctypes.data_as(ctypes.c_void_p))
    return out


def weights(rows, cols, block):
    """Blocks of normals at magnitudes 2^-140 to 2^120, with midpoints of both
    formats' codes, zeros of both signs, infinities, NaN and a whole block of
    each special value."""
    rng = np.random.default_rng(rows * 100003 + cols)
    w = rng.standard_normal((rows * cols) // block * block).astype(np.float32).reshape(-1, block)
    w *= np.exp2(rng.integers(-140, 121, (w.shape[0], 1))).astype(np.float32)
    plain = rng.random(w.shape[0]) < 0.6
    w[plain] = (rng.integers(-4096, 4097, (int(plain.sum()), block)) / 512.0).astype(np.float32)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45, -1e-45, 3e38], np.float32)
    for k, v in enumerate(special):
        w[(3 * k + 1) % w.shape[0], (5 * k) % block] = v
        if w.shape[0] > 40:
            w[20 + k, :] = v
    out = np.zeros(rows * cols, np.float32)
    out[:w.size] = w.reshape(-1)
    return out


def device(torch, w, shift):
    """w on the GPU, `shift` floats past a 16-byte boundary."""
    t = torch.zeros(w.size + shift, dtype=torch.float32, device="cuda")
    t[shift:] = torch.from_numpy(w).cuda()
    return t[shift:]


# 1024 float4 a workgroup: one block, a whole workgroup, one block more, many.
@pytest.mark.parametrize("rows,cols,shift", [(1, 32, 0), (1, 4096, 0), (3, 1376, 0), (57, 2976, 0), (57, 2976, 1)])
def test_mxfp4_edges(torch_gpu, l2c, rows, cols, shift):
    torch = torch_gpu
    print(f"case mxfp4 edges {rows}x{cols}+{shift}", flush=True)
    w = weights(rows, cols, 32)
    codes = torch.full((rows * cols // 2,), 0xAA, dtype=torch.uint8, device="cuda")
    scales = torch.full((rows * cols // 32,), 0xAA, dtype=torch.uint8, device="cuda")
    l2c.quantize_mxfp4(codes, scales, device(torch, w, shift), rows, cols)
    torch.cuda.synchronize()
    blocks = w.reshape(-1, 32)
    amax = np.fmax.reduce(np.abs(blocks), axis=1, initial=0.0).astype(np.float32)
    bits = amax.view(np.uint32)
    field = (bits >> 23).astype(np.int64) & 0xFF
    x = np.where(field == 0, -127, np.clip(field - 130 + ((bits >> 22) & 1), -127, 127))
    with np.errstate(over="ignore", invalid="ignore", divide="ignore"):
        scaled = blocks * np.exp2(-x[:, None].astype(np.float64)).astype(np.float32)
    want = encode(0, scaled).reshape(-1, 32)
    want[~(amax > 0)] = 0
    np.testing.assert_array_equal(scales.cpu().numpy(), (x + 127).astype(np.uint8))
    np.testing.assert_array_equal(codes.cpu().numpy(), (want.reshape(-1, 2)[:, 0] | want.reshape(-1, 2)[:, 1] << 4))


# Each register-resident instance at its first and last length, rows that are
# no multiple of the workgroup's, the streamed form past 16384, for a length
# that is no multiple of four and for misaligned weights.
@pytest.mark.parametrize("rows,cols,shift", [(5, 4, 0), (7, 512, 0), (6, 516, 0), (9, 1024, 0), (5, 1028, 0),
                                             (6, 2048, 0), (5, 2052, 0), (65, 4096, 0), (3, 4100, 0), (3, 8192, 0),
                                             (2, 8196, 0), (2, 16384, 0), (2, 16388, 0), (9, 1001, 0), (9, 1000, 1)])
def test_fp8_edges(torch_gpu, l2c, rows, cols, shift):
    torch = torch_gpu
    print(f"case fp8 edges {rows}x{cols}+{shift}", flush=True)
    w = weights(rows, cols, cols).reshape(rows, cols)
    # Rows of tiny scales, below the range of the quotient's short form.
    rng = np.random.default_rng(cols)
    for r, top in enumerate((448.0 * 2.0 ** -100, 448.0 * 2.0 ** -101, 2.0 ** -130)[:rows - 1]):
        w[r] = (rng.uniform(-1, 1, cols) * top).astype(np.float32)
        w[r, 0] = top
    codes = torch.full((rows * cols,), 0xAA, dtype=torch.uint8, device="cuda")
    scales = torch.zeros(rows, dtype=torch.float32, device="cuda")
    l2c.quantize_fp8(codes, scales, device(torch, w.reshape(-1), shift), rows, cols)
    torch.cuda.synchronize()
    amax = np.fmax.reduce(np.abs(w), axis=1, initial=0.0).astype(np.float32)
    scale = np.where(amax > 0, amax / np.float32(448.0), np.float32(1.0)).astype(np.float32)
    with np.errstate(over="ignore", invalid="ignore", divide="ignore"):
        want = encode(2, w / scale[:, None])
    np.testing.assert_array_equal(scales.cpu().numpy(), scale)
    np.testing.assert_array_equal(codes.cpu().numpy(), want)


# By 16-byte loads and, one float past the boundary, by the streamed form.
@pytest.mark.parametrize("shift", [0, 1])
def test_fp8_midpoints_at_small_scales(torch_gpu, l2c, shift):
    torch = torch_gpu
    print(f"case fp8 midpoints +{shift}", flush=True)
    w = fp8_midpoint_rows(range(-101, -90), SIGNIFICANDS)
    rows, cols = w.shape
    codes = torch.full((rows * cols,), 0xAA, dtype=torch.uint8, device="cuda")
    scales = torch.zeros(rows, dtype=torch.float32, device="cuda")
    l2c.quantize_fp8(codes, scales, device(torch, w.reshape(-1), shift), rows, cols)
    torch.cuda.synchronize()
    scale = w[:, 75] / np.float32(448.0)
    np.testing.assert_array_equal(scales.cpu().numpy(), scale)
    np.testing.assert_array_equal(codes.cpu().numpy(), encode(2, w / scale[:, None]))
