"""The bf16-activation contractions on k-split tiles at their edges: K of one
32-deep unit to several steps and remainders, tiles one row short and one over,
every tile size, and the large kernels on both sides of the choice, against
float64 products of the dequantized operands."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MXFP4, FP8, BF16 = 0, 1, 2
E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def operands(torch, fmt, batch, cols, rows, scale_shift=0):
    """Random codes (every E2M1 code, every finite E4M3 code, scale bytes of
    100 to 150) and bf16 activations, with the values in float64."""
    gen = torch.Generator("cuda").manual_seed(batch * 7919 + cols * 31 + rows)
    x = torch.randn(batch, cols, device="cuda", generator=gen).bfloat16()
    if fmt == BF16:
        w = torch.randn(rows, cols, device="cuda", generator=gen).bfloat16()
        return x, w.view(torch.int16), None, w.double()
    if fmt == FP8:
        codes = torch.randint(0, 256, (rows, cols), device="cuda", generator=gen, dtype=torch.int32)
        codes = torch.where((codes & 0x7F) == 0x7F, codes - 1, codes).to(torch.uint8)
        scales = torch.rand(rows, device="cuda", generator=gen) + 0.5
        return x, codes, scales, codes.view(torch.float8_e4m3fn).double() * scales.double()[:, None]
    codes = torch.randint(0, 256, (rows, cols // 2), device="cuda", generator=gen, dtype=torch.int32)
    table = torch.tensor(E2M1 + [-v for v in E2M1], dtype=torch.float64, device="cuda")
    values = torch.stack((table[(codes & 15).long()], table[(codes >> 4).long()]), -1).reshape(rows, cols)
    sbytes = torch.randint(100, 151, (rows, cols // 32), device="cuda", generator=gen, dtype=torch.int32)
    values = values.reshape(rows, -1, 32) * ((sbytes - 127 + 1023).long() << 52).view(torch.float64)[:, :, None]
    scales = torch.zeros(scale_shift + sbytes.numel(), dtype=torch.uint8, device="cuda")
    scales[scale_shift:] = sbytes.to(torch.uint8).reshape(-1)
    return x, codes.to(torch.uint8), scales[scale_shift:], values.reshape(rows, cols)


def check(torch, l2c, fmt, batch, cols, rows, scale_shift=0):
    print(f"case q ksplit fmt={fmt} {batch}x{cols}x{rows}+{scale_shift}", flush=True)
    x, codes, scales, W = operands(torch, fmt, batch, cols, rows, scale_shift)
    xbits = x.view(torch.int16)
    alpha = torch.tensor([0.375], dtype=torch.float32, device="cuda")
    outs = []
    for _ in range(2):
        buf = torch.full((batch + 2, rows), 7.0, dtype=torch.float32, device="cuda")
        if fmt == BF16:
            l2c.matmul_bf16(buf[1:], xbits, codes, batch, cols, rows, alpha=alpha)
        else:
            l2c.matmul_q(buf[1:], xbits, codes, scales, fmt, batch, cols, rows)
        torch.cuda.synchronize()
        assert bool((buf[0] == 7.0).all()) and bool((buf[-1] == 7.0).all())
        outs.append(buf[1:-1])
    assert torch.equal(outs[0].view(torch.int32), outs[1].view(torch.int32))
    a = 0.375 if fmt == BF16 else 1.0
    ref, mag = a * (x.double() @ W.T), a * (x.double().abs() @ W.abs().T)
    # Exact products: any order of K fp32 additions, and one product with a scale.
    assert bool(((outs[0].double() - ref).abs() <= (cols + 8) * 2.0 ** -24 * mag).all())


@pytest.mark.parametrize("fmt", [MXFP4, FP8, BF16])
@pytest.mark.parametrize("batch,cols,rows", [(1, 32, 1), (1, 64, 15), (15, 96, 17), (16, 128, 16), (17, 160, 33),
                                             (2, 512, 31), (33, 1024, 40), (7, 1056, 65), (48, 2080, 47)])
def test_edges(torch_gpu, l2c, fmt, batch, cols, rows):
    check(torch_gpu, l2c, fmt, batch, cols, rows)


# (batch, rows) and the workgroup's lanes and tile by the choice on this shape.
@pytest.mark.parametrize("batch,rows,block,bm,bn", [(5, 300, 512, 16, 16), (3, 4099, 512, 16, 32),
                                                    (9, 8215, 256, 16, 64), (82, 2705, 256, 32, 32),
                                                    (17, 8285, 256, 32, 64), (33, 8381, 256, 48, 64)])
def test_every_tile(torch_gpu, l2c, batch, rows, block, bm, bn):
    for fmt in (MXFP4, FP8):
        grid = -(-batch // bm) * -(-rows // bn)
        assert l2c.launch_shape(l2c.OP_MATMUL_Q, batch, 352, rows, fmt)[:2] == (grid, block)
    for fmt in (MXFP4, FP8, BF16):
        check(torch_gpu, l2c, fmt, batch, 352, rows)


def test_tile_of_48_by_32(torch_gpu, l2c):
    assert l2c.launch_shape(l2c.OP_MATMUL_Q, 33, 288, 5467, FP8)[:2] == (171, 256)
    check(torch_gpu, l2c, FP8, 33, 288, 5467)
    check(torch_gpu, l2c, BF16, 33, 288, 5467)


def test_mxfp4_scales_at_an_odd_address(torch_gpu, l2c):
    check(torch_gpu, l2c, MXFP4, 19, 416, 70, scale_shift=1)


# The large kernels on ragged edges: one step, fewer steps than their rings
# hold, and K % 64 == 32.
@pytest.mark.parametrize("fmt", [MXFP4, FP8, BF16])
@pytest.mark.parametrize("cols", [64, 192, 288, 640])
def test_large_tiles(torch_gpu, l2c, fmt, cols):
    batch, rows = 1021, 8185
    if fmt != BF16:
        assert l2c.launch_shape(l2c.OP_MATMUL_Q, batch, cols, rows, fmt)[1] == 512
    check(torch_gpu, l2c, fmt, batch, cols, rows)
