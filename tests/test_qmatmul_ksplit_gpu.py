"""The bf16-activation contractions on k-split tiles at their edges: K of one
32-deep unit to several steps and remainders, tiles one row short and one over,
every tile size, and the 128 x 128 and large kernels beside them in the choice,
against float64 products of the dequantized operands."""
import numpy as np
import pytest

import choices

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


# Shapes with the waves and tile the choice takes: (batch, cols, rows), fmt,
# waves, batch rows, weight rows.
TILES = [((5, 128, 300), 0, 4, 16, 16), ((3, 672, 294), 0, 8, 16, 16), ((15, 128, 4351), 0, 2, 16, 32),
         ((7, 384, 4209), 0, 4, 16, 32), ((19, 128, 4168), 0, 2, 32, 32), ((9, 512, 8500), 0, 4, 16, 64),
         ((608, 896, 400), 0, 4, 32, 32),
         ((19, 672, 8733), 0, 4, 32, 64), ((34, 480, 5682), 0, 4, 48, 32), ((65, 128, 7380), 0, 2, 48, 64),
         ((310, 2560, 1608), 0, 4, 48, 64), ((165, 128, 4262), 0, 2, 64, 64), ((5, 128, 300), 1, 4, 16, 16),
         ((3, 320, 304), 1, 8, 16, 16), ((15, 128, 4351), 1, 2, 16, 32), ((7, 192, 4129), 1, 4, 16, 32),
         ((19, 128, 4168), 1, 2, 32, 32), ((9, 512, 8500), 1, 4, 16, 64),
         ((600, 512, 409), 1, 4, 32, 32), ((18, 576, 8222), 1, 4, 32, 64),
         ((38, 256, 5479), 1, 4, 48, 32), ((65, 128, 7380), 1, 2, 48, 64), ((37, 1248, 9047), 1, 4, 48, 64),
         ((115, 320, 6157), 1, 4, 64, 64)]


@pytest.mark.parametrize("shape,fmt,waves,bm,bn", TILES)
def test_every_tile(torch_gpu, l2c, shape, fmt, waves, bm, bn):
    batch, cols, rows = shape
    grid = -(-batch // bm) * -(-rows // bn)
    assert l2c.launch_shape(l2c.OP_MATMUL_Q, batch, cols, rows, fmt)[:2] == (grid, 64 * waves)
    check(torch_gpu, l2c, fmt, batch, cols, rows)
    if fmt == FP8:
        check(torch_gpu, l2c, BF16, batch, cols, rows)


# bf16 weights, whose choice no l2c_launch_shape operation reports: waves, batch rows
# and weight rows of every tile.
@pytest.mark.parametrize("waves,bm,bn", [(8, 16, 16), (4, 16, 16), (4, 16, 32), (4, 16, 64), (4, 32, 32), (4, 48, 32),
                                         (4, 32, 64), (4, 48, 64), (4, 64, 64), (2, 16, 32), (2, 32, 32), (2, 48, 64)])
def test_every_bf16_tile(torch_gpu, l2c, waves, bm, bn):
    shape = choices.shape_on(lambda *s: choices.bf16_activations(BF16, *s), 32, waves, bm, bn)
    check(torch_gpu, l2c, BF16, *shape)


def test_mxfp4_scales_at_an_odd_address(torch_gpu, l2c):
    check(torch_gpu, l2c, MXFP4, 19, 416, 70, scale_shift=1)


# The 128 x 128 tiles: one 64-deep slice, fewer and more than their rings hold, odd
# and even counts, tiles one row over and one short.
@pytest.mark.parametrize("fmt", [MXFP4, FP8, BF16])
@pytest.mark.parametrize("batch,cols,rows", [(513, 64, 6500), (897, 128, 4095), (385, 192, 8190), (510, 320, 8191),
                                             (1009, 384, 4001), (1024, 384, 4096), (385, 2112, 8190),
                                             (255, 4096, 11009)])
def test_mid_tiles(torch_gpu, l2c, fmt, batch, cols, rows):
    grid = -(-batch // 128) * -(-rows // 128)
    assert choices.bf16_activations(fmt, batch, cols, rows) == (grid, 512)
    if fmt != BF16:
        assert l2c.launch_shape(l2c.OP_MATMUL_Q, batch, cols, rows, fmt)[:2] == (grid, 512)
    check(torch_gpu, l2c, fmt, batch, cols, rows)


def test_mid_shape_with_mxfp4_scales_at_an_odd_address(torch_gpu, l2c):
    check(torch_gpu, l2c, MXFP4, 385, 2112, 8190, scale_shift=1)


# The large kernels on ragged edges: one step, fewer steps than their rings
# hold, and K % 64 == 32.
@pytest.mark.parametrize("fmt", [MXFP4, FP8, BF16])
@pytest.mark.parametrize("cols", [64, 192, 1056, 1088])
def test_large_tiles(torch_gpu, l2c, fmt, cols):
    batch, rows = 1021, 23040064 // cols + 1
    assert choices.bf16_activations(fmt, batch, cols, rows) is None
    if fmt != BF16:
        bm, bn = (128, 256) if fmt == FP8 and cols % 64 == 0 else (256, 128)
        grid = -(-batch // bm) * -(-rows // bn)
        assert l2c.launch_shape(l2c.OP_MATMUL_Q, batch, cols, rows, fmt)[:2] == (grid, 512)
    check(torch_gpu, l2c, fmt, batch, cols, rows)
