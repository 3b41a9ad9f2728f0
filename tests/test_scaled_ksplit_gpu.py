"""The block-scaled contractions on k-split tiles: every tile at ragged edges,
one step to more steps than waves, and the large kernels beside them, to the
bounds of the tests of l2c_matmul_qs and l2c_matmul_mxfp6."""
import numpy as np
import pytest

import choices
import lowprec_oracle as lo
import oracle
from test_lowprec_gpu import check_bound, dev, inputs, mxfp6_buffers
from test_quant_scaled_gpu import check_qs

pytestmark = pytest.mark.gpu

EDGES = [(1, 128, 1), (15, 256, 17), (17, 384, 15), (16, 640, 33), (33, 1152, 31), (5, 2176, 64)]
# Shapes with the waves and tile the choice takes for MXFP4 and fp8 weights: (batch, cols, rows), waves, batch
# rows, weight rows.
TILES = [((5, 128, 293), 4, 16, 16), ((3, 640, 295), 8, 16, 16), ((15, 128, 4107), 2, 16, 32),
         ((7, 384, 4108), 4, 16, 32), ((9, 640, 8500), 4, 16, 64),
         ((17, 128, 4754), 2, 32, 32), ((17, 896, 4621), 4, 32, 32),
         ((17, 896, 9778), 4, 32, 64), ((34, 384, 5957), 4, 48, 32), ((65, 128, 6720), 2, 48, 64),
         ((36, 2432, 9256), 4, 48, 64), ((225, 512, 3277), 4, 64, 64)]


def check_mxfp6(torch, l2c, batch, cols, rows):
    print(f"case mxfp6 ksplit {batch}x{cols}x{rows}", flush=True)
    x, w = inputs("random", batch, cols), inputs("random", rows, cols)
    xc, xs = oracle.quantize_mxfp6(x, batch, cols)
    wc, ws = oracle.quantize_mxfp6(w, rows, cols)
    dxc, dxs = mxfp6_buffers(torch, l2c, batch, cols)
    dwc, dws = mxfp6_buffers(torch, l2c, rows, cols)
    l2c.quantize_mxfp6(dxc, dxs, dev(torch, x), batch, cols)
    l2c.quantize_mxfp6(dwc, dws, dev(torch, w), rows, cols)
    buf = torch.full((batch + 2, rows), 7.0, dtype=torch.float32, device="cuda")
    l2c.matmul_mxfp6(buf[1:], dxc, dxs, dwc, dws, batch, cols, rows)
    torch.cuda.synchronize()
    assert bool((buf[0] == 7.0).all()) and bool((buf[-1] == 7.0).all())
    check_bound(buf[1:-1].cpu().numpy(), lo.dequantize_mxfp6(xc, xs, batch, cols),
                lo.dequantize_mxfp6(wc, ws, rows, cols), 1.0, cols)


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("batch,cols,rows", EDGES)
def test_qs_edges(torch_gpu, l2c, orc, fmt, batch, cols, rows):
    inp = orc.fill("normal", 11, batch, cols, rows)
    check_qs(torch_gpu, l2c, orc, fmt, batch, cols, rows, inp.input, inp.matrix, "ksplit")


@pytest.mark.parametrize("batch,cols,rows", EDGES)
def test_mxfp6_edges(torch_gpu, l2c, batch, cols, rows):
    check_mxfp6(torch_gpu, l2c, batch, cols, rows)


@pytest.mark.parametrize("shape,waves,bm,bn", TILES)
def test_every_tile(torch_gpu, l2c, orc, shape, waves, bm, bn):
    batch, cols, rows = shape
    inp = orc.fill("normal", 12, batch, cols, rows)
    for fmt in (0, 1):
        grid = -(-batch // bm) * -(-rows // bn)
        assert l2c.launch_shape(l2c.OP_MATMUL_QS, batch, cols, rows, fmt)[:2] == (grid, 64 * waves)
        check_qs(torch_gpu, l2c, orc, fmt, batch, cols, rows, inp.input, inp.matrix, "ksplit tile")
    check_mxfp6(torch_gpu, l2c, batch, cols, rows)


# MXFP6, whose choice no l2c_launch_shape operation reports: waves, batch rows and
# weight rows of every tile.
@pytest.mark.parametrize("waves,bm,bn", [(8, 16, 16), (4, 16, 16), (4, 16, 32), (4, 16, 64), (4, 32, 32), (4, 48, 32),
                                         (4, 32, 64), (4, 48, 64), (4, 64, 64), (2, 16, 32), (2, 32, 32), (2, 48, 64)])
def test_every_mxfp6_tile(torch_gpu, l2c, waves, bm, bn):
    shape = choices.shape_on(lambda *s: choices.block_scaled(choices.MXFP6, *s), 128, waves, bm, bn)
    check_mxfp6(torch_gpu, l2c, *shape)


# The large kernels on ragged edges, one step and more than their rings hold.
@pytest.mark.parametrize("cols", [128, 640])
def test_large_tiles(torch_gpu, l2c, orc, cols):
    batch, rows = 1021, 1930
    inp = orc.fill("normal", 14, batch, cols, rows)
    for fmt in (0, 1):
        assert l2c.launch_shape(l2c.OP_MATMUL_QS, batch, cols, rows, fmt)[1] == 512
        check_qs(torch_gpu, l2c, orc, fmt, batch, cols, rows, inp.input, inp.matrix, "large")


def test_large_mxfp6_tiles(torch_gpu, l2c):
    assert choices.block_scaled(choices.MXFP6, 1021, 640, 8185) is None
    check_mxfp6(torch_gpu, l2c, 1021, 640, 8185)
