"""The fp32 contraction's k-split tiles at their edges: K below, at and above
one step and one round of the waves, tiles with one row, one short and one
over, every tile size, aligned and unaligned rows, and the large and the scalar
kernel beside them in the choice, against float64."""
import numpy as np
import pytest

import choices

pytestmark = pytest.mark.gpu

# (Aligned products of at most 256 x 128 keep the large kernel's one tile.)
EDGES = [(1, 1, 1), (1, 3, 2), (15, 31, 17), (16, 32, 144), (17, 33, 15), (2, 255, 33), (16, 256, 144), (5, 257, 31),
         (33, 288, 168), (48, 996, 175), (33, 1001, 31), (7, 4097, 65), (257, 64, 5), (40, 96, 16)]
# A shape for each tile: (batch, cols, rows), the workgroup's lanes and the grid.
TILES = [((8, 768, 2048), 512, 128), ((108, 2048, 719), 512, 180), ((8, 326, 6744), 512, 211),
         ((141, 676, 5960), 256, 935), ((128, 3000, 1501), 512, 188), ((330, 2048, 3072), 256, 672),
         ((59, 1024, 5632), 256, 236), ((1024, 384, 4096), 256, 1024)]


def check(torch, l2c, batch, cols, rows, shift=0):
    print(f"case ksplit {batch}x{cols}x{rows}+{shift}", flush=True)
    rng = np.random.default_rng(batch * 7919 + cols * 31 + rows)
    X = rng.uniform(-1, 1, (batch, cols)).astype(np.float32)
    W = rng.uniform(-1, 1, (rows, cols)).astype(np.float32)

    def device(a):
        t = torch.zeros(a.size + shift, dtype=torch.float32, device="cuda")
        t[shift:] = torch.from_numpy(a.reshape(-1)).cuda()
        return t[shift:]

    x, w = device(X), device(W)
    outs = []
    for _ in range(2):
        # A guard row on either side: nothing past the result is written.
        buf = torch.full(((batch + 2) * rows,), 7.0, dtype=torch.float32, device="cuda")
        l2c.matmul(buf[rows:], x, w, batch, cols, rows)
        torch.cuda.synchronize()
        outs.append(buf.cpu().numpy().reshape(batch + 2, rows))
    np.testing.assert_array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    assert np.all(outs[0][[0, -1]] == 7.0)
    ref = X.astype(np.float64) @ W.astype(np.float64).T
    # Any order of K fp32 multiply-adds is within K u of the sum of magnitudes.
    bound = (cols + 8) * 2.0 ** -24 * (np.abs(X).astype(np.float64) @ np.abs(W).astype(np.float64).T)
    assert np.all(np.abs(outs[0][1:-1] - ref) <= bound)


@pytest.mark.parametrize("batch,cols,rows", EDGES)
@pytest.mark.parametrize("shift", [0, 1])
def test_edges(torch_gpu, l2c, batch, cols, rows, shift):
    check(torch_gpu, l2c, batch, cols, rows, shift)


@pytest.mark.parametrize("shape,block,grid", TILES)
def test_every_tile(torch_gpu, l2c, shape, block, grid):
    assert l2c.launch_shape(l2c.OP_MATMUL, *shape)[:2] == (grid, block)
    check(torch_gpu, l2c, *shape)
    check(torch_gpu, l2c, shape[0], shape[1] - 1, shape[2])


# The 256 x 128 tiles on ragged edges: K below, at and above one 32-deep step, its
# remainders, several tiles either way.
@pytest.mark.parametrize("batch,cols,rows", [(1021, 4, 8185), (1000, 32, 8190), (1021, 60, 8185), (1000, 96, 16300),
                                             (1021, 1028, 8185), (1000, 4100, 8190)])
def test_large_tiles(torch_gpu, l2c, batch, cols, rows):
    assert choices.fp32(batch, cols, rows) is None
    assert l2c.launch_shape(l2c.OP_MATMUL, batch, cols, rows)[:2] == (-(-batch // 256) * -(-rows // 128), 512)
    check(torch_gpu, l2c, batch, cols, rows)


# Unaligned rows of short K with many outputs, on the scalar kernel's ragged edges.
@pytest.mark.parametrize("batch,cols,rows", [(1021, 1, 4889), (818, 7, 6799), (1000, 31, 7772), (734, 33, 8013)])
def test_scalar_kernel(torch_gpu, l2c, batch, cols, rows):
    assert choices.fp32(batch, cols, rows, aligned=False) is None
    check(torch_gpu, l2c, batch, cols, rows)


def test_scalar_kernel_for_the_longest_rows(torch_gpu, l2c):
    """Rows past the large kernel's 32-bit offsets; sums of small integers are exact."""
    torch = torch_gpu
    batch, cols, rows = 3, 2097156, 5
    print(f"case scalar kernel {batch}x{cols}x{rows}", flush=True)
    assert choices.fp32(batch, cols, rows) is None
    gen = torch.Generator("cuda").manual_seed(9)
    x = torch.randint(-1, 2, (batch, cols), device="cuda", generator=gen).float()
    w = torch.randint(-1, 2, (rows, cols), device="cuda", generator=gen).float()
    buf = torch.full((batch + 2, rows), 7.0, device="cuda")
    l2c.matmul(buf[1:], x, w, batch, cols, rows)
    assert torch.equal(buf[1:-1].double(), (x.double()[:, None] * w.double()[None]).sum(-1))
    assert bool((buf[0] == 7.0).all()) and bool((buf[-1] == 7.0).all())


def test_padding_does_not_touch_infinities_and_nan(torch_gpu, l2c):
    """An infinite and a NaN value reach their own row and column only, also
    through the clamped rows and the padded k of a partial step."""
    torch = torch_gpu
    batch, cols, rows = 18, 37, 19
    X, W = torch.ones(batch, cols, device="cuda"), torch.ones(rows, cols, device="cuda")
    X[17, 36], W[18, 36] = float("inf"), float("nan")
    out = torch.empty(batch, rows, device="cuda")
    l2c.matmul(out, X, W, batch, cols, rows)
    torch.cuda.synchronize()
    want = torch.full((batch, rows), 37.0)
    want[17, :] = float("inf")
    want[:, 18] = float("nan")
    torch.testing.assert_close(out.cpu(), want, equal_nan=True, rtol=0, atol=0)


def test_more_rows_than_small_tiles_can_be_launched_for(torch_gpu, l2c):
    """16 x 16 tiles of this shape have more than 2^32 lanes."""
    torch = torch_gpu
    rows = 273172763
    print(f"case ksplit 1x1x{rows}", flush=True)
    W = torch.arange(rows, dtype=torch.int32, device="cuda").bitwise_and_(0xFFFF).float()
    out = torch.full((rows,), float("nan"), device="cuda")
    l2c.matmul(out, torch.tensor([3.0], device="cuda"), W, 1, 1, rows)
    assert torch.equal(out, W.mul_(3.0))
