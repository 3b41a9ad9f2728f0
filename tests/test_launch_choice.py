"""The contractions' tile choices stay within what HIP launches, the lanes of all
workgroups together below 2^32, and leave the large tiles what they are faster on
(CPU: the choice alone)."""
import math
import random

import pytest

import choices


def _log_int(rng, low, high):
    return int(math.exp(rng.uniform(math.log(low), math.log(high))))


def test_chosen_grids_can_be_launched():
    """Tall and narrow products of up to 2^31 vectors or rows, as far as their
    operands fit 288 GB (1 x 1 x 273172763 among them, 2 GB)."""
    rng = random.Random(20)
    shapes = [(1, 1, 273172763), (2 ** 28, 32, 16), (1, 32, 1166382684)]
    while len(shapes) < 6000:
        batch, cols, rows = _log_int(rng, 2 ** 24, 2 ** 31 - 512), _log_int(rng, 1, 4096), _log_int(rng, 1, 256)
        if batch * (cols + rows) < 70e9:
            shapes.append((batch, cols, rows) if rng.random() < 0.5 else (rows, cols, batch))
    chosen = 0
    for batch, cols, rows in shapes:
        c32, c128 = -(-cols // 32) * 32, -(-cols // 128) * 128
        for choice in (choices.fp32(batch, cols, rows, True), choices.fp32(batch, cols, rows, False),
                       *(choices.bf16_activations(fmt, batch, c32, rows) for fmt in range(3)),
                       *(choices.block_scaled(fmt, batch, c128, rows) for fmt in range(3))):
            if choice:
                chosen += 1
                assert choice[0] * choice[1] < 2 ** 32, (batch, cols, rows, choice)
    assert chosen > 6000


# (batch, cols, rows): us on k-split tiles and on 256 x 128 tiles.
@pytest.mark.parametrize("shape,split,large", [
    ((716, 40, 5338), 24.8, 16.4), ((945, 32, 4625), 19.0, 13.2), ((760, 176, 8364), 56, 36),
    ((411, 112, 8840), 26.0, 22.6), ((631, 528, 9585), 88, 78), ((963, 1040, 7370), 158, 136),
    ((997, 1868, 7706), 269, 228), ((781, 2760, 7587), 285, 324), ((1025, 648, 3155), 57, 83),
    ((359, 2572, 5113), 99, 289), ((64, 2048, 8192), 22, 232)])
def test_fp32_tiles_are_the_faster_ones(shape, split, large):
    assert (choices.fp32(*shape) is not None) == (split < large)


# Rows that are not 16-byte aligned: us on k-split tiles and on the scalar kernel.
@pytest.mark.parametrize("shape,split,large", [
    ((818, 7, 6799), 26.4, 14.6), ((1000, 17, 7772), 33.6, 20.1), ((382, 31, 7280), 14.9, 10.8),
    ((734, 30, 8013), 27.5, 17.4), ((1078, 1, 4888), 23.2, 13.6), ((130, 5003, 1501), 28.8, 774), ((142, 3197, 2210), 26.5, 36.5)])
def test_unaligned_rows_take_the_faster_kernel(shape, split, large):
    assert (choices.fp32(*shape, aligned=False) is not None) == (split < large)


# K % 64 == 32, where the large kernel is l2c_qgemm.hip's: us on k-split tiles and on it,
# MXFP4 and bf16 weights.
@pytest.mark.parametrize("fmt,shape,split,large", [
    (0, (1011, 352, 7772), 56.3, 17.4), (0, (1018, 32, 7294), 22.4, 11.1), (0, (161, 32, 10576), 11.7, 6.4),
    (0, (969, 96, 2221), 11.9, 8.8), (0, (800, 864, 1807), 11.9, 17.7), (0, (72, 3168, 3049), 7.6, 41.6),
    (2, (1011, 352, 7772), 35.3, 17.8), (2, (1018, 32, 7294), 22.3, 11.3), (2, (969, 96, 2221), 11.7, 9.0),
    (2, (398, 608, 8821), 22.2, 16.8), (2, (59, 864, 9445), 8.7, 17.3), (2, (529, 3872, 400), 10.9, 56.7)])
def test_half_steps_take_the_faster_kernel(fmt, shape, split, large):
    assert (choices.bf16_activations(fmt, *shape) is not None) == (split < large)


# MXFP6: us on k-split tiles and on the large ones.
@pytest.mark.parametrize("shape,split,large", [
    ((449, 7936, 4725), 47.2, 44.4), ((754, 5376, 2765), 36.4, 34.1), ((387, 6016, 4745), 38.5, 36.5),
    ((363, 4608, 6074), 32.2, 30.8), ((588, 2688, 2547), 19.6, 22.4), ((699, 128, 2303), 7.6, 11.5)])
def test_mxfp6_takes_the_faster_tiles(shape, split, large):
    assert (choices.block_scaled(choices.MXFP6, *shape) is not None) == (split < large)
