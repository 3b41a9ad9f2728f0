"""The tile choices of the k-split contractions, called in libl2c.so on the CPU
(csrc/l2c_common.h declares them). Each returns (workgroups, lanes), or None where
a large kernel is preferred."""
import ctypes
import random

import l2c

_I, _P = ctypes.c_int, ctypes.POINTER(ctypes.c_int)
BF16 = MXFP6 = 2  # beside the l2c_qformat values


def _call(symbol, types, *args):
    fn = getattr(l2c.load(), symbol)
    fn.restype, fn.argtypes = ctypes.c_bool, [*types, _P, _P, ctypes.POINTER(ctypes.c_void_p)]
    grid, block, kernel = _I(), _I(), ctypes.c_void_p()
    chosen = fn(*args, ctypes.byref(grid), ctypes.byref(block), ctypes.byref(kernel))
    return (grid.value, block.value) if chosen else None


def fp32(batch, cols, rows, aligned=True):
    return _call("_Z28l2c_gemm_ksplit_launch_shapeiiibPiS_PPKv", [_I, _I, _I, ctypes.c_bool], batch, cols, rows, aligned)


def bf16_activations(fmt, batch, cols, rows):
    """fmt: MXFP4, fp8 or BF16 weights (and so the 128 x 128 tiles where preferred)."""
    bm, bn = (128, 256) if fmt == l2c.Q_FP8 and cols % 64 == 0 else (256, 128)
    return _call("_Z29l2c_qgemm_ksplit_launch_shapeiiiixPiS_PPKv", [_I, _I, _I, _I, ctypes.c_longlong], fmt, batch, cols,
                 rows, -(-batch // bm) * -(-rows // bn))


def block_scaled(fmt, batch, cols, rows):
    """fmt: MXFP4 or fp8 weights with MXFP8 activations, or MXFP6 operands."""
    return _call("_Z30l2c_scgemm_ksplit_launch_shapeiiiiPiS_PPKv", [_I, _I, _I, _I], fmt, batch, cols, rows)


def shape_on(choice, granule, waves, bm, bn, tries=20000):
    """A ragged (batch, cols, rows), cols a multiple of `granule`, which `choice`
    sends to tiles of bm x bn by `waves` waves, and to no other tile's grid."""
    rng = random.Random(waves * 10000 + bm * 100 + bn)
    log_int = lambda low, high: int(round(low * (high / low) ** rng.random()))  # noqa: E731
    tiles = {(w, m, n) for w in (2, 4, 8) for m in (16, 32, 48, 64) for n in (16, 32, 48, 64)}
    for _ in range(tries):
        batch, cols, rows = log_int(1, 700), granule * log_int(1, 8192 // granule), log_int(16, 11008)
        if batch % bm == 0 or rows % bn == 0 or batch * cols * rows > 2e9:
            continue
        grids = {t: (-(-batch // t[1]) * -(-rows // t[2]), 64 * t[0]) for t in tiles}
        mine = grids.pop((waves, bm, bn))
        if mine not in grids.values() and choice(batch, cols, rows) == mine:
            return batch, cols, rows
    raise AssertionError(f"no shape goes to {bm} x {bn} tiles of {waves} waves")
