"""Products of at most 64 rows or columns on the skinny kernel, through the automatic choice: the long
operand on either side, every layout (int8: both operands K-contiguous), one row, ragged tiles, a ragged
last unit of K and an odd number of units, about a tile per CU with a longer K.  Reference: numpy in 64
bits (integers exactly); floating tolerance: fp32 sums of K terms, each step's relative rounding at
most 2^-23, random over the terms: sqrt(K) 2^-23."""
import math

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def _takes(dt, shape, layout):
    """Int8 takes this kernel with both operands K-contiguous only; a 16-bit M- or N-contiguous extent holds
    whole 16-byte chunks."""
    arow, brow = bool(layout & 1), bool(layout & 2)
    if dt == "i8":
        return arow and not brow
    return (arow or shape[0] % 8 == 0) and (not brow or shape[1] % 8 == 0)


@pytest.mark.parametrize("dt,shape,layout", [(dt, shape, layout) for dt, shape in [
    ("f16", (64, 128, 1024)), ("bf16", (40, 200, 1096)), ("f16", (1, 72, 1160)), ("bf16", (264, 64, 2040)),
    ("f16", (1032, 8, 1024)), ("bf16", (16, 12352, 2056)), ("f16", (16376, 24, 4104)), ("i8", (33, 12290, 4112)),
    ("i8", (15600, 17, 4112)), ("i8", (64, 12288, 8192))] for layout in range(8) if _takes(dt, shape, layout)])
def test_gemm_skinny(gpu, dt, shape, layout):
    lh = gpu
    M, N, K = shape
    arow, brow, crow = bool(layout & 1), bool(layout & 2), bool(layout & 4)
    announce(f"gemm skinny {dt} layout={layout} M={M} N={N} K={K}")
    rng = np.random.default_rng(M + layout)
    def operand(rows, cols, row_major):
        if dt == "i8":
            v = rng.integers(-128, 128, (rows, cols)).astype(np.int8)
            wide = v.astype(np.float64)   # exact: the sums stay below 2^53
        elif dt == "f16":
            v = rng.uniform(-1, 1, (rows, cols)).astype(np.float16)
            wide = v.astype(np.float64)
        else:
            v = (rng.uniform(-1, 1, (rows, cols)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
            wide = (v.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        return lh.HIPDeviceArray.from_numpy(v, dt, order="C" if row_major else "F"), wide
    A, wa = operand(M, K, arow)
    B, wb = operand(K, N, brow)
    inner, pad = (N if crow else M), 3 if layout in (1, 4, 5) else 4
    C = lh.HIPDeviceArray("i32" if dt == "i8" else "f32", (M if crow else N, inner + pad), order="C")
    C.fill_bytes(0xEE)
    lh.kernel_log_clear()
    lh.gemm_raw(dt, C.dtype, A.ptr, B.ptr, C.ptr, M, N, K, K if arow else M, N if brow else K, inner + pad, layout)
    assert lh.kernel_log() == ["gemm_skinny_kernel"], lh.kernel_log()
    got = C.to_numpy()
    assert (np.ascontiguousarray(got[:, inner:]).view(np.uint8) == 0xEE).all(), "C's padding was written"
    got = got[:, :inner] if crow else got[:, :inner].T
    want = wa @ wb
    if dt == "i8":
        np.testing.assert_array_equal(got, want.astype(np.int64))
    else:
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert err <= math.sqrt(K) * 2.0 ** -23, err
