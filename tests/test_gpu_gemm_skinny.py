"""Products of at most 64 rows or columns on the skinny kernel, through the automatic choice: the long
operand on either side, every layout (int8: both operands K-contiguous), one row, ragged tiles, a ragged
last unit of K and an odd number of units, about a tile per CU with a longer K; rows of whole 128-byte lines
(padded, the padding NaN) and rows that cross them.  And the calls that stay on the small-product kernel:
where that one splits K on few tiles, and more rows that cross lines than pay.  Reference:
numpy in 64 bits (integers exactly); floating tolerance: fp32 sums of K terms, each step's relative rounding
at most 2^-23, random over the terms: sqrt(K) 2^-23."""
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


SKINNY = [
    ("f16", (64, 128, 1024), False), ("bf16", (40, 200, 1096), False), ("f16", (1, 72, 1160), False),
    ("bf16", (264, 64, 1784), False), ("bf16", (264, 64, 1784), True), ("f16", (1032, 8, 1024), False),
    ("bf16", (16, 12352, 2056), False), ("f16", (16376, 24, 4104), False), ("f16", (15608, 64, 4104), True),
    ("i8", (33, 12290, 4112), False), ("i8", (15600, 17, 4112), False), ("i8", (64, 12288, 8192), False)]
SMALL = [("bf16", (264, 64, 2040), True, 5), ("f16", (64, 64, 1920), False, 3), ("bf16", (64, 12480, 1736), False, 5),
         ("f16", (15608, 48, 6480), False, 1), ("f16", (64, 15608, 4104), False, 7), ("i8", (64, 12672, 7792), False, 5),
         ("i8", (33, 12290, 7696), False, 1)]


@pytest.mark.parametrize("dt,shape,lines,layout", [(dt, shape, lines, layout) for dt, shape, lines in SKINNY
                                                   for layout in range(8) if _takes(dt, shape, layout)])
def test_gemm_skinny(gpu, dt, shape, lines, layout):
    _run(gpu, dt, shape, lines, layout, "gemm_skinny_kernel")


@pytest.mark.parametrize("dt,shape,lines,layout", SMALL)
def test_gemm_skinny_left_to_the_small_kernel(gpu, dt, shape, lines, layout):
    _run(gpu, dt, shape, lines, layout, "gemm_small_kernel")


def _run(lh, dt, shape, lines, layout, kernel):
    M, N, K = shape
    arow, brow, crow = bool(layout & 1), bool(layout & 2), bool(layout & 4)
    announce(f"gemm skinny {dt} layout={layout} M={M} N={N} K={K} lines={lines}: {kernel}")
    rng = np.random.default_rng(M + layout)

    def operand(rows, cols, row_major):
        """(device array, leading dimension, values in 64 bits)."""
        if dt == "i8":
            v = rng.integers(-128, 128, (rows, cols)).astype(np.int8)
            wide = v.astype(np.float64)   # exact: the sums stay below 2^53
        elif dt == "f16":
            v = rng.uniform(-1, 1, (rows, cols)).astype(np.float16)
            wide = v.astype(np.float64)
        else:
            v = (rng.uniform(-1, 1, (rows, cols)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
            wide = (v.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        v = v if row_major else v.T
        per = 128 // v.itemsize
        ld = -(-v.shape[1] // per) * per if lines else v.shape[1]
        buf = np.zeros((v.shape[0], ld), v.dtype)
        buf.view(np.uint8)[:] = 0xFF   # NaN in f16 and bf16
        buf[:, :v.shape[1]] = v
        return lh.HIPDeviceArray.from_numpy(buf, dt, order="C"), ld, wide

    A, lda, wa = operand(M, K, arow)
    B, ldb, wb = operand(K, N, brow)
    inner, pad = (N if crow else M), 3 if layout in (1, 4, 5) else 4
    C = lh.HIPDeviceArray("i32" if dt == "i8" else "f32", (M if crow else N, inner + pad), order="C")
    C.fill_bytes(0xEE)
    lh.kernel_log_clear()
    lh.gemm_raw(dt, C.dtype, A.ptr, B.ptr, C.ptr, M, N, K, lda, ldb, inner + pad, layout)
    log = [k for k in lh.kernel_log() if k not in ("splitk_sum_kernel", "fill_bytes_kernel")]   # (the workspace's first use)
    assert log == [kernel], lh.kernel_log()
    got = C.to_numpy()
    assert (np.ascontiguousarray(got[:, inner:]).view(np.uint8) == 0xEE).all(), "C's padding was written"
    got = got[:, :inner] if crow else got[:, :inner].T
    want = wa @ wb
    if dt == "i8":
        np.testing.assert_array_equal(got, want.astype(np.int64))
    else:
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert err <= math.sqrt(K) * 2.0 ** -23, err
