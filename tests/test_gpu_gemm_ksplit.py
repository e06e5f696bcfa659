"""The K-split form of the mid-size kernel, through the automatic choice: every operand layout and C
order, whole and ragged tiles, an even and an odd number of 128-byte units of K (the last pass half
empty) and a ragged last unit, padded rows of C.  Reference: numpy in 64 bits (integers exactly);
floating tolerance: fp32 sums of K terms, each step's relative rounding at most 2^-23, random over the
terms: sqrt(K) 2^-23."""
import math

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


KSPLIT = ["gemm_mid_kernel", "gemm_mid_ksplit_kernel"]


# the last two have fewer than 128 tiles: on padded rows of whole 128-byte lines
@pytest.mark.parametrize("layout", range(8))
@pytest.mark.parametrize("dt,shape", [
    ("bf16", (2048, 1024, 2048)), ("f16", (1168, 2008, 2112)), ("f16", (1088, 2192, 2120)),
    ("bf16", (528, 2824, 4168)), ("i8", (2048, 1024, 4096)), ("i8", (1168, 2032, 4240)), ("i8", (592, 2064, 8336))])
def test_gemm_mid_ksplit(gpu, dt, shape, layout):
    _run(gpu, dt, shape, layout, shape[0] in (528, 592), KSPLIT)


@pytest.mark.parametrize("dt,shape,layout", [("bf16", (528, 2824, 4168), 5), ("bf16", (528, 2824, 4168), 0),
                                             ("f16", (512, 3072, 8200), 1), ("i8", (592, 2064, 8336), 7)])
def test_gemm_mid_ksplit_left_to_the_small_kernel(gpu, dt, shape, layout):
    """Fewer than 128 tiles and K-contiguous rows that cross 128-byte lines: both operands', or one's with a K
    below 12288 bytes."""
    _run(gpu, dt, shape, layout, False, ["gemm_small_kernel"])


def _run(lh, dt, shape, layout, lines, kernel):
    M, N, K = shape
    announce(f"gemm K-split {dt} layout={layout} M={M} N={N} K={K} lines={lines}")
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

    A, lda, wa = operand(M, K, layout & 1)
    B, ldb, wb = operand(K, N, layout & 2)
    crow = bool(layout & 4)
    inner, pad = (N if crow else M), 3 if layout in (3, 4) else 4
    C = lh.HIPDeviceArray("i32" if dt == "i8" else "f32", (M if crow else N, inner + pad), order="C")
    C.fill_bytes(0xEE)
    lh.kernel_log_clear()
    lh.gemm_raw(dt, C.dtype, A.ptr, B.ptr, C.ptr, M, N, K, lda, ldb, inner + pad, layout)
    assert lh.kernel_log() == kernel, lh.kernel_log()
    got = C.to_numpy()
    assert (np.ascontiguousarray(got[:, inner:]).view(np.uint8) == 0xEE).all(), "C's padding was written"
    got = got[:, :inner] if crow else got[:, :inner].T
    want = wa @ wb
    if dt == "i8":
        np.testing.assert_array_equal(got, want.astype(np.int64))
    else:
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert err <= math.sqrt(K) * 2.0 ** -23, err
