"""W8A16 batches on the tiled kernel: both tiles, ragged rows and columns, one, an even and an odd
number of 128-k stages with partial last ones, X and Y in either order (X also copied row-major first),
padded leading dimensions.  Reference: numpy in 64 bits; tolerance: fp32 sums of K terms, each step's
relative rounding at most 2^-23, random over the terms: sqrt(K) 2^-23."""
import math

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,xo,yo,pad,bn", [
    (65, 4128, 128, "C", "C", 0, 64), (128, 5001, 144, "C", "F", 0, 64), (129, 4097, 272, "C", "C", 16, 64),
    (72, 4160, 1040, "F", "F", 0, 64), (65, 4130, 400, "F", "C", 0, 64), (200, 2084, 16, "F", "C", 0, 64),
    (256, 8321, 144, "C", "C", 0, 128), (136, 8330, 272, "F", "F", 0, 128), (250, 8320, 1040, "C", "F", 16, 128),
    (255, 8448, 128, "F", "C", 0, 128)])
def test_w8a16_tiled(gpu, M, N, K, xo, yo, pad, bn):
    lh = gpu
    announce(f"w8a16 tiled M={M} N={N} K={K} X {xo} Y {yo} pad={pad}")
    rng = np.random.default_rng(M + N + K)
    x = rng.standard_normal((M, K)).astype(np.float16)
    w = rng.integers(-128, 128, (K, N)).astype(np.int8)
    s = rng.uniform(0.001, 0.02, N).astype(np.float16)
    ldx = (K if xo == "C" else M) + (pad if xo == "C" else 0)
    xbuf = np.full((M if xo == "C" else K, ldx), np.nan, np.float16)   # NaN in the padding
    xbuf[:, :K if xo == "C" else M] = x if xo == "C" else x.T
    X = lh.HIPDeviceArray.from_numpy(xbuf, "f16", order="C")
    wbuf = np.full((N, K + pad), 127, np.int8)
    wbuf[:, :K] = w.T
    W = lh.HIPDeviceArray.from_numpy(wbuf, "i8", order="C")
    S = lh.HIPDeviceArray.from_numpy(s, "f16")
    ldy = (N if yo == "C" else M) + pad
    Y = lh.HIPDeviceArray("f32", (M if yo == "C" else N, ldy), order="C")
    Y.fill_bytes(0xEE)
    layout = (1 if xo == "C" else 0) | (4 if yo == "C" else 0)
    lh.kernel_log_clear()
    lh.w8a16_raw(X.ptr, W.ptr, S.ptr, Y.ptr, M, N, K, ldx, K + pad, ldy, layout)
    assert f"w8a16_batch_kernel<128,{bn}>" in lh.kernel_log(), lh.kernel_log()
    got = Y.to_numpy()
    inner = N if yo == "C" else M
    assert (np.ascontiguousarray(got[:, inner:]).view(np.uint8) == 0xEE).all(), "Y's padding was written"
    got = got[:, :inner] if yo == "C" else got[:, :inner].T
    want = (x.astype(np.float64) @ w.astype(np.float64)) * s.astype(np.float64)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= math.sqrt(K) * 2.0 ** -23, err
