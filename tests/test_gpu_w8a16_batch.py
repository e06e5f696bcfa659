"""W8A16 batches on the tiled kernel: both tiles, ragged rows and columns, one, an even and an odd
number of 128-k stages with partial last ones, X and Y in either order (X also copied row-major first),
padded leading dimensions; and the batches that its rule leaves to the streaming kernel.  Reference: numpy in 64 bits; tolerance: fp32 sums of K terms, each step's
relative rounding at most 2^-23, random over the terms: sqrt(K) 2^-23."""
import math

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,xo,yo,pad,bn", [
    (65, 8224, 128, "C", "C", 0, 64), (128, 8201, 144, "C", "F", 0, 64), (129, 5601, 272, "C", "C", 16, 64),
    (72, 4160, 1040, "F", "F", 0, 64), (65, 8226, 400, "F", "C", 0, 64), (200, 4132, 16, "F", "C", 0, 64),
    (70, 4130, 1552, "C", "C", 16, 64), (256, 8321, 144, "C", "C", 0, 128), (136, 8330, 272, "F", "F", 0, 128),
    (250, 8320, 1040, "C", "F", 16, 128), (255, 8448, 128, "F", "C", 0, 128)])
def test_w8a16_tiled(gpu, M, N, K, xo, yo, pad, bn):
    _run(gpu, M, N, K, xo, yo, pad, f"w8a16_batch_kernel<128,{bn}>")


@pytest.mark.parametrize("M,N,K,xo", [(65, 4128, 128, "C"), (129, 4097, 272, "C"), (72, 4160, 1008, "F"),
                                      (128, 5001, 1520, "C"), (65, 4130, 1040, "F"), (128, 4096, 2048, "C")])
def test_w8a16_left_to_the_streaming_kernel(gpu, M, N, K, xo):
    """At most 512 blocks of 64 x 32 and a K too short for the tiles, or at most 256 blocks."""
    _run(gpu, M, N, K, xo, "C", 0, "w8a16_kmajor_kernel<mb4>")


def _run(lh, M, N, K, xo, yo, pad, kernel):
    announce(f"w8a16 batch M={M} N={N} K={K} X {xo} Y {yo} pad={pad}: {kernel}")
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
    assert kernel in lh.kernel_log(), lh.kernel_log()
    got = Y.to_numpy()
    inner = N if yo == "C" else M
    assert (np.ascontiguousarray(got[:, inner:]).view(np.uint8) == 0xEE).all(), "Y's padding was written"
    got = got[:, :inner] if yo == "C" else got[:, :inner].T
    want = (x.astype(np.float64) @ w.astype(np.float64)) * s.astype(np.float64)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= math.sqrt(K) * 2.0 ** -23, err
