"""GEMM operands of any alignment, leading dimension and extent, on the kernels' any-alignment forms:
rows that start at every byte (element) of a 16-byte chunk, K, M and N that split one, K ranges of the
split product, and nothing read past a row's end (the padding holds NaN, or 255 for the integers).  A K too
short for the automatic choice to take unsigned bytes there runs with the small-product kernel pinned; and the
products on both sides of that rule.
Reference: numpy in 64 bits.  Floating tolerance: fp32 sums of K terms, each step's relative rounding
at most 2^-23, random over the terms: sqrt(K) 2^-23 (7.7e-6 at the largest K here)."""
import math

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

NP = {"f16": np.float16, "bf16": np.uint16, "i8": np.int8, "u8": np.uint8}
ACC = {"f16": "f32", "bf16": "f32", "i8": "i32", "u8": "u32"}


def _operand(lh, rng, dt, rows, cols, row_major, pad, shift):
    """(device array holding the operand, its address, leading dimension, values in 64 bits)."""
    outer, inner = (rows, cols) if row_major else (cols, rows)
    ld = inner + pad
    if dt in ("i8", "u8"):
        info = np.iinfo(NP[dt])
        vals = rng.integers(info.min, info.max + 1, (outer, inner)).astype(NP[dt])
        wide = vals.astype(np.int64)
    else:
        x = rng.uniform(-1, 1, (outer, inner)).astype(np.float32)
        if dt == "f16":
            vals = x.astype(np.float16)
            wide = vals.astype(np.float64)
        else:
            vals = (x.view(np.uint32) >> 16).astype(np.uint16)
            wide = (vals.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    buf = np.full(shift + (outer - 1) * ld + inner, 0, NP[dt])
    buf.view(np.uint8)[:] = 0xFF   # NaN in f16 and bf16
    at = shift + np.arange(outer)[:, None] * ld + np.arange(inner)[None, :]
    buf[at] = vals
    dev = lh.HIPDeviceArray.from_numpy(buf, dt)
    return dev, dev.pointer(1 + shift), ld, wide if row_major else wide.T


@pytest.fixture
def pin_gemm(gpu):
    yield lambda choice: gpu.set_kernel_override(gpu.FAMILY_GEMM, choice)
    gpu.set_kernel_override(gpu.FAMILY_GEMM, 0)


@pytest.mark.parametrize("layout", range(8))
@pytest.mark.parametrize("dt", ["f16", "bf16", "i8", "u8"])
@pytest.mark.parametrize("shape", [(16, 16, 16), (17, 31, 23), (64, 65, 257), (129, 63, 513), (70, 33, 4099)])
def test_gemm_any_alignment(gpu, pin_gemm, dt, layout, shape):
    if dt == "u8" and shape[2] <= 28:
        pin_gemm(2)
    _run(gpu, dt, layout, shape, "gemm_small_kernel<u8,any>" if dt == "u8" else "gemm_small_kernel<any>")


@pytest.mark.parametrize("dt,layout,shape,kernel", [
    ("f16", 5, (1025, 1031, 32), "gemm_staged_kernel"), ("f16", 5, (1025, 1031, 33), "gemm_small_kernel<any>"),
    ("bf16", 2, (1025, 1031, 17), "gemm_staged_kernel"), ("bf16", 0, (1019, 1023, 31), "gemm_small_kernel<any>"),
    ("i8", 5, (1025, 1031, 17), "gemm_small_kernel<any>"), ("u8", 5, (50, 70, 28), "gemm_u8_generic_kernel"),
    ("u8", 1, (510, 509, 17), "gemm_u8_generic_kernel"), ("u8", 5, (50, 70, 29), "gemm_small_kernel<u8,any>"),
    ("u8", 7, (50, 70, 20), "gemm_small_kernel<u8,any>"), ("u8", 1, (520, 520, 17), "gemm_small_kernel<u8,any>")])
def test_gemm_any_short_k(gpu, dt, layout, shape, kernel):
    """The automatic choice on both sides of its bounds on K and on the tiles."""
    _run(gpu, dt, layout, shape, kernel)


def _run(lh, dt, layout, shape, kernel):
    M, N, K = shape
    for pad, shift in ((0, 0), (1, 1), (3, 5)):
        announce(f"gemm any {dt} layout={layout} M={M} N={N} K={K} pad={pad} shift={shift}")
        rng = np.random.default_rng(1000 * layout + M + pad)
        A, pa, lda, wa = _operand(lh, rng, dt, M, K, layout & 1, pad, shift)
        B, pb, ldb, wb = _operand(lh, rng, dt, K, N, layout & 2, pad, shift)
        crow = bool(layout & 4)
        ldc = (N if crow else M) + pad
        C = lh.HIPDeviceArray(ACC[dt], (ldc, M if crow else N))
        C.fill_bytes(0xEE)
        lh.kernel_log_clear()
        lh.gemm_raw(dt, ACC[dt], pa, pb, C.ptr, M, N, K, lda, ldb, ldc, layout)
        if pad:
            assert kernel in lh.kernel_log(), lh.kernel_log()
        got = C.to_numpy().T
        inner = N if crow else M
        assert (got[:, inner:].copy().view(np.uint8) == 0xEE).all(), "C's padding was written"
        got = got[:, :inner] if crow else got[:, :inner].T
        if dt in ("i8", "u8"):
            want = (wa @ wb) & 0xFFFFFFFF
            np.testing.assert_array_equal(got.astype(np.int64) & 0xFFFFFFFF, want)
        else:
            want = wa @ wb
            err = np.linalg.norm(got - want) / np.linalg.norm(want)
            assert err <= math.sqrt(K) * 2.0 ** -23, err


@pytest.mark.parametrize("layout", [0, 3, 5, 7])
def test_gemm_ex_any_alignment(gpu, layout):
    """The fused epilogue on unaligned operands: bias, residual and relu into f32."""
    lh = gpu
    M, N, K = 75, 133, 300
    announce(f"gemm_ex any layout={layout}")
    rng = np.random.default_rng(7 + layout)
    A, pa, lda, wa = _operand(lh, rng, "f16", M, K, layout & 1, 1, 3)
    B, pb, ldb, wb = _operand(lh, rng, "f16", K, N, layout & 2, 1, 1)
    crow = bool(layout & 4)
    order = "C" if crow else "F"
    bias = rng.standard_normal(M).astype(np.float32)
    res = rng.standard_normal((M, N)).astype(np.float32)
    D = lh.HIPDeviceArray("f32", (M, N), order=order)
    dres = lh.HIPDeviceArray.from_numpy(res, "f32", order=order)
    dbias = lh.HIPDeviceArray.from_numpy(bias, "f32")
    lh.kernel_log_clear()
    ld = N if crow else M
    lh.gemm_ex_raw("f16", "f32", pa, pb, D.ptr, M, N, K, lda, ldb, ld, layout, dbias.ptr, dres.ptr, ld, "relu")
    assert lh.kernel_log() == ["gemm_small_kernel", "gemm_small_kernel<any>"], lh.kernel_log()
    want = np.maximum(wa @ wb + bias[:, None].astype(np.float64) + res, 0)
    err = np.linalg.norm(D.to_numpy() - want) / np.linalg.norm(want)
    assert err <= math.sqrt(K) * 2.0 ** -23, err
