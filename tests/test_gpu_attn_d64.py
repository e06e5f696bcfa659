"""Attention at D = 56 and 64 on the kernel that keeps both products in one wavefront: grids that give its
64-query groups (many heads) and its 32-query ones (few), for each an odd number of key blocks (the last step
half empty), ragged and whole, and an even one, S at the edges of a block, scales that keep the running maximum still and that move it, strided rows, O rows
8-byte aligned.  The wide causal grids near S = 2200 lie within the rule's 4 % margin and keep the score/output
kernel; those above 4096 leave it.  Reference: softmax in 64 bits; bar: the attention configurations' relative Frobenius
error of 2e-3 (fp16 probabilities and result, 2^-11 each)."""
import math

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("E,L,H,B,scale,pad", [
    (64, 1025, 4, 1, None, 0), (64, 1152, 3, 2, 0.6, 0), (56, 1313, 4, 1, None, 8), (64, 1089, 2, 1, 0.02, 4),
    (64, 2176, 36, 4, None, 0), (56, 2113, 32, 5, 0.5, 8), (64, 2300, 30, 5, 0.6, 4),
    (64, 4161, 32, 4, None, 0), (56, 4480, 30, 5, 0.5, 8), (64, 4607, 28, 5, 0.6, 4),
    (64, 4133, 32, 4, 0.6, 4), (64, 4160, 32, 4, None, 0)])
def test_flash_d64_one_wavefront(gpu, E, L, H, B, scale, pad, causal):
    lh = gpu
    announce(f"flash D={E} one wavefront S={L} H={H} B={B} scale={scale} pad={pad} causal={causal}")
    Q, K, V = (lh.HIPDeviceArray("f16", (E + 8, L, H, B)) for _ in range(3))   # rows E + 8 apart
    for t, a in enumerate((Q, K, V)):
        lh.fill_normal(a, lh.seed(31, t))
    O = lh.HIPDeviceArray("f16", (E + pad, L, H, B))
    O.fill_bytes(0xFF)
    sc = 1 / math.sqrt(E) if scale is None else scale
    lh.kernel_log_clear()
    lh.flash_attn_fwd_raw(Q.ptr, K.ptr, V.ptr, O.ptr, B, H, L, E, Q.strides(), O.strides(), sc, causal)
    if causal and 2000 < L < 2400:   # estimated at 0.976 to 0.98 of the score/output kernel's time
        kernel = ["flash_fwd5_kernel"]
    else:
        kernel = ["flash_fwd6_kernel"] if H * B > 100 else ["flash_fwd6_kernel", "flash_fwd6_kernel<32>"]
    assert lh.kernel_log() == kernel, lh.kernel_log()
    q, k, v, got = (a.to_numpy() for a in (Q, K, V, O))
    assert not np.isnan(got[:E].astype(np.float32)).any()
    assert (np.ascontiguousarray(got[E:]).view(np.uint16) == 0xFFFF).all(), "row padding of O written"
    for h, b in {(0, 0), (H - 1, B - 1), (H // 2, B // 2)}:
        s = q[:E, :, h, b].T.astype(np.float64) @ k[:E, :, h, b].astype(np.float64) * sc
        if causal:
            s = np.where(np.tril(np.ones((L, L), bool)), s, -np.inf)
        p = np.exp(s - s.max(axis=1, keepdims=True))
        want = (p / p.sum(axis=1, keepdims=True)) @ v[:E, :, h, b].T.astype(np.float64)
        err = np.linalg.norm(got[:E, :, h, b].T - want) / np.linalg.norm(want)
        assert err <= 2e-3, (h, b, err)
