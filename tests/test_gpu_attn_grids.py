"""Both widths of the score/output attention kernel: grids that give its 64-query pairs (many heads)
and its 32-query ones (few), with S at the edges of a key block, a 128- and a 256-query workgroup.
Reference: softmax in 64 bits; bar: the attention configurations' relative Frobenius error of 2e-3
(fp16 probabilities and result, 2^-11 each)."""
import math

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def _kernel(E, L, heads):
    """The log of the width that the rule takes: 64-query pairs where many heads fill the CUs with them
    (a sequence of at most 128 has no use for more than one 128-query workgroup a head)."""
    if E == 64 and heads == 3 and L == 321:   # few heads, more than two key blocks a wavefront
        return ["flash_fwd6_kernel", "flash_fwd6_kernel<32>"]
    wide = heads > 256 and L > 128
    return ["flash_fwd5_kernel"] if wide else ["flash_fwd5_kernel", "flash_fwd5_kernel<32>"]


@pytest.mark.parametrize("E,L,H,B,kernel", [
    (32, 1300, 16, 3, ["flash_fwd5_kernel"]), (128, 380, 32, 4, ["flash_fwd5_kernel"]),
    (80, 1289, 16, 3, ["flash_fwd5_kernel"]), (128, 1537, 32, 1, ["flash_fwd5_kernel", "flash_fwd5_kernel<32>"]),
    (96, 513, 16, 2, ["flash_fwd5_kernel", "flash_fwd5_kernel<32>"])])
def test_flash_width_near_the_rule(gpu, E, L, H, B, kernel):
    """Causal grids on both sides of the margin: estimated at 0.95 to 0.96 of the wide pairs' time, and well
    below it."""
    _run(gpu, E, L, H, B, True, kernel)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("H,B", [(32, 16), (3, 1)])
@pytest.mark.parametrize("E", [32, 64, 80, 128])
@pytest.mark.parametrize("L", [1, 33, 64, 97, 129, 192, 256, 321])
def test_flash_both_widths(gpu, E, L, H, B, causal):
    _run(gpu, E, L, H, B, causal, _kernel(E, L, H * B))


def _run(lh, E, L, H, B, causal, kernel):
    announce(f"flash widths D={E} S={L} H={H} B={B} causal={causal}")
    rng = np.random.default_rng(E + L + H)
    q, k, v = (np.asfortranarray(rng.standard_normal((E, L, H, B)).astype(np.float16)) for _ in range(3))
    Q, K, V = (lh.HIPDeviceArray.from_numpy(t, "f16") for t in (q, k, v))
    O = lh.HIPDeviceArray("f16", (E, L, H, B))
    O.fill_bytes(0xFF)
    lh.kernel_log_clear()
    lh.flash_attn_fwd(O, Q, K, V, causal=causal)
    assert lh.kernel_log() == kernel, lh.kernel_log()
    got = O.to_numpy()
    assert not np.isnan(got).any()
    for h, b in {(0, 0), (H - 1, B - 1), (H // 2, B // 2)}:
        s = q[:, :, h, b].T.astype(np.float64) @ k[:, :, h, b].astype(np.float64) / math.sqrt(E)
        if causal:
            s = np.where(np.tril(np.ones((L, L), bool)), s, -np.inf)
        p = np.exp(s - s.max(axis=1, keepdims=True))
        want = (p / p.sum(axis=1, keepdims=True)) @ v[:, :, h, b].T.astype(np.float64)
        err = np.linalg.norm(got[:, :, h, b].T - want) / np.linalg.norm(want)
        assert err <= 2e-3, (h, b, err)


@pytest.mark.parametrize("H,B", [(32, 16), (3, 1)])
@pytest.mark.parametrize("low", [1.75, 0.9375])
@pytest.mark.parametrize("E", [32, 128])
def test_flash_scores_near_the_lowest(gpu, E, low, H, B):
    """Every score -57328 (-30712) in base 2, halfway between two fp16 numbers 32 (16) apart: all keys weigh the
    same, and the result is the mean of V, not what an fp16 maximum 16 below the scores would make of it."""
    lh, L = gpu, 321
    announce(f"flash low scores D={E} low={low} H={H} B={B}")
    q, k = (np.zeros((E, L, H, B), np.float16, order="F") for _ in range(2))
    q[0], k[0] = low, -65504
    q[1], k[1] = 1, -24 if low == 1.75 else -14   # base 2: -65504 low / 2 + k[1] / 2
    v = np.asfortranarray(np.random.default_rng(E).standard_normal((E, L, H, B)).astype(np.float16))
    Q, K, V = (lh.HIPDeviceArray.from_numpy(t, "f16") for t in (q, k, v))
    O = lh.HIPDeviceArray("f16", (E, L, H, B))
    lh.kernel_log_clear()
    lh.flash_attn_fwd_raw(Q.ptr, K.ptr, V.ptr, O.ptr, B, H, L, E, Q.strides(), O.strides(), 0.5 * math.log(2), False)
    assert lh.kernel_log() == _kernel(E, L, H * B), lh.kernel_log()
    got = O.to_numpy().astype(np.float64)
    want = np.broadcast_to(v.astype(np.float64).mean(axis=1, keepdims=True), got.shape)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= 2e-3, err
