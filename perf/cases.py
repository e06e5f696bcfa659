"""The work that a user of lava_hip has it do, as cases that can be timed.

A case is one call of a public entry point (GEMM, GEMM with the fused epilogue, W8A16 GEMM, flash
attention) on operands that the caller's program already holds on the GPU, output buffer included,
as with the destination-first calls of the package.  `listed()` names the twelve that stand for the
range, `draw()` takes others from it.

Matrices are torch tensors whose shape is the storage order: (rows, cols) for a row-major operand,
(cols, rows) for a column-major one, packed.  Attention tensors are (B, H, S, D) ("bhsd") or
(B, S, H, D) ("bshd"), the head dimension contiguous either way.
"""
import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "lava.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

import lava_hip as lh  # noqa: E402

_TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32, "i8": torch.int8, "u8": torch.uint8}
# uint32 words are held as int32: the sums of these sizes stay below 2^31
_ACC = {"f16": ("f32", torch.float32), "bf16": ("f32", torch.float32), "i8": ("i32", torch.int32),
        "u8": ("u32", torch.int32)}
_BYTES = {"f16": 2, "bf16": 2, "f32": 4, "i8": 1, "u8": 1}
A_ROW, B_ROW, C_ROW = 1, 2, 4   # layout bits; 0 is all column-major, Julia's default


def listed():
    return [
        # the smallest product of the benchmark: a tile-sized call where launch latency is all there is
        {"name": "gemm_f16_256", "op": "gemm", "dtype": "f16", "M": 256, "N": 256, "K": 256, "layout": 7},
        # an ordinary square product in Julia's own storage order, too small to fill the chip with large tiles
        {"name": "gemm_bf16_2048_colmajor", "op": "gemm", "dtype": "bf16", "M": 2048, "N": 2048, "K": 2048,
         "layout": 0},
        # the largest product of the benchmark
        {"name": "gemm_bf16_8192", "op": "gemm", "dtype": "bf16", "M": 8192, "N": 8192, "K": 8192, "layout": 5},
        # the int8 product of the benchmark, bit-exact
        {"name": "gemm_i8_4096", "op": "gemm", "dtype": "i8", "M": 4096, "N": 4096, "K": 4096, "layout": 5},
        # a projection of a batch of 64 decoded tokens: skinny, bound by the weights
        {"name": "gemm_bf16_decode64", "op": "gemm", "dtype": "bf16", "M": 64, "N": 14336, "K": 4096, "layout": 5},
        # extents that nobody rounded (a packed column-major array of odd height): no row is 16-byte aligned
        {"name": "gemm_f16_odd", "op": "gemm", "dtype": "f16", "M": 1111, "N": 1333, "K": 777, "layout": 0},
        # a layer of an MLP, features by tokens as in Julia: bias per feature, residual, gelu, narrowed result
        {"name": "gemm_ex_bf16_mlp", "op": "gemm_ex", "dtype": "bf16", "out": "bf16", "M": 4096, "N": 2048, "K": 4096,
         "layout": 0, "bias": True, "residual": True, "act": "gelu_tanh"},
        # the decode shape of the benchmark: weights streamed once for 16 rows
        {"name": "w8a16_decode16", "op": "w8a16", "M": 16, "N": 14336, "K": 4096, "layout": 5},
        # the same weights for a large batch, the largest whose row blocks the tests go through
        {"name": "w8a16_batch256", "op": "w8a16", "M": 256, "N": 14336, "K": 4096, "layout": 5},
        # the attention of the benchmark: long causal prefill
        {"name": "attn_causal_4096", "op": "attn", "B": 4, "H": 32, "S": 4096, "D": 128, "causal": True,
         "order": "bhsd"},
        # an encoder's attention: short ragged sequences, not causal, D = 64, heads interleaved
        {"name": "attn_encoder_777", "op": "attn", "B": 4, "H": 12, "S": 777, "D": 64, "causal": False,
         "order": "bshd"},
        # one prompt's prefill: a single sequence of an odd length
        {"name": "attn_prompt_1537", "op": "attn", "B": 1, "H": 32, "S": 1537, "D": 128, "causal": True,
         "order": "bhsd"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _to(n, step):
    return max(step, n // step * step)


def draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "gemm_ex", "w8a16", "w8a16", "attn", "attn", "attn"])
    if op in ("gemm", "gemm_ex"):
        dtype = rng.choice(["f16", "bf16", "f16", "bf16", "i8", "u8"] if op == "gemm" else ["f16", "bf16"])
        odd = dtype != "u8" and rng.random() < 0.3
        top = 1536 if odd else 8192 if op == "gemm" else 4096
        dims = [_log(rng, 16, top) for _ in range(3)]
        if not odd:   # sizes that a program chose: multiples of 16, larger ones of 64
            dims = [_to(n, 64 if n >= 512 else 16) for n in dims]
        case = {"op": op, "dtype": dtype, "M": dims[0], "N": dims[1], "K": dims[2], "layout": rng.randrange(8)}
        if op == "gemm_ex":
            case.update(out=rng.choice(["f32", "f16", "bf16"]), bias=rng.random() < 0.8, residual=rng.random() < 0.5,
                        act=rng.choice(["none", "relu", "gelu_tanh", "gelu_erf"]))
        return case
    if op == "w8a16":
        layout = rng.choice([5, 5, 0, 7])
        n = _log(rng, 256, 16384)
        return {"op": op, "M": _log(rng, 1, 256), "N": n if rng.random() < 0.2 and not layout & B_ROW else _to(n, 32),
                "K": _to(_log(rng, 256, 14336), 32), "layout": layout}
    case = {"op": op, "B": rng.randint(1, 4), "H": rng.choice([1, 4, 8, 12, 16, 32]), "S": _log(rng, 16, 4096),
            "D": rng.choice([32, 64, 64, 80, 96, 128, 128, 128, 256]), "causal": rng.random() < 0.6,
            "order": rng.choice(["bhsd", "bhsd", "bshd"])}
    while _attn_flops(case) > 3e11:   # the largest listed call's time, at the rate of the slowest head size
        case["S"] = case["S"] * 3 // 4
    return case


def _attn_flops(case):
    s = case["S"]
    pairs = s * (s + 1) / 2 if case["causal"] else s * s
    return 4.0 * case["B"] * case["H"] * pairs * case["D"]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _matrix(gen, rows, cols, row_major, dtype):
    shape = (rows, cols) if row_major else (cols, rows)
    if dtype == "i8":
        return torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=gen)
    if dtype == "u8":
        return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen)
    x = torch.rand(shape, dtype=torch.float32, device="cuda", generator=gen)
    return x.mul_(2).sub_(1).to(_TORCH[dtype])


def _inputs(case, seed):
    g = _gen(seed)
    if case["op"] == "attn":
        shape = _attn_shape(case)
        return {n: torch.randn(shape, dtype=torch.float32, device="cuda", generator=g).to(torch.float16) for n in "QKV"}
    M, N, K, lay = case["M"], case["N"], case["K"], case["layout"]
    if case["op"] == "w8a16":
        return {"X": torch.randn((M, K) if lay & A_ROW else (K, M), dtype=torch.float32, device="cuda",
                                 generator=g).to(torch.float16),
                "W": torch.randint(-127, 128, (K, N) if lay & B_ROW else (N, K), dtype=torch.int8, device="cuda",
                                   generator=g),
                "scale": torch.rand(N, device="cuda", generator=g).mul_(0.019).add_(0.001).to(torch.float16)}
    got = {"A": _matrix(g, M, K, lay & A_ROW, case["dtype"]), "B": _matrix(g, K, N, lay & B_ROW, case["dtype"])}
    if case["op"] == "gemm_ex":
        got["bias"] = torch.randn(M, device="cuda", generator=g) if case["bias"] else None
        got["residual"] = (torch.randn((M, N) if lay & C_ROW else (N, M), device="cuda", generator=g)
                           if case["residual"] else None)
    return got


def _attn_shape(case):
    b, h, s, d = case["B"], case["H"], case["S"], case["D"]
    return (b, h, s, d) if case["order"] == "bhsd" else (b, s, h, d)


def _attn_strides(case):
    """Element strides of (D, S, H, B)."""
    h, s, d = case["H"], case["S"], case["D"]
    return (1, d, s * d, h * s * d) if case["order"] == "bhsd" else (1, h * d, d, s * h * d)


def prepare(case, seed):
    lh.init()
    state = {"case": case, **_inputs(case, seed)}
    if case["op"] == "attn":
        state["out"] = torch.empty(_attn_shape(case), dtype=torch.float16, device="cuda")
        state["strides"] = _attn_strides(case)
    else:
        shape = (case["M"], case["N"]) if case["layout"] & C_ROW else (case["N"], case["M"])
        dtype = {"gemm": lambda: _ACC[case["dtype"]][1], "gemm_ex": lambda: _TORCH[case["out"]],
                 "w8a16": lambda: torch.float32}[case["op"]]()
        state["out"] = torch.empty(shape, dtype=dtype, device="cuda")
    return state


def run(state):
    case, out = state["case"], state["out"]
    stream = torch.cuda.current_stream().cuda_stream
    op = case["op"]
    if op == "attn":
        lh.flash_attn_fwd_raw(state["Q"].data_ptr(), state["K"].data_ptr(), state["V"].data_ptr(), out.data_ptr(),
                              case["B"], case["H"], case["S"], case["D"], state["strides"], causal=case["causal"],
                              stream=stream)
        return out
    M, N, K, lay = case["M"], case["N"], case["K"], case["layout"]
    lda, ldb, ldc = K if lay & A_ROW else M, N if lay & B_ROW else K, N if lay & C_ROW else M
    if op == "w8a16":
        lh.w8a16_raw(state["X"].data_ptr(), state["W"].data_ptr(), state["scale"].data_ptr(), out.data_ptr(), M, N, K,
                     lda, ldb, ldc, lay, stream)
    elif op == "gemm":
        lh.gemm_raw(case["dtype"], _ACC[case["dtype"]][0], state["A"].data_ptr(), state["B"].data_ptr(),
                    out.data_ptr(), M, N, K, lda, ldb, ldc, lay, stream)
    else:
        bias, res = state["bias"], state["residual"]
        lh.gemm_ex_raw(case["dtype"], case["out"], state["A"].data_ptr(), state["B"].data_ptr(), out.data_ptr(), M, N,
                       K, lda, ldb, ldc, lay, bias.data_ptr() if bias is not None else 0,
                       res.data_ptr() if res is not None else 0, ldc, case["act"], stream)
    return out


def work(case):
    if case["op"] == "attn":
        return {"bytes": 4 * 2 * case["B"] * case["H"] * case["S"] * case["D"], "flops": _attn_flops(case)}
    M, N, K = case["M"], case["N"], case["K"]
    flops = 2.0 * M * N * K
    if case["op"] == "w8a16":
        return {"bytes": 2 * M * K + K * N + 2 * N + 4 * M * N, "flops": flops}
    got = _BYTES[case["dtype"]] * (M * K + K * N)
    if case["op"] == "gemm":
        return {"bytes": got + 4 * M * N, "flops": flops}
    got += _BYTES[case["out"]] * M * N + 4 * M * case["bias"] + 4 * M * N * case["residual"]
    return {"bytes": got, "flops": flops}


def tolerance(case):
    if case["op"] == "gemm" and case["dtype"] in ("i8", "u8"):
        return "exact"
    if case["op"] == "attn":
        # fp16 result and fp16 probabilities
        return {"rel": 1.5e-3, "max": 0.03}
    if case["op"] == "gemm_ex" and case["out"] != "f32":
        # one rounding to the result's type
        return {"rel": 7e-3, "max": 0.02} if case["out"] == "bf16" else {"rel": 1e-3, "max": 3e-3}
    # fp32 sums in another order
    return {"rel": 2e-6, "max": 4e-5}


def exact(case, seed):
    x = _inputs(case, seed)
    if case["op"] == "attn":
        return _exact_attn(case, x)
    lay = case["layout"]

    def matrix(name, row_major):
        return x[name].double() if row_major else x[name].double().t()

    if case["op"] == "w8a16":
        c = (matrix("X", lay & A_ROW) @ matrix("W", lay & B_ROW)) * x["scale"].double()[None, :]
    else:
        c = matrix("A", lay & A_ROW) @ matrix("B", lay & B_ROW)
    if case["op"] == "gemm_ex":
        if x["bias"] is not None:
            c = c + x["bias"].double()[:, None]
        if x["residual"] is not None:
            c = c + matrix("residual", lay & C_ROW)
        if case["act"] == "relu":
            c = c.clamp_min(0)
        elif case["act"] == "gelu_tanh":
            c = 0.5 * c * (1 + torch.tanh(math.sqrt(2 / math.pi) * (c + 0.044715 * c ** 3)))
        elif case["act"] == "gelu_erf":
            c = 0.5 * c * (1 + torch.erf(c / math.sqrt(2)))
    c = (c if lay & C_ROW else c.t()).contiguous()
    return c.to(torch.int32) if case["op"] == "gemm" and case["dtype"] in ("i8", "u8") else c


def _exact_attn(case, x):
    b, h, s, d = case["B"], case["H"], case["S"], case["D"]
    out = torch.empty(_attn_shape(case), dtype=torch.float64, device="cuda")
    keep = torch.ones(s, s, dtype=torch.bool, device="cuda").tril() if case["causal"] else None
    for i in range(b):
        for j in range(h):
            at = (i, j) if case["order"] == "bhsd" else (i, slice(None), j)
            q, k, v = (x[n][at].double().contiguous() for n in "QKV")
            p = (q @ k.t().contiguous()) / math.sqrt(d)
            if keep is not None:
                p = p.masked_fill(~keep, -math.inf)
            out[at] = torch.softmax(p, dim=-1) @ v
    return out
