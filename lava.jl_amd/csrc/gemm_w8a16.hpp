// gemm_w8a16.hpp -- what the W8A16 kernels share (internal).
#pragma once
#include <hip/hip_runtime.h>

#include "lava_coopmat.hpp"

namespace lava {

// 8 int8 weights (two dwords, k ascending) -> the 8 fp16 values of a B operand: the byte
// (w ^ 0x80) under the high byte 0x64 is the fp16 value 1152 + w, then subtract 1152 (exact).
__device__ __forceinline__ f16x8 w8_dequant(uint32_t lo, uint32_t hi) {
    const uint32_t x0 = lo ^ 0x80808080u, x1 = hi ^ 0x80808080u;
    // bytes 0-3 of the selector's source pair are the 0x64 register, 4-7 the weights
    uint4 v;
    v.x = __builtin_amdgcn_perm(x0, 0x64646464u, 0x00050004u);
    v.y = __builtin_amdgcn_perm(x0, 0x64646464u, 0x00070006u);
    v.z = __builtin_amdgcn_perm(x1, 0x64646464u, 0x00050004u);
    v.w = __builtin_amdgcn_perm(x1, 0x64646464u, 0x00070006u);
    const f16x8 bias = {(f16)-1152.f, (f16)-1152.f, (f16)-1152.f, (f16)-1152.f,
                        (f16)-1152.f, (f16)-1152.f, (f16)-1152.f, (f16)-1152.f};
    return __builtin_bit_cast(f16x8, v) + bias;
}

// The tiled kernel for batches (gemm_w8a16_batch.hip), W column-major, any M and N, K a multiple of
// 16; X row-major, or column-major with M a multiple of 8, 16-byte aligned either way.  bn: 128 x 128
// or 128 x 64 tiles.
bool w8a16_batch_fits(int64_t M, int64_t N, int64_t ldx, int64_t K, int64_t ldw, bool xrow);
int launch_w8a16_batch(const f16* X, const int8_t* W, const f16* scale, float* Y, int64_t M, int64_t N, int64_t K,
                       int64_t ldx, int64_t ldw, int64_t ldy, bool xrow, bool yrow, int bn, hipStream_t s);

}  // namespace lava
