// gemm_w8a16_batch.hip -- W8A16 for batches, W column-major: a two-dimensionally tiled product whose
// weight fragments are dequantized on the way from LDS to the MFMA.
//
// The weight-streaming kernel (w8a16_kmajor_kernel) reads 16 to 64 rows of X for every 32 columns
// of W, so past a few tens of rows it is bound by X's L2 -> LDS traffic (64 rows: 512 KB of X against
// 128 KB of W per workgroup at K = 4096; time grows linearly with M).  Here a workgroup owns 128 rows x
// BN = 64 or 128 columns of Y and X is read once per BN columns:
//  * a stage is 128 k: X as two slices of 64 k in the GEMM kernels' staging (TnSide: row- or
//    column-major X, LDS-DMA, swizzled), W as BN columns x 128 bytes (16-byte chunk c of column n at slot
//    c ^ (n / 2 % 8), which spreads an 8-byte fragment read's 16 columns over all banks);
//  * 8 wavefronts, 4 along the stage's k (one 32-k MFMA step each) and 2 side by side, of 128 x 64
//    (BN = 128) or 64 x 64 sub-tiles: with 64 x 64 x 2 k-steps at BN = 128 every W fragment is
//    dequantized twice and LDS serves 6 KB instead of 5 per 16 MFMAs (35.6 against 33.4 us at 256 x
//    14336 x 4096);
//  * a ring of 3 or 4 stages, one barrier per stage; a stage's buffer is requested again as soon as
//    it has been read, so a request has 2 or 3 stages to land;
//  * the four partial sums meet in LDS (fixed order), are scaled per column and stored as whole rows.
// 256 x 14336 x 4096: 89.0 -> 33.4 us (900 TFLOP/s), 128 x 14336 x 4096 45.6 -> 21.5, X and Y
// column-major 157 -> 34.3 at 256 rows.  A 128 x 128 stage costs about 1024 cycles of MFMA, as many
// of LDS (80 KB of fragment reads, 48 KB written by the DMA) and 770 of DMA, so no one of them alone
// bounds it: without the MFMAs (timing copy) it ran 28.9 us, without the DMA 26.0.
#include <hip/hip_runtime.h>

#include "gemm_tn_kernel.hpp"
#include "gemm_w8a16.hpp"

namespace lava {

namespace {
constexpr int WB_SEG = 128;   // k per stage
constexpr int WB_WAVES = 8;

template <int BM, int BN>
struct WbCfg {
    static constexpr int KS = 4;                              // wavefronts along k: one 32-k step of a stage each
    static constexpr int NN = BN / 64, NM = WB_WAVES / (NN * KS);   // wavefronts side by side
    static constexpr int NI = BM / NM / 16;                   // 16-row blocks per wavefront (of 4 16-column blocks)
    static constexpr int SLICE = BM * 128;                    // X, 64 k
    static constexpr int STAGE = 2 * SLICE + BN * WB_SEG;
    static constexpr int BUFS = BN == 128 ? 3 : 4;
    static constexpr int X_INSTR = BM / 32;                   // X DMA instructions per wavefront and stage
    static constexpr int W_INSTR = BN / 64;                   // W DMA instructions per wavefront and stage
    static constexpr int PER = X_INSTR + W_INSTR;
    static constexpr int RED = 2 * (BM > BN ? BM * (BN + 4) : BN * (BM + 4)) * 4;
    static constexpr int LDS = BUFS * STAGE > RED ? BUFS * STAGE : RED;
    static_assert(LDS <= 160 * 1024, "LDS");
};
}  // namespace

template <int BM, int BN, bool XROW, bool YROW>
__global__ void __launch_bounds__(64 * WB_WAVES)
    w8a16_batch_kernel(const f16* __restrict__ X, const int8_t* __restrict__ W, const f16* __restrict__ scale,
                       float* __restrict__ Y, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldy, int tiles_m,
                       int tiles_n, int yvec) {
    using Cfg = WbCfg<BM, BN>;
    constexpr int NI = Cfg::NI, MF = 4 * NI;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[Cfg::LDS];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane & 15, g = lane >> 4;
    int tm, tn;
    xcd_tile(blockIdx.x, tiles_m, tiles_n, 4, tm, tn);
    const int wm = w % Cfg::NM, wn = w / Cfg::NM % Cfg::NN, ks = w / (Cfg::NM * Cfg::NN);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int rows_in = (int)min((int64_t)BM, M - m0), cols_in = (int)min((int64_t)BN, N - n0);

    // X: wavefronts 0-3 fill the stage's first 64-k slice, 4-7 its second
    TnSide<f16, XROW, BM> sx;
    sx.init(X, ldx * 2, tm, rows_in, M, K, w & 3, Cfg::NM == 2 ? wm : 0, lane);
    const int xh = w >> 2;
    // W: wavefront w's instruction i covers columns 8 (W_INSTR w + i) + lane / 8, slot lane % 8
    const v4i w_rs = make_rsrc(W + n0 * ldw, (uint32_t)(cols_in * ldw));
    uint32_t w_off[Cfg::W_INSTR];
    int w_k[Cfg::W_INSTR];
#pragma unroll
    for (int i = 0; i < Cfg::W_INSTR; ++i) {
        const int col = 8 * (Cfg::W_INSTR * w + i) + (lane >> 3);
        w_k[i] = 16 * ((lane & 7) ^ ((col >> 1) & 7));
        w_off[i] = col < cols_in ? (uint32_t)(col * ldw + w_k[i]) : OOB_OFS;
    }
    const uint32_t lds_x = lds_addr(smem) + xh * Cfg::SLICE + (w & 3) * (Cfg::SLICE / 4);
    const uint32_t lds_w = lds_addr(smem) + 2 * Cfg::SLICE + w * Cfg::W_INSTR * 1024;
    // request i of stage st (past the last stage too: those read zero and keep the waits' counts)
    auto dma = [&](int i, int st, int buf) __attribute__((always_inline)) {
        const uint32_t kx = (uint32_t)(st * WB_SEG + 64 * xh) * 2;
        if (i < Cfg::X_INSTR) {
            dma16(sx.rs, sx.valid(i, kx, 2 * K) ? sx.voff(i) : OOB_OFS, sx.soff(i, kx),
                  lds_x + buf * Cfg::STAGE + 1024 * i);
        } else {
            const int j = i - Cfg::X_INSTR;
            dma16(w_rs, st * WB_SEG + w_k[j] < K ? w_off[j] : OOB_OFS, (uint32_t)(st * WB_SEG),
                  lds_w + buf * Cfg::STAGE + 1024 * j);
        }
    };

    f32x4 acc[NI][4];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // this wavefront's k-step of a stage: X fragments, dequantized W fragments -- two sets, the MFMAs
    // read one while the next step's operands fill the other -- and raw W fragments.  Of 8 X
    // fragments only the last has a place in either set (two whole sets pass 256 registers): the
    // others (ac) are refilled in place, each behind its own MFMAs.
    constexpr int AD = NI == 8 ? 1 : 4;
    struct Set {
        uint4 a[AD];
        f16x8 b[4];
    } s0, s1;
    uint4 ac[NI - AD + 1];
    uint2 r[4];
    const int x_rd = (ks >> 1) * Cfg::SLICE + (XROW ? 0 : (ks & 1) * 32 * 256);
    if constexpr (XROW) sx.sl16[0] = sx.sl16[0] ^ (64 * (ks & 1));
    const int w_rd = 2 * Cfg::SLICE + (64 * wn + q) * WB_SEG + 16 * ((2 * ks + (g >> 1)) ^ (q >> 1)) + 8 * (g & 1);
    auto rd_w = [&](const uint8_t* st, int j) __attribute__((always_inline)) {
        r[j] = *reinterpret_cast<const uint2*>(st + w_rd + 16 * WB_SEG * j);
    };
    auto rd_x = [&](Set& f, const uint8_t* st, int i) __attribute__((always_inline)) {
        (i < NI - AD ? ac[i < NI - AD ? i : 0] : f.a[i < NI - AD ? 0 : i - (NI - AD)]) = sx.read16(st + x_rd, 0, i);
    };
    auto mma = [&](const Set& f, int t) __attribute__((always_inline)) {
        const int i = t / 4, j = t % 4;
        const f16x8 av = __builtin_bit_cast(f16x8, i < NI - AD ? ac[i < NI - AD ? i : 0] : f.a[i < NI - AD ? 0 : i - (NI - AD)]);
        // YROW: register r of lane (q, g) is Y[16 i + q][16 j + 4 g + r], else Y[16 i + 4 g + r][16 j + q]
        acc[i][j] = YROW ? __builtin_amdgcn_mfma_f32_16x16x32_f16(f.b[j], av, acc[i][j], 0, 0, 0)
                         : __builtin_amdgcn_mfma_f32_16x16x32_f16(av, f.b[j], acc[i][j], 0, 0, 0);
    };
    // The step's MF MFMAs, and beside them the reads of the next one from `from` (W's first), its
    // four dequants, and the requests of stage `st`.  The dequants (10 VALU instructions per 16 x 32
    // W fragment) are pinned to their places: left alone the compiler gathers them ahead of the first
    // MFMA.
    auto step = [&](const Set& now, Set& then, const uint8_t* from, int st, int buf)
                    __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < MF; ++t) {
            mma(now, t);
            if (t < 4) rd_w(from, t);
            if (t % 4 == 3 && t / 4 < NI - AD) rd_x(then, from, t / 4);
            if (t >= 4 && t < 4 + AD) rd_x(then, from, NI - AD + t - 4);
#pragma unroll
            for (int i = 0; i < Cfg::PER; ++i)
                if (i * MF / Cfg::PER == t) dma(i, st, buf);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (t == MF / 2 + j * MF / 8) {
                    uint4 v = __builtin_bit_cast(uint4, w8_dequant(r[j].x, r[j].y));
                    asm volatile("; dequant" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w));
                    then.b[j] = __builtin_bit_cast(f16x8, v);
                }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // a wait for all but the newest BUFS - 2 stages of this wavefront's requests, and for its LDS
    // reads; after the barrier, for everyone's
    auto turn = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((Cfg::BUFS - 2) * Cfg::PER) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    const int stages = (K + WB_SEG - 1) / WB_SEG;
#pragma unroll
    for (int b = 0; b < Cfg::BUFS; ++b)
#pragma unroll
        for (int i = 0; i < Cfg::PER; ++i) dma(i, b, b);
    turn();   // stages 0 and 1 landed
#pragma unroll
    for (int j = 0; j < 4; ++j) rd_w(smem, j);
#pragma unroll
    for (int i = 0; i < NI; ++i) rd_x(s0, smem, i);
#pragma unroll
    for (int j = 0; j < 4; ++j) s0.b[j] = w8_dequant(r[j].x, r[j].y);
    int buf = 0;
    // stage s + 1's operands are read beside stage s's MFMAs while stage s's buffer is refilled (an
    // odd count of stages runs one of zeros more)
    auto pass = [&](const Set& now, Set& then, int s) __attribute__((always_inline)) {
        turn();   // stage s + 1 landed, stage s read
        const int free = buf;
        buf = buf == Cfg::BUFS - 1 ? 0 : buf + 1;
        step(now, then, smem + buf * Cfg::STAGE, s + Cfg::BUFS, free);
    };
    for (int s = 0; s < stages; s += 2) {
        pass(s0, s1, s);
        pass(s1, s0, s + 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the requests past K have landed too
    __syncthreads();

    // partial sums [ks % 2][row][col] (YROW) or [..][col][row], rows padded by 16 bytes: steps 2 and 3
    // leave theirs, 0 and 1 add their own
    constexpr int R = YROW ? BM : BN, C = YROW ? BN : BM, PITCH = C + 4;
    float* red = reinterpret_cast<float*>(smem);
    auto place = [&](int i, int j) __attribute__((always_inline)) {
        const int rr = YROW ? 16 * (NI * wm + i) + q : 64 * wn + 16 * j + q;
        const int cc = YROW ? 64 * wn + 16 * j + 4 * g : 16 * (NI * wm + i) + 4 * g;
        return reinterpret_cast<f32x4*>(red + ((ks & 1) * R + rr) * PITCH + cc);
    };
    if (ks >= 2) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) *place(i, j) = acc[i][j];
    }
    __syncthreads();
    if (ks < 2) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) *place(i, j) = acc[i][j] + *place(i, j);
    }
    __syncthreads();
    const int rl = YROW ? rows_in : cols_in, cl = YROW ? cols_in : rows_in;
    for (int e = threadIdx.x; e < R * (C / 4); e += 64 * WB_WAVES) {
        const int r = e / (C / 4), c = 4 * (e % (C / 4));
        if (r >= rl || c >= cl) continue;
        f32x4 v = *reinterpret_cast<const f32x4*>(red + r * PITCH + c) +
                  *reinterpret_cast<const f32x4*>(red + (R + r) * PITCH + c);
        // the dequant scale of each element's column (from a clamped index past the last)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int64_t n = YROW ? n0 + min(c + t, cols_in - 1) : n0 + r;
            v[t] *= (float)scale[n];
        }
        float* y = YROW ? Y + (m0 + r) * ldy + n0 + c : Y + (n0 + r) * ldy + m0 + c;
        if (yvec && c + 4 <= cl) {
            *reinterpret_cast<f32x4*>(y) = v;
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (c + t < cl) y[t] = v[t];
        }
    }
}

bool w8a16_batch_fits(int64_t M, int64_t N, int64_t ldx, int64_t K, int64_t ldw, bool xrow) {
    // 32-bit buffer offsets over 128 rows (column-major X: all K k-lines) of X and 128 columns of W,
    // the requests past K included
    const int64_t lim = int64_t(1) << 31;
    return 128 * ldw + 1024 < lim && (xrow ? 132 * ldx * 2 + 4096 : (K + 1024) * ldx * 2) < lim &&
           ((M + 127) / 128) * ((N + 63) / 64) < lim;
}

int launch_w8a16_batch(const f16* X, const int8_t* W, const f16* scale, float* Y, int64_t M, int64_t N, int64_t K,
                       int64_t ldx, int64_t ldw, int64_t ldy, bool xrow, bool yrow, int bn, hipStream_t s) {
    constexpr int bm = 128;
    const int tiles_m = (int)((M + bm - 1) / bm), tiles_n = (int)((N + bn - 1) / bn);
    const int yvec = ldy % 4 == 0 && aligned(Y, 16);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n)), dim3(64 * WB_WAVES), 0, s, X, W, scale, Y, (int)M,
                           (int)N, (int)K, ldx, ldw, ldy, tiles_m, tiles_n, yvec);
    };
    auto by_tile = [&](auto xr, auto yr) {
        constexpr bool XR = decltype(xr)::value, YR = decltype(yr)::value;
        if (bn == 128)
            go(w8a16_batch_kernel<128, 128, XR, YR>);
        else
            go(w8a16_batch_kernel<128, 64, XR, YR>);
    };
    typedef std::integral_constant<bool, true> T_;
    typedef std::integral_constant<bool, false> F_;
    if (xrow)
        yrow ? by_tile(T_{}, T_{}) : by_tile(T_{}, F_{});
    else
        yrow ? by_tile(F_{}, T_{}) : by_tile(F_{}, F_{});
    LAVA_LAUNCH_CHECK(bn == 128 ? "w8a16_batch_kernel<128,128>" : "w8a16_batch_kernel<128,64>");
    return LAVA_HIP_OK;
}

}  // namespace lava
