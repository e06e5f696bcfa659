// gemm_mid_ksplit.hip -- the mid-size GEMM kernel's K-split form (gemm_mid_ksplit_kernel): one 128 x 128
// tile of C per CU, its four wavefronts splitting K.  Plain products, f16 / bf16 / int8, any operand
// layout.
//
// gemm_mid_kernel gives each wavefront a 64 x 64 sub-tile.  That reads 8 KB of LDS per 16 MFMAs, 125
// bytes a cycle over a CU's four wavefronts before the staged bytes are written, at an LDS that serves
// about 115; a second workgroup on the CU hides the waits, but with at most 256 tiles there is none.
// Here every wavefront computes the whole tile (8 x 8 accumulators, 4 KB per 16 MFMAs, as in the tile
// kernel) over a quarter of K:
//  * a pass is 256 bytes of K, one 64-byte k-step and 64 MFMAs per wavefront, staged by all four as two
//    units of 128 bytes of K (TnSide at 128 rows, A and B, 32 KB) in a ring of five;
//  * one barrier a pass, in its middle (the loop below);
//  * the four partial sums meet in LDS in a fixed order at the end (192 KB each way, about 1.6 us: K
//    has to be long enough to pay for that, mid_ksplit_preferred).
// What bounds it now is the latency of the loads: a pass takes 0.81 us against about 0.5 for its MFMAs,
// with the 96 KB that five units leave in flight (all CUs walk K together, so most lines come from
// beyond the L2); twice the depth in gemm_mid_kernel (four stages) did not help that one.
// bf16, A row-major and B column-major, before -> after (us): 2048^2 x 8192 73.2 -> 60.1 (1143
// TFLOP/s), 1536^2 x 8192 72.8 -> 53.2, 1024 x 4096 x 4096 42.0 -> 33.8, 512 x 4096 x 4096 39.0 -> 31.5,
// 2048^3 23.0 -> 21.3 (all column-major 23.9 -> 21.3).
#include "gemm_tn_kernel.hpp"

namespace lava {

namespace {
constexpr int TM_TILE = 128;
constexpr int TK_SLICE = TM_TILE * TN_KB;   // 16 KB of A or B
constexpr int TK_UNIT = 2 * TK_SLICE;
constexpr int TK_RING = 5;
}  // namespace

template <typename T, bool RAGGED, bool AK, bool BK>
__global__ void __launch_bounds__(256, 1)
    gemm_mid_ksplit_kernel(const T* __restrict__ A, const T* __restrict__ B, typename Mfma16<T>::acc_elem* __restrict__ C,
                           int tiles_m, int tiles_n, int ktiles, int64_t lda_b, int64_t ldb_b, int64_t ldc, TnBounds bnd) {
    using AccV = typename Mfma16<T>::acc_t;
    typedef typename Mfma16<T>::acc_elem Acc;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[TK_RING * TK_UNIT];

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int tm, tn;
    xcd_tile(blockIdx.x, tiles_m, tiles_n, 4, tm, tn);

    // rows (m, n) of this tile inside the matrix: all unless RAGGED and the tile is the last
    int a_rows = TM_TILE, b_rows = TM_TILE;
    if constexpr (RAGGED) {
        a_rows = (int)(bnd.m - (int64_t)tm * TM_TILE < TM_TILE ? bnd.m - (int64_t)tm * TM_TILE : TM_TILE);
        b_rows = (int)(bnd.n - (int64_t)tn * TM_TILE < TM_TILE ? bnd.n - (int64_t)tn * TM_TILE : TM_TILE);
    }
    const int kelems = bnd.kb / (int)sizeof(T);
    TnSide<T, AK, TM_TILE> sa;
    TnSide<T, BK, TM_TILE> sb;
    sa.init(A, lda_b, tm, a_rows, bnd.m, kelems, w, 0, lane);
    sb.init(B, ldb_b, tn, b_rows, bnd.n, kelems, w, 0, lane);
    // wave w fills the w-th quarter of each slice, instruction i 1 KB of it
    const uint32_t lds0 = lds_addr(smem) + w * (TK_SLICE / 4);

    // DMA load q of unit n of K (past the last one: zeros) into ring slot `slot`
    auto dma = [&](int q, int n, int slot) __attribute__((always_inline)) {
        const uint32_t kofs = (uint32_t)min(n, ktiles - 1) * TN_KB;
        const uint32_t dst = lds0 + slot * TK_UNIT + (q >> 2) * TK_SLICE + 1024 * (q & 3);
        bool in = n < ktiles;
        if (q < 4) {
            if constexpr (RAGGED) in = in && sa.valid(q, kofs, bnd.kb);
            dma16(sa.rs, in ? sa.voff(q) : OOB_OFS, sa.soff(q, kofs), dst);
        } else {
            if constexpr (RAGGED) in = in && sb.valid(q - 4, kofs, bnd.kb);
            dma16(sb.rs, in ? sb.voff(q - 4) : OOB_OFS, sb.soff(q - 4, kofs), dst);
        }
    };

    AccV acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0;

    // This wavefront's k-step of a pass: unit w / 2 of it, half w % 2 of the unit's bytes.
    uint4 fa[8], fb[8];
    const int sub = w >> 1, half = w & 1;
    if constexpr (AK) sa.sl16[0] ^= 64 * half;
    if constexpr (BK) sb.sl16[0] ^= 64 * half;
    const int a_ofs = AK ? 0 : half * (TK_SLICE / 2);
    const int b_ofs = TK_SLICE + (BK ? 0 : half * (TK_SLICE / 2));
    auto rd_a = [&](const uint8_t* unit, int i) __attribute__((always_inline)) { fa[i] = sa.read16(unit + a_ofs, 0, i); };
    auto rd_b = [&](const uint8_t* unit, int j) __attribute__((always_inline)) { fb[j] = sb.read16(unit + b_ofs, 0, j); };
    auto slot_of = [](int s) __attribute__((always_inline)) { return s >= TK_RING ? s - TK_RING : s; };

    const int passes = (ktiles + 1) / 2;
#pragma unroll
    for (int n = 0; n < TK_RING; ++n)
#pragma unroll
        for (int q = 0; q < 8; ++q) dma(q, n, n);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 * (TK_RING - 2)) : "memory");   // pass 0's units
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const uint8_t* unit = smem + sub * TK_UNIT;
#pragma unroll
    for (int i = 0; i < 4; ++i) rd_a(unit, i);
#pragma unroll
    for (int j = 0; j < 8; ++j)
        if (j != 3) rd_b(unit, j);

    // A pass's 64 MFMAs walk the quadrants (a 0-3, b 0-3), (0-3, 4-7), (4-7, 4-7), (4-7, 0-3), column
    // by column, so that every fragment register is free at least 12 MFMAs before the next pass
    // first reads it and one set of fragments is enough: the next pass's a 0-3, b 4-7 and b 0-2
    // are read in the second half, b 3 and a 4-7 at the start of their own pass.  The barrier sits
    // between the halves: every read of this pass's units has returned, so they are requested again
    // in the second half, and the next pass's have landed (one unit newer than they may be in flight).
    // MFMA A operand = B fragment, B operand = A fragment: acc[i][j] register r of lane l is
    // C[m][n], m = 16 i + l % 16, n = 16 j + 4 (l / 16) + r.
    int s0 = 0;   // ring slot of the pass's first unit
    for (int p = 0; p < passes; ++p) {
        const int s1 = slot_of(s0 + 2);
        const uint8_t* next = smem + slot_of(s1 + sub) * TK_UNIT;
        constexpr int ND = 2 * 8;
#pragma unroll
        for (int t = 0; t < 64; ++t) {
            const int qd = t >> 4, i = (t & 3) + (qd >= 2 ? 4 : 0), j = ((t >> 2) & 3) + (qd == 1 || qd == 2 ? 4 : 0);
            if (t == 32) {
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(8) : "memory");
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
            acc[i][j] = Mfma16<T>::run(fb[j], fa[i], acc[i][j]);
            if (t == 0) rd_b(unit, 3);
            if (t >= 1 && t <= 4) rd_a(unit, 3 + t);
            if (t >= 32 && t < 36) rd_a(next, t - 32);
            if (t >= 36 && t < 52 && t % 4 == 0) rd_b(next, 4 + (t - 36) / 4);
            if (t >= 52 && t % 4 == 0) rd_b(next, (t - 52) / 4);
            if (t >= 32 && t % 2 == 1 && (t - 33) / 2 < ND) {
                const int d = (t - 33) / 2;
                dma(d % 8, 2 * p + TK_RING + d / 8, slot_of(s0 + d / 8));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        s0 = s1;
        unit = next;
    }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the requests past K have landed too
    __syncthreads();

    // ---- the partial sums and the store.  Wavefront w finishes row blocks 2 w and 2 w + 1, one a
    // round: every wavefront leaves the others' blocks of the round in LDS, adds to its own what they
    // left (in the order of their k-steps) and stages the sums as whole rows (padded to 528 bytes, so
    // the 16 rows of one staging store start on distinct banks), which it then stores 512 bytes a row.
    constexpr int EP_PITCH = 128 * 4 + 16;
    constexpr int BOX = 8 * 1024;                 // one wavefront's blocks of a round
    constexpr int EP = 4 * (4 - 1) * BOX;         // the staging areas start behind the boxes
    static_assert(EP + 4 * 16 * EP_PITCH <= TK_RING * TK_UNIT, "boxes and staging rows fit the ring");
    typedef Acc Acc4 __attribute__((ext_vector_type(4)));
    uint8_t* ep = smem + EP + w * (16 * EP_PITCH);
    // the box of wavefront `from` for `to`: three of each wavefront, in order of `to`
    auto box = [&](int from, int to) __attribute__((always_inline)) {
        return reinterpret_cast<Acc4*>(smem + (from * 3 + to - (to > from ? 1 : 0)) * BOX) + lane;
    };
    const int rc = lane & 31, rsub = lane >> 5;   // read-back: the lane's 16-byte chunk, row within 2
    const int64_t col0 = (int64_t)tn * TM_TILE;
    int cols_in = 4;   // columns of this lane's 4-column group inside the matrix (RAGGED: 0..4)
    if constexpr (RAGGED) {
        const int64_t left = bnd.n - (col0 + 4 * rc);
        cols_in = left >= 4 ? 4 : (left > 0 ? (int)left : 0);
    }
    // round is a template constant so that acc stays in registers
    auto finish = [&](auto roundtag) __attribute__((always_inline)) {
        constexpr int RD = decltype(roundtag)::value;
        const int64_t row0 = (int64_t)tm * TM_TILE + 16 * (2 * w + RD);
        Acc* cbase = C + row0 * ldc + col0;
        // acc's blocks are compile-time indices: one branch per wavefront
        auto give_to = [&](auto metag, auto totag) __attribute__((always_inline)) {
            constexpr int ME = decltype(metag)::value, TO = decltype(totag)::value;
            if constexpr (ME != TO) {
                Acc4* out = box(ME, TO);
#pragma unroll
                for (int j = 0; j < 8; ++j) out[j * 64] = acc[2 * TO + RD][j];
            }
        };
        auto give = [&](auto me) __attribute__((always_inline)) {
            give_to(me, std::integral_constant<int, 0>{});
            give_to(me, std::integral_constant<int, 1>{});
            give_to(me, std::integral_constant<int, 2>{});
            give_to(me, std::integral_constant<int, 3>{});
        };
        auto plus = [](Acc4 v, Acc4 o) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (std::is_same<Acc, int32_t>::value)
                    v[r] = (int32_t)((uint32_t)v[r] + (uint32_t)o[r]);
                else
                    v[r] += o[r];
            }
            return v;
        };
        auto take = [&](auto metag) __attribute__((always_inline)) {
            constexpr int ME = decltype(metag)::value;
            const Acc4* o0 = box(ME == 0 ? 1 : 0, ME);
            const Acc4* o1 = box(ME <= 1 ? 2 : 1, ME);
            const Acc4* o2 = box(ME <= 2 ? 3 : 2, ME);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                *reinterpret_cast<Acc4*>(ep + (lane & 15) * EP_PITCH + (16 * j + 4 * (lane >> 4)) * 4) =
                    plus(plus(plus(acc[2 * ME + RD][j], o0[j * 64]), o1[j * 64]), o2[j * 64]);
        };
        // (the branches differ only in acc's indices: merged into one, they would index it at run time and
        // put it in memory, hence an asm comment of its own at both ends of each)
        auto step_is = [&](auto metag, auto f) __attribute__((always_inline)) {
            asm volatile("; k-step %0 begin" ::"n"(decltype(metag)::value));
            f(metag);
            asm volatile("; k-step %0 end" ::"n"(decltype(metag)::value));
        };
        auto by_step = [&](auto f) __attribute__((always_inline)) {
            if (w == 0) step_is(std::integral_constant<int, 0>{}, f);
            else if (w == 1) step_is(std::integral_constant<int, 1>{}, f);
            else if (w == 2) step_is(std::integral_constant<int, 2>{}, f);
            else step_is(std::integral_constant<int, 3>{}, f);
        };
        by_step(give);
        __syncthreads();
        by_step(take);
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the wave's staged rows are in LDS
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const int row = 2 * t + rsub;
            const Acc4 v = *reinterpret_cast<const Acc4*>(ep + row * EP_PITCH + rc * 16);
            Acc* dst = cbase + (int64_t)row * ldc + 4 * rc;
            if (RAGGED && row0 + row >= bnd.m) continue;
            if (!RAGGED || (cols_in == 4 && bnd.cvec)) {
                __builtin_nontemporal_store(v, reinterpret_cast<Acc4*>(dst));
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (k < cols_in) dst[k] = v[k];
            }
        }
    };
    finish(std::integral_constant<int, 0>{});
    __syncthreads();   // the boxes are read
    finish(std::integral_constant<int, 1>{});
}


template <typename T>
int launch_gemm_mid_ksplit(const T* A, const T* B, typename Mfma16<T>::acc_elem* C, int64_t M, int64_t N, int64_t K,
                           int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s, bool ragged, bool ak, bool bk) {
    const int tiles_m = (int)((M + TM_TILE - 1) / TM_TILE), tiles_n = (int)((N + TM_TILE - 1) / TM_TILE);
    const int64_t ke = TN_KB / (int64_t)sizeof(T);
    const int ktiles = (int)((K + ke - 1) / ke);
    TnBounds bnd;
    bnd.m = M;
    bnd.n = N;
    bnd.kb = (int)(K * (int64_t)sizeof(T));
    bnd.cvec = ldc % 4 == 0 && aligned(C, 16);
    const int64_t lda_b = lda * (int64_t)sizeof(T), ldb_b = ldb * (int64_t)sizeof(T);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n)), dim3(256), 0, s, A, B, C, tiles_m, tiles_n,
                           ktiles, lda_b, ldb_b, ldc, bnd);
    };
    auto by_layout = [&](auto rtag) {
        constexpr bool R = decltype(rtag)::value;
        if (!ak && !bk) go(gemm_mid_ksplit_kernel<T, R, false, false>);
        else if (!ak) go(gemm_mid_ksplit_kernel<T, R, false, true>);
        else if (!bk) go(gemm_mid_ksplit_kernel<T, R, true, false>);
        else go(gemm_mid_ksplit_kernel<T, R, true, true>);
    };
    ragged ? by_layout(std::true_type{}) : by_layout(std::false_type{});
    LAVA_LAUNCH_CHECK("gemm_mid_kernel+gemm_mid_ksplit_kernel");   // a form's name follows its kernel's
    return LAVA_HIP_OK;
}
template int launch_gemm_mid_ksplit<f16>(const f16*, const f16*, float*, int64_t, int64_t, int64_t, int64_t, int64_t,
                                         int64_t, hipStream_t, bool, bool, bool);
template int launch_gemm_mid_ksplit<bf16>(const bf16*, const bf16*, float*, int64_t, int64_t, int64_t, int64_t, int64_t,
                                          int64_t, hipStream_t, bool, bool, bool);
template int launch_gemm_mid_ksplit<int8_t>(const int8_t*, const int8_t*, int32_t*, int64_t, int64_t, int64_t, int64_t,
                                            int64_t, int64_t, hipStream_t, bool, bool, bool);

// Measured (us, the other kernel / this; the operands resident in the caches between calls, in brackets read from
// HBM, those of each call elsewhere in 1 GiB; ranges over drawn calls are this one's time over the other's):
//  * against gemm_mid_kernel (128 to 256 tiles), from 4096 bytes of K 0.64 to 1.03 (0.62 to 0.94): 2048^2 x 2048
//    bf16 23.8 / 21.5 (29.9 / 25.1), x 4096 42.2 / 34.7, 1536^2 x 2048 21.6 / 20.0; int8 2048^2 x 4096 23.2 / 22.1,
//    x 8192 41.7 / 35.2; below, 2048^2 x 1024 bf16 14.4 / 15.0, x 1536 19.6 / 20.4, int8 x 2048 14.0 / 15.7;
//  * against the small-product kernel, where that has more than 256 tiles of 64 x 64 and so no K split (65 to
//    127 of 128 x 128), from 8192 bytes of K 0.52 to 1.09 (0.65 to 1.20), median 0.82 (0.98): 512 x 2816 x 8192
//    bf16 69.5 / 52.4 (71.4 / 72.2).  A K-contiguous operand whose rows cross 128-byte lines costs this one more, its
//    units being 128 bytes of K against that one's 512: one of them 0.88 to 1.06 (1.01 to 1.30) below 12288 bytes of
//    K, 0.66 to 1.03 (0.86 to 1.37) above; both 0.84 to 1.20 (1.14 to 1.61), f16 512 x 3072 x 11432 104.1 / 109.6
//    (113.6 / 156.9).  Two extents of 512 at least: 128 x 14336 x 4096, a weight stream, 40.8 / 47.6; 1100 x
//    1000 x 2048 20.6 / 22.9.
// Above 256 tiles gemm_mid_kernel has its two workgroups per CU (2048 x 4096 x 4096 56.6 / 67.7).
bool mid_ksplit_preferred(int64_t M, int64_t N, int64_t k_bytes, int crossing) {
    const int64_t t128 = ((M + TM_TILE - 1) / TM_TILE) * ((N + TM_TILE - 1) / TM_TILE);
    if (t128 > 256) return false;
    if (t128 >= 128) return k_bytes >= 4096;
    return crossing < 2 && k_bytes >= (crossing ? 12288 : 8192) && M >= 512 && N >= 512 && ((M + 63) / 64) * ((N + 63) / 64) > 256;
}

}  // namespace lava
