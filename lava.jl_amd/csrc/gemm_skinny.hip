// gemm_skinny.hip -- GEMM with at most 64 rows or columns (a projection of a few decoded tokens): one
// 64 x 64 tile of C per workgroup over all of K, f16 / bf16 / int8, plain output.
//
// Such a product is bound by reading its long operand (the weights) once: 117 MB at 64 x 14336 x 4096
// bf16, 18 to 23 us at what HBM streams.  26.6 us a call here (4.4 TB/s), whether the weights come from HBM (every
// call's elsewhere in 1 GiB) or lie in the last-level cache from the call before, 23.0 at 16 rows (23.2
// from HBM), so the short operand's L2 traffic, as many bytes again at 64 rows, is what is left.  The
// small-product kernel, 27.7 to 29.9 us resident and 30.6 from HBM (16 rows 23.9 and 27.4), keeps one K chunk per
// operand in flight in registers, splits K in two to fill the chip and adds the parts in a second kernel;
// here the loads go straight to LDS and four stages of 32 KB are in flight per CU, so one workgroup per CU
// hides HBM's latency and K needs no split from about one tile per CU on:
//  * 4 wavefronts, each all of the tile (4 x 4 accumulators) over one 64-byte k-step of every 256 bytes
//    of K, summed through LDS at the end in a fixed order;
//  * a stage is 256 bytes of K: two units of 128 bytes (TnSide at 64 rows), A and B, 8 KB each; a ring
//    of five, one barrier a stage, each request four stages ahead;
//  * the long operand's loads carry the nontemporal hint (it is read once).
#include "gemm_tn_kernel.hpp"

namespace lava {

namespace {
constexpr int SK_TILE = 64;
constexpr int SK_SLICE = SK_TILE * TN_KB;   // 8 KB of A or B, 128 bytes of K
constexpr int SK_STAGE = 4 * SK_SLICE;      // A, A, B, B
constexpr int SK_RING = 5;
}  // namespace

// M/N-contiguous (16-bit) at 64 columns per tile: the slice is 64 rows of K x 128 bytes, two rows per
// 256-byte bank window.  Row r's logical chunk c is stored at slot c ^ S(r), S(r) = 2 (r / 2 % 2) + 4
// ((r / 8 + r / 16) % 2).  A fragment's transposing reads are the 128-column form's; a 32-lane pass
// touches 8 k rows x 2 adjacent chunks, whose row parity and chunk pair S makes distinct whether the
// pass is 16-lane groups {0, 1} or {0, 2} / {1, 3} (row bits 0, 1 and 3 or 4 vary).
template <typename T>
struct TnSide<T, false, 64> {
    static_assert(sizeof(T) == 2, "M/N-contiguous staging reads 16-bit elements transposed");
    v4i rs;
    uint32_t off[2];   // per instruction: the row's swizzle depends on it
    uint32_t step;     // soffset per instruction: 8 rows of K
    uint32_t ld;       // bytes per row of K
    int klim;          // instruction i's row is inside iff k0 + 8 i < klim
    bool cin[2];       // the lane's chunk lies inside M (N)
    int mr16;          // fragment reads: the lane's row and byte offset
    int c16[4];        // fragment reads: the stored chunk of column block t, times 16

    __device__ __forceinline__ static int swz(int r) { return 2 * ((r >> 1) & 1) + 4 * (((r >> 3) ^ (r >> 4)) & 1); }

    __device__ __forceinline__ void init(const T* X, int64_t ld_b, int tile, int, int64_t mn_total, int K, int w, int,
                                         int lane) {
        const int64_t col0 = (int64_t)tile * 64;
        rs = make_rsrc(reinterpret_cast<const char*>(X) + col0 * (int64_t)sizeof(T),
                       (uint32_t)((int64_t)K * ld_b - col0 * (int64_t)sizeof(T)));
        // DMA: instruction i covers k rows 16 w + 8 i + lane / 8, slot lane % 8
        const int rr = lane >> 3, p = lane & 7;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = p ^ swz(16 * w + 8 * i + rr);
            off[i] = (uint32_t)((16 * w + rr) * ld_b + 16 * c);
            cin[i] = col0 + 8 * c < mn_total;
        }
        step = (uint32_t)(8 * ld_b);
        ld = (uint32_t)ld_b;
        klim = K - 16 * w - rr;
        // fragments: source lane ss of 16-lane group g points at k row 8 g + 4 r + ss / 4 (+ 32 u), columns
        // 16 t + 4 (ss % 4); that row's swizzle is S(8 g + ss / 4) for every u, t and r (bits 2 and 5 do
        // not enter S)
        const int ss = lane & 15, g = lane >> 4;
        const int f = swz(8 * g + (ss >> 2));
        mr16 = (8 * g + (ss >> 2)) * 128 + 8 * (ss & 1);
#pragma unroll
        for (int t = 0; t < 4; ++t) c16[t] = ((2 * t + ((ss & 3) >> 1)) ^ f) * 16;
    }
    __device__ __forceinline__ bool valid(int i, uint32_t kofs, int) const {
        return (int)(kofs / sizeof(T)) + 8 * i < klim && cin[i];
    }
    __device__ __forceinline__ uint32_t voff(int i) const { return off[i]; }
    __device__ __forceinline__ uint32_t soff(int i, uint32_t kofs) const {
        return (kofs / (uint32_t)sizeof(T)) * ld + i * step;
    }
    __device__ __forceinline__ uint4 read16(const uint8_t* slice, int u, int t) const {
        const uint8_t* b = slice + u * 32 * 128 + mr16 + c16[t];
        const tn_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) tn_s16x4*)(const __attribute__((address_space(3))) uint8_t*)b);
        const tn_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) tn_s16x4*)(const __attribute__((address_space(3))) uint8_t*)(b + 4 * 128));
        return __builtin_bit_cast(uint4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
};

template <typename T, bool AK, bool BK, bool BLONG>
__global__ void __launch_bounds__(256, 1)
    gemm_skinny_kernel(const T* __restrict__ A, const T* __restrict__ B, typename Mfma16<T>::acc_elem* __restrict__ C,
                       int stages, int64_t lda_b, int64_t ldb_b, int64_t ldc, TnBounds bnd) {
    using AccV = typename Mfma16<T>::acc_t;
    typedef typename Mfma16<T>::acc_elem Acc;
    typedef Acc Acc4 __attribute__((ext_vector_type(4)));
    __shared__ __attribute__((aligned(1024))) uint8_t smem[SK_RING * SK_STAGE];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tm = BLONG ? 0 : blockIdx.x, tn = BLONG ? blockIdx.x : 0;
    const int a_rows = (int)min((int64_t)SK_TILE, bnd.m - (int64_t)tm * SK_TILE);
    const int b_rows = (int)min((int64_t)SK_TILE, bnd.n - (int64_t)tn * SK_TILE);
    const int kelems = bnd.kb / (int)sizeof(T), ktiles = (bnd.kb + TN_KB - 1) / TN_KB;
    TnSide<T, AK, SK_TILE> sa;
    TnSide<T, BK, SK_TILE> sb;
    sa.init(A, lda_b, tm, a_rows, bnd.m, kelems, w, 0, lane);
    sb.init(B, ldb_b, tn, b_rows, bnd.n, kelems, w, 0, lane);
    // wave w fills the w-th quarter of each 8 KB slice, instruction i 1 KB of it
    const uint32_t lds0 = lds_addr(smem) + w * (SK_SLICE / 4);
    // requests stage s (past the last one too: those read zero and keep the waits' counts)
    auto issue = [&](int s, int slot) __attribute__((always_inline)) {
        const uint32_t dst = lds0 + slot * SK_STAGE;
#pragma unroll
        for (int q = 0; q < 4; ++q) {   // unit q / 2, instruction q % 2
            // units past K: no address, and the last unit's offset, so that none leaves 2 GiB
            const int unit = 2 * s + (q >> 1);
            const uint32_t kofs = (uint32_t)min(unit, ktiles - 1) * TN_KB;
            const bool live = unit < ktiles;
            const int i = q & 1;
            const uint32_t va = live && sa.valid(i, kofs, bnd.kb) ? sa.voff(i) : OOB_OFS;
            const uint32_t vb = live && sb.valid(i, kofs, bnd.kb) ? sb.voff(i) : OOB_OFS;
            if constexpr (BLONG) {
                dma16(sa.rs, va, sa.soff(i, kofs), dst + (q >> 1) * SK_SLICE + 1024 * i);
                dma16_stream(sb.rs, vb, sb.soff(i, kofs), dst + (2 + (q >> 1)) * SK_SLICE + 1024 * i);
            } else {
                dma16_stream(sa.rs, va, sa.soff(i, kofs), dst + (q >> 1) * SK_SLICE + 1024 * i);
                dma16(sb.rs, vb, sb.soff(i, kofs), dst + (2 + (q >> 1)) * SK_SLICE + 1024 * i);
            }
        }
    };
    AccV acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0;
    // this wavefront's k-step of a stage: unit w / 2, half w % 2 of the unit's bytes
    const int half = w & 1;
    if constexpr (AK) sa.sl16[0] ^= 64 * half;
    if constexpr (BK) sb.sl16[0] ^= 64 * half;
    const int a_ofs = (w >> 1) * SK_SLICE + (AK ? 0 : half * (SK_SLICE / 2));
    const int b_ofs = (2 + (w >> 1)) * SK_SLICE + (BK ? 0 : half * (SK_SLICE / 2));

#pragma unroll
    for (int s = 0; s < SK_RING - 1; ++s) issue(s, s);
    int slot = 0, fill = SK_RING - 1;
    for (int s = 0; s < stages; ++s) {
        // this wavefront's part of stage s landed and its reads of stage s - 1 returned; everyone's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(8 * (SK_RING - 2)) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        issue(s + SK_RING - 1, fill);
        const uint8_t* st = smem + slot * SK_STAGE;
        uint4 a[4], b[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            a[t] = sa.read16(st + a_ofs, 0, t);
            b[t] = sb.read16(st + b_ofs, 0, t);
        }
        // MFMA A operand = B fragment, B operand = A fragment: acc[i][j] register r of lane l is
        // C[m][n], m = 16 i + l % 16, n = 16 j + 4 (l / 16) + r
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = Mfma16<T>::run(b[j], a[i], acc[i][j]);
        fill = slot;
        slot = slot == SK_RING - 1 ? 0 : slot + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the requests past K have landed too
    __syncthreads();

    // the four partial sums [wave][row][col], rows padded to 272 bytes, added in wave order
    constexpr int PITCH = SK_TILE * 4 + 16;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<Acc4*>(smem + ((w * SK_TILE + 16 * i + (lane & 15)) * PITCH + (16 * j + 4 * (lane >> 4)) * 4)) =
                acc[i][j];
    __syncthreads();
    const int c = 4 * (threadIdx.x & 15), cols_in = min(4, b_rows - c);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int row = 16 * t + (threadIdx.x >> 4);
        if (row >= a_rows || cols_in <= 0) continue;
        Acc4 v = *reinterpret_cast<const Acc4*>(smem + row * PITCH + c * 4);
#pragma unroll
        for (int z = 1; z < 4; ++z) {
            const Acc4 o = *reinterpret_cast<const Acc4*>(smem + (z * SK_TILE + row) * PITCH + c * 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (std::is_same<Acc, int32_t>::value)
                    v[r] = (int32_t)((uint32_t)v[r] + (uint32_t)o[r]);
                else
                    v[r] += o[r];
            }
        }
        Acc* dst = C + ((int64_t)tm * SK_TILE + row) * ldc + (int64_t)tn * SK_TILE + c;
        if (cols_in == 4 && bnd.cvec) {
            *reinterpret_cast<Acc4*>(dst) = v;
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (k < cols_in) dst[k] = v[k];
        }
    }
}

template <typename T>
int launch_gemm_skinny(const T* A, const T* B, typename Mfma16<T>::acc_elem* C, int64_t M, int64_t N, int64_t K,
                       int64_t lda, int64_t ldb, int64_t ldc, hipStream_t s, bool ak, bool bk) {
    const bool blong = M <= SK_TILE;
    const int tiles = (int)((blong ? N : M) + SK_TILE - 1) / SK_TILE;
    const int64_t sz = (int64_t)sizeof(T);
    TnBounds bnd;
    bnd.m = M;
    bnd.n = N;
    bnd.kb = (int)(K * sz);
    bnd.cvec = ldc % 4 == 0 && aligned(C, 16);
    const int stages = (int)((K * sz + 2 * TN_KB - 1) / (2 * TN_KB));
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)tiles), dim3(256), 0, s, A, B, C, stages, lda * sz, ldb * sz, ldc, bnd);
    };
    auto by_long = [&](auto ltag) {
        constexpr bool L = decltype(ltag)::value;
        if constexpr (sizeof(T) == 1) {
            go(gemm_skinny_kernel<T, true, true, L>);
        } else {
            if (!ak && !bk) go(gemm_skinny_kernel<T, false, false, L>);
            else if (!ak) go(gemm_skinny_kernel<T, false, true, L>);
            else if (!bk) go(gemm_skinny_kernel<T, true, false, L>);
            else go(gemm_skinny_kernel<T, true, true, L>);
        }
    };
    blong ? by_long(std::true_type{}) : by_long(std::false_type{});
    LAVA_LAUNCH_CHECK("gemm_skinny_kernel");
    return LAVA_HIP_OK;
}
template int launch_gemm_skinny<f16>(const f16*, const f16*, float*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                                     hipStream_t, bool, bool);
template int launch_gemm_skinny<bf16>(const bf16*, const bf16*, float*, int64_t, int64_t, int64_t, int64_t, int64_t,
                                      int64_t, hipStream_t, bool, bool);
template int launch_gemm_skinny<int8_t>(const int8_t*, const int8_t*, int32_t*, int64_t, int64_t, int64_t, int64_t,
                                        int64_t, int64_t, hipStream_t, bool, bool);

// Measured against the small-product kernel (us, that / this; the operands resident in the caches between
// calls, in brackets read from HBM, those of each call elsewhere in 1 GiB; ranges over drawn calls are this one's
// time over that one's):
//  * with 192 to 256 tiles (240 above 8192 bytes of K) and a long operand whose rows are whole 128-byte lines,
//    0.60 to 1.00 (0.49 to 0.98), whether that one splits K or not: 64 x 14336 x 4096 bf16 29.2 / 26.9, W
//    N-contiguous 32.5 / 29.0, 64 x 16384 x 4096 46.6 / 29.6.  Fewer tiles leave CUs idle, more make a second
//    round: 11008 (172) 25.1 / 25.5, 4096 (64) 14.1 / 22.1, 28672 (448) 53.7 / 57.1;
//  * rows that cross lines cost this one more: its units are 128 bytes of K, which then lie in two lines each, that
//    one's are 512.  Both operands K-contiguous: up to 32 rows 0.60 to 1.17 (0.49 to 1.07), median 0.91; to 48
//    0.75 to 1.11 (0.59 to 1.05) where that one does not split K, but 0.91 to 1.36 (0.82 to 1.17) where it does; 64 rows
//    0.76 to 1.52 (0.59 to 1.39): i8 64 x 14400 x 8096 27.9 / 39.0 (31.9 / 38.5), bf16 64 x 15360 x 16200 103.7 /
//    145.5 (102.4 / 141.9).  One of them M/N-contiguous: 0.71 to 1.15 (0.59 to 1.07) up to 8192 bytes of K, 64
//    rows above that 0.89 to 1.30 (0.85 to 1.13).  From 255 tiles that kernel gives way to the mid-size one, which
//    this one leads on any rows (0.54 to 0.97);
//  * fewer tiles and less than 4096 bytes of K: 0.65 to 0.91 (0.64 to 1.09) while that one does not split K, 1.14
//    to 1.77 (1.08 to 2.02) where it does: bf16 1344 x 64 x 2024 8.5 / 14.7 (9.6 / 19.3).  Below 2048 bytes of K
//    0.81 to 1.03 (0.75 to 1.10), int8 at 1024 bytes and 12288 columns 6.3 / 6.7: left to that one.
bool skinny_gemm_preferred(int64_t M, int64_t N, int64_t k_bytes, size_t elem, bool ak, bool bk, bool lines) {
    const int64_t few = M < N ? M : N;
    if (few > SK_TILE || (elem == 1 && !(ak && bk))) return false;
    const int64_t tiles = ((M < N ? N : M) + SK_TILE - 1) / SK_TILE;
    const bool splits = k_bytes > (tiles > 128 ? 15 : 7) * 512;   // the small-product kernel would (small_gemm_splits)
    if (k_bytes < 4096) {
        if (elem != 2 || k_bytes < 2048 || tiles > 256 || splits) return false;
        if (tiles <= 128) return true;
    } else if (tiles > 256 || tiles < (k_bytes <= 8192 ? 192 : 240)) {
        return false;
    }
    return lines || tiles >= 255 || few <= (splits ? 32 : 48) || (!(ak && bk) && k_bytes <= 8192);
}

}  // namespace lava
