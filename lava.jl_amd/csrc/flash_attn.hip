// flash_attn.hip -- causal flash-attention forward, fp16 in/out, fp32 softmax state.
//
// The reference is the coopmat2 flash kernel Lava's vocabulary was shaped for
// (`attn_flash_rows!` / flash_attn_cm2, src/vocabulary/coopmat.jl:158;
// src/device/coopmat_intrinsics.jl:535-755): per query block, per key block,
//   S = Q K^T; rowmax = reduce(max, S, Row); M = max(rowmax, Mold);
//   P = exp(S - M); O = O * exp(Mold - M) + P V; L = L * exp(Mold - M) + rowsum(P)
// and finally O / L, converted to fp16 (RNE).
//
// Kernels (the dispatcher at the end of the file picks one):
//  * flash_fwd5_kernel -- D <= 128 (the headline shape D = 128), any softmax scale: on each SIMD
//    a score wavefront and an output wavefront share 64 queries (described at the kernel);
//  * flash_fwd6_kernel -- D = 56 and 64 with a positive scale, where it is the faster one (fa_cost):
//    64 queries' both products in each wavefront, two wavefronts splitting the key blocks;
//  * flash_fwd3_kernel -- D = 256 with a positive scale (and D = 64 or 128 on request):
//    ping-pong pairs of 32-query wavefronts;
//  * flash_generic_kernel -- any D <= 256, one thread per query (every other case).
//
// The common CDNA4 formulation:
//  * everything is computed transposed, S^T = K Q^T and O^T = V^T P^T, on the 32x32x16
//    fp16 MFMA.  In that form the accumulator lane owns ONE query (lane % 32; lanes l and
//    l ^ 32 share it) and holds that query's scores for 16 keys per 32-key tile, so the row
//    max and row sum are in-lane reductions plus one exchange with lane ^ 32, the rescale of
//    O is one multiplier per lane, and the score accumulator converts in place to the B
//    operand P^T of the second product (keys in-lane), with no relayout;
//  * Q^T stays in registers for the whole key loop;
//  * K and V blocks of 64 keys are staged in LDS by LDS-DMA, 16-byte chunks XOR-swizzled so
//    that the K fragment reads and the transposing V reads are bank-conflict-free;
//  * softmax in base 2 (s * scale * log2 e, v_exp_f32) with lazy rescaling;
//  * causal: key blocks above the diagonal are never loaded, and only the diagonal block is
//    masked per element;
//  * workgroups are ordered XCD by XCD so that all query blocks of one (batch, head) run on
//    one XCD and share its K and V through that XCD's L2; causal: longest query blocks first
//    across groups of the XCD's heads (fa_order).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>

#include "lava_coopmat.hpp"
#include "lava_hip_internal.hpp"
#include "lds_dma.hpp"

namespace lava {

constexpr int FA_D = 128;

struct FaParams {
    const f16* Q;
    const f16* K;
    const f16* V;
    f16* O;
    int64_t sl, sh, sb;      // strides of L, H, B (elements) for Q/K/V
    int64_t osl, osh, osb;   // for O
    int S, H, B;
    float scale_log2;        // softmax scale * log2(e)
    int causal;
    int o16;                 // O and its strides allow 16-byte row stores
    int D;                   // head dimension (the score/output kernel zero-pads it to 128)
    int dv;                  // the ping-pong kernel at DQK = 256: V / O columns of this launch's half
};

// Workgroup -> (batch * head, query block).  Workgroups are dispatched round-robin
// over the 8 XCDs (blockIdx % 8).  Non-causal: every block costs the same, and each
// XCD takes a contiguous range of (head, block) pairs, so one head's K and V stay in
// one XCD's L2.  Causal: query block qb costs qb + 1 key blocks, so each XCD takes
// whole heads (when 8 divides B * H), in groups of 4 heads (when 4 divides the
// XCD's count), and runs a group's heaviest blocks first, then the next lighter
// ones: longest first across the group keeps the dispatch tail short, and one
// group's K and V (8 MiB at D = 128, S = 4096) is what the XCD streams at a time.
// Measured at B = 4, H = 32, S = 4096: groups of 4 heads 934-937 TFLOP/s, of all 16
// of the XCD's heads 886-893, one head at a time 835.  Without the split by XCD,
// heavy first over all heads.
__device__ __forceinline__ void fa_order(int nqb, int nbh, bool causal, int& bh, int& qb) {
    const int bid = blockIdx.x;
    if (causal) {
        if ((nbh & 7) == 0) {
            const int h8 = nbh >> 3, local = bid >> 3;
            const int G = (h8 & 3) == 0 ? 4 : h8;   // heads per group
            const int grp = local / (G * nqb), r = local % (G * nqb);
            qb = nqb - 1 - r / G;
            bh = (bid & 7) * h8 + grp * G + r % G;
        } else {
            qb = nqb - 1 - bid / nbh;
            bh = bid % nbh;
        }
    } else {
        const int total = nqb * nbh;
        const int b2 = (total & 7) == 0 ? (bid & 7) * (total >> 3) + (bid >> 3) : bid;
        bh = b2 / nqb;
        qb = b2 % nqb;
    }
}

// ---------------------------------------------------------------------------
// Version 3 (the fast path): 8 wavefronts x 32 queries = 256 queries per
// workgroup; K and V blocks of 64 keys move global -> LDS by buffer_load ... lds,
// so no VGPRs stage them and each block is loaded once per 256 queries; V^T
// operands come from the row-major V tile through ds_read_b64_tr_b16.
//
// Ping-pong schedule.  Each wavefront alternates an MFMA phase (O += V^T P^T for
// the previous block, then S^T = K Q^T for this one: 32 MFMAs) and a softmax
// phase (VALU only), with a workgroup barrier after every phase.  Wavefronts 4-7
// start one phase late, so each SIMD (holding wavefronts w and w + 4) always has
// one wavefront in its MFMA phase and the other in its softmax phase, and the
// matrix core and the VALU work at the same time instead of taking turns.
//
// K and V have three LDS stages each.  The MFMA phase of iteration kb issues the
// DMA of K block kb + 2 and V block kb + 1 (4 instructions per wavefront at D = 128,
// 6 with 512-byte K rows) and each phase ends with s_waitcnt vmcnt(that count), so a
// wavefront's DMAs have landed by the end of its next MFMA phase; the barrier after
// it publishes them.  The stage a DMA
// overwrites was last read by the late wavefronts one phase before it is issued.
//
// LDS layout: K [64 keys][256 B] and V [64 keys][256 B] per stage, 16-byte chunks
// XOR-swizzled -- K by key % 16 (a fragment read is 32 keys x one chunk), V by
// 4 (key % 4) (a transposing read is 4 keys x 32 bytes per 16-lane group) -- so
// neither read pattern has bank conflicts.
//
// ds_read_b64_tr_b16: in a 16-lane group, output lane i value j is the 16-bit word
// at (address of source lane 4 j + i / 4) + 2 (i % 4).  Source lane 4 jj + q points
// at V[key0 + jj][d0 + 4 q], so output lane i receives V[key0 .. key0 + 3][d0 + i]:
// four keys of one head-dimension column, the k-slots of the V^T operand.
//
// Lazy rescaling: the running maximum moves (and O, L are rescaled) only when a
// block's maximum exceeds it by more than 2^8; P = exp2(s - m) then stays <= 256,
// exact enough in fp16, and O / L is unchanged in exact arithmetic.
constexpr int F3_WAVES = 8;
constexpr int F3_BQ = 32 * F3_WAVES;        // 256 queries per workgroup
constexpr int F3_BK = 64;
constexpr int F3_STAGES = 3;
constexpr float F3_RESCALE = 8.0f;
constexpr int F3_PREFETCH = 4;        // MFMA-phase operations between an LDS read and its use

template <bool B>
struct f3_tag {
    static constexpr bool value = B;
};

typedef short f3_s16x4 __attribute__((ext_vector_type(4)));
typedef short f3_s16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f3_s16x4 f3_read_tr(const uint8_t* p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) f3_s16x4*)(const __attribute__((address_space(3))) uint8_t*)p);
}

// Asm uses (a comment: the backend drops empty asm) that pin a value's computation before this point: without them the
// compiler sinks the softmax's exp / convert / sum (used only by the next phase's
// MFMAs) across the barrier into the MFMA phase, which undoes the ping-pong.
__device__ __forceinline__ void f3_pin(const f16x8& v) {
    const uint4 u = __builtin_bit_cast(uint4, v);
    asm volatile("; pin" ::"v"(u.x), "v"(u.y), "v"(u.z), "v"(u.w));
}
__device__ __forceinline__ void f3_pin(const f32x16& v) {
#pragma unroll
    for (int i = 0; i < 16; i += 4) asm volatile("; pin" ::"v"(v[i]), "v"(v[i + 1]), "v"(v[i + 2]), "v"(v[i + 3]));
}

// All waits for the DMAs of the phase before last (N = the DMA instructions one
// phase issues), then the workgroup barrier.
template <int N>
__device__ __forceinline__ void f3_phase_end() {
    static_assert(N == 6 || N == 4 || N == 2, "K + V DMA instructions per wavefront and phase");
    if constexpr (N == 6)
        asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    else if constexpr (N == 4)
        asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else
        asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
    __syncthreads();
}

// DQK (the Q / K head dimension: 64, 128 or 256) and DV (the V / O one: 64 or 128; DQK = 256
// runs with DV = 128, once per half of V's columns) set the row sizes (D * 2 bytes = CH chunks
// of 16 bytes), the number of S^T k-steps (DQK / 16) and of O^T row tiles (DV / 32), and the
// swizzles: K chunk ^ (key % 16) for rows of 16 or more chunks, ^ ((key % 8) ^ (key / 8 % 2))
// for 8-chunk rows (a fragment read, 32 keys x one chunk, spread over the banks); V chunk
// ^ 4 (key % 4), resp. ^ 2 (key % 4) (a transposing read, 4 keys x 2 chunks per 16-lane group).
template <bool CAUSAL, int DQK, int DV>
__global__ void __launch_bounds__(64 * F3_WAVES, 1) flash_fwd3_kernel(FaParams p) {
    static_assert((DQK == DV && (DV == 128 || DV == 64)) || (DQK == 256 && DV == 128),
                  "head dimensions 64, 128, or 256 for Q/K with 128 for V/O");
    constexpr int RBK = DQK * 2, RBV = DV * 2;             // bytes per K / V row
    constexpr int CHK = RBK / 16, CHV = RBV / 16;          // 16-byte chunks per row
    constexpr int TILEK = F3_BK * RBK, TILEV = F3_BK * RBV;   // one K / V block
    constexpr int NKS = DQK / 16;                          // S^T MFMAs per key tile
    constexpr int NDT = DV / 32;                           // O^T row tiles
    constexpr int NPV = 4 * NDT;                           // O^T MFMAs per block
    constexpr int NOPS = NPV + 2 * NKS;                    // MFMAs of a full phase
    constexpr int DPTK = TILEK / (1024 * F3_WAVES);        // DMA instructions per wavefront per tile
    constexpr int DPTV = TILEV / (1024 * F3_WAVES);
    constexpr int RPIK = 64 / CHK, RPIV = 64 / CHV;        // rows per DMA instruction
    // LDS operand reads ahead of their MFMA (3 at DQK = 256, where the 16 Q^T fragments fill the
    // registers)
    constexpr int PREF = DQK == 256 ? 3 : F3_PREFETCH;
    __shared__ __attribute__((aligned(1024))) uint8_t kbuf[F3_STAGES][TILEK];   // [stage][key][RBK]
    __shared__ __attribute__((aligned(1024))) uint8_t vbuf[F3_STAGES][TILEV];
    auto kswz = [](int row) { return CHK >= 16 ? (row & 15) : ((row & 7) ^ ((row >> 3) & 1)); };
    auto vswz = [](int row) { return CHV == 16 ? 4 * (row & 3) : 2 * (row & 3); };

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool late = w >= F3_WAVES / 2;        // one phase behind its SIMD partner w - 4
    const int nqb = (p.S + F3_BQ - 1) / F3_BQ;   // the last query block may be partial
    const int nbh = p.H * p.B;
    int bh, qb;
    fa_order(nqb, nbh, CAUSAL, bh, qb);
    const int hh = bh % p.H, bb = bh / p.H;
    const int64_t head = (int64_t)hh * p.sh + (int64_t)bb * p.sb;
    f16* Ob = p.O + (int64_t)hh * p.osh + (int64_t)bb * p.osb;

    const int q0 = qb * F3_BQ + w * 32;         // this wave's first query
    const int r32 = lane & 31, h = lane >> 5;
    const int my_q = q0 + r32;

    // Q^T as B operand: lane (query my_q, half h) holds d = 16 ks + 8 h + [0, 8);
    // queries past S (a ragged last block) compute on zeros and are not stored
    f16x8 qf[NKS];
    {
        const f16* qrow = p.Q + head + (int64_t)my_q * p.sl + 8 * h;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) qf[ks] = f16x8{};
        if (my_q < p.S) {
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks)
                if (DQK != 256 || 16 * ks + 8 * h < p.D) qf[ks] = *reinterpret_cast<const f16x8*>(qrow + 16 * ks);
        }
    }

    // ---- LDS-DMA: wave w moves rows [8 w, 8 w + 8) of a K (V) tile in DPTK (DPTV)
    // instructions: instruction i covers rows 8 w + RPI i + lane / CH, physical chunk lane % CH.
    const uint32_t row_bytes = (uint32_t)(p.sl * 2);
    const v4i rk = make_rsrc(p.K + head, (uint32_t)p.S * row_bytes);
    const v4i rv = make_rsrc(p.V + head, (uint32_t)p.S * row_bytes);
    uint32_t voff_k[DPTK], voff_v[DPTV];
    // At DQK = 256 a head dimension D < 256 is zero-padded: a lane whose logical chunk lies at or
    // past D (K) or past this launch's dv columns (V) takes an offset beyond the resource, so the
    // DMA writes zeros (zero K columns add nothing to the scores; zero V columns give O columns
    // that are not stored).
#pragma unroll
    for (int i = 0; i < DPTK; ++i) {
        const int row = 8 * w + RPIK * i + lane / CHK;
        const int c = (lane % CHK) ^ kswz(row);
        voff_k[i] = (DQK != 256 || 8 * c < p.D) ? (uint32_t)row * row_bytes + 16u * (uint32_t)c : 0x80000000u;
    }
#pragma unroll
    for (int i = 0; i < DPTV; ++i) {
        const int row = 8 * w + RPIV * i + lane / CHV;
        const int c = (lane % CHV) ^ vswz(row);
        voff_v[i] = (DQK != 256 || 8 * c < p.dv) ? (uint32_t)row * row_bytes + 16u * (uint32_t)c : 0x80000000u;
    }
    const uint32_t lds_k = lds_addr(&kbuf[0][0]) + (uint32_t)w * 8 * RBK;
    const uint32_t lds_v = lds_addr(&vbuf[0][0]) + (uint32_t)w * 8 * RBV;
    const int nkb_s = (p.S + F3_BK - 1) / F3_BK;   // key blocks holding keys < S
    const int nkb = CAUSAL ? min((qb * F3_BQ + F3_BQ) / F3_BK, nkb_s) : nkb_s;
    // block j -> stage j % F3_STAGES; blocks past the end re-read the last one so
    // that every MFMA phase issues the same number of DMAs (the vmcnt accounting).
    // A row at or past S gets an offset beyond the resource (2^31 > S * row bytes,
    // no wrap with soffset), so it reads zero whether or not the range check counts
    // soffset; its scores are masked.
    // (ntag: DMA instructions per tile; ctag: chunks per row, so 64 / CH rows per instruction)
    auto issue = [&](auto ntag, auto ctag, const v4i& rsrc, const uint32_t* voff, uint32_t lds, int tile, int j) {
        constexpr int DPT = decltype(ntag)::value, CH = decltype(ctag)::value;
        const int src = j < nkb ? j : nkb - 1;
        const uint32_t soff = (uint32_t)src * F3_BK * row_bytes;
        const uint32_t dst = lds + (uint32_t)(j % F3_STAGES) * tile;
        uint32_t v[DPT];
#pragma unroll
        for (int i = 0; i < DPT; ++i) v[i] = voff[i];
        if ((src + 1) * F3_BK > p.S) {   // uniform: only the ragged last block checks rows
#pragma unroll
            for (int i = 0; i < DPT; ++i)
                v[i] = src * F3_BK + 8 * w + (64 / CH) * i + lane / CH < p.S ? v[i] : 0x80000000u;
        }
#pragma unroll
        for (int i = 0; i < DPT; ++i) dma16(rsrc, v[i], soff, dst + 1024 * i);
    };
    auto issue_k = [&](int j) {
        issue(std::integral_constant<int, DPTK>{}, std::integral_constant<int, CHK>{}, rk, voff_k, lds_k, TILEK, j);
    };
    auto issue_v = [&](int j) {
        issue(std::integral_constant<int, DPTV>{}, std::integral_constant<int, CHV>{}, rv, voff_v, lds_v, TILEV, j);
    };
    constexpr int DPP = DPTK + DPTV;   // DMA instructions per wavefront and MFMA phase

    // K fragment (kt, ks): row 32 kt + r32, logical chunk 2 ks + h, stored at chunk ^ kswz(row)
    // (kswz depends on row % 16 = r32 % 16 only)
    // (2 ks + h) ^ kswz = 2 ks ^ (h ^ kswz) with kswz < 16 and the row's byte offset a multiple of
    // 32 chunks, so k_off[ks] = k_off[0] ^ 32 ks; at DQK = 256 that XOR is done per read instead of
    // holding 16 offsets in registers
    constexpr bool K_XOR = NKS > 8;
    int k_off[K_XOR ? 1 : NKS];
#pragma unroll
    for (int ks = 0; ks < (K_XOR ? 1 : NKS); ++ks) k_off[ks] = r32 * RBK + (((2 * ks + h) ^ kswz(r32)) << 4);
    auto k_ofs = [&](int ks) { return K_XOR ? (k_off[0] ^ (32 * ks)) : k_off[ks]; };
    // V^T fragment (dt, kk = 32 kt + 16 ks, read t = 0/1): source lane jj = (lane % 16) / 4,
    // q = lane % 4, dh = (lane / 16) % 2 addresses V[kk + 8 t + 4 h + jj][32 dt + 16 dh + 4 q],
    // logical chunk 4 dt + 2 dh + q / 2 stored at chunk ^ vswz(jj) (jj = key % 4 as kk % 8 == 0).
    int v_off[NDT];
    {
        const int jj = (lane & 15) >> 2, q = lane & 3, dh = (lane >> 4) & 1;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
            v_off[dt] = (4 * h + jj) * RBV + (((4 * dt + 2 * dh + (q >> 1)) ^ vswz(jj)) << 4) + ((q & 1) << 3);
    }

    f32x16 o[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
    float m_run = -INFINITY;   // running max of the scaled scores (log2 units)
    float l_run = 0.f;         // this lane's partial row sum
    const float c = p.scale_log2;
    f32x16 st[2];              // S^T of the current block: st[kt] register r = key 32 kt + 8 (r / 4) + 4 h + r % 4
    f16x8 pf[2][2];            // P^T of the previous block, B operand [kt][ks]: keys 32 kt + 16 ks + 8 (i / 4) + 4 h + i % 4

    // The MFMA phase as one list of NOPS operations -- ops [0, NPV): O^T += V^T P^T
    // for the previous block (kt = i / (2 NDT), ks = i / NDT % 2, dt = i % NDT); ops
    // [NPV, NOPS): S^T = K Q^T (ks = (i - NPV) / 2, kt = i % 2) -- whose LDS operand
    // reads run PREF operations ahead of the MFMAs (the partner wavefront is in
    // its softmax phase, so nothing else hides the LDS latency).
    auto read_op = [&](int i, const uint8_t* vbase, const uint8_t* kbase) -> f16x8 {
        if (i < NPV) {
            const int kk = 32 * (i / (2 * NDT)) + 16 * ((i / NDT) & 1), dt = i % NDT;
            const f3_s16x4 lo = f3_read_tr(vbase + v_off[dt] + kk * RBV);
            const f3_s16x4 hi = f3_read_tr(vbase + v_off[dt] + (kk + 8) * RBV);
            return __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
        const int j = i - NPV;
        return *reinterpret_cast<const f16x8*>(kbase + k_ofs(j >> 1) + (j & 1) * 32 * RBK);
    };
    auto mma_op = [&](int i, f16x8 a) {
        if (i < NPV) {
            o[i % NDT] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pf[i / (2 * NDT)][(i / NDT) & 1], o[i % NDT], 0,
                                                                 0, 0);
        } else {
            const int j = i - NPV;
            st[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[j >> 1], j < 2 ? f32x16{} : st[j & 1], 0, 0, 0);
        }
    };
    auto mfma_phase = [&](auto pv_tag, auto s_tag, const uint8_t* vbase, const uint8_t* kbase) {
        constexpr int first = decltype(pv_tag)::value ? 0 : NPV;
        constexpr int last = decltype(s_tag)::value ? NOPS : NPV;
        f16x8 buf[PREF];
#pragma unroll
        for (int t = 0; t < PREF; ++t)
            if (first + t < last) buf[t] = read_op(first + t, vbase, kbase);
#pragma unroll
        for (int i = first; i < last; ++i) {
            const f16x8 a = buf[(i - first) % PREF];
            if (i + PREF < last) buf[(i - first) % PREF] = read_op(i + PREF, vbase, kbase);
            mma_op(i, a);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (decltype(s_tag)::value) {
            f3_pin(st[0]);
            f3_pin(st[1]);
        }
    };

    issue_k(0);
    // Consume Q here so the compiler's own wait for its loads happens once, before
    // the loop, instead of as vmcnt waits inside it (which would also cover the
    // DMAs issued in the loop, since it does not count those).
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        const uint4 u = __builtin_bit_cast(uint4, qf[ks]);
        asm volatile("" ::"v"(u.x), "v"(u.y), "v"(u.z), "v"(u.w));
    }
    issue_k(1);
    issue_v(0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (late) __builtin_amdgcn_s_barrier();

    // Online softmax of block kb (base 2, the scale folded into the exponent's fma):
    // masks the diagonal block, rescales O and L when the maximum moves (lazily),
    // and leaves P^T in pf for the next MFMA phase.
    auto softmax = [&](int kb) {
        const int key0 = kb * F3_BK;
        if (CAUSAL && key0 + F3_BK - 1 > q0) {
            // (for a query < S every key past S is also past the query)
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = key0 + 32 * kt + 8 * (r >> 2) + 4 * h + (r & 3);
                    st[kt][r] = key > my_q ? -INFINITY : st[kt][r];
                }
        } else if (!CAUSAL && key0 + F3_BK > p.S) {   // the ragged last key block
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = key0 + 32 * kt + 8 * (r >> 2) + 4 * h + (r & 3);
                    st[kt][r] = key >= p.S ? -INFINITY : st[kt][r];
                }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, st[kt][r]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * c;
        if (__builtin_amdgcn_ballot_w64(mx > m_run + F3_RESCALE)) {
            const float m_new = fmaxf(m_run, mx);
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
            m_run = m_new;
        }
        const float mneg = -m_run;
        float lsum = 0.f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                f16x8 pv;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float e = __builtin_amdgcn_exp2f(fmaf(st[kt][8 * ks + i], c, mneg));
                    lsum += e;
                    pv[i] = (f16)e;
                }
                pf[kt][ks] = pv;
            }
        l_run += lsum;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) f3_pin(pf[kt][ks]);
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) f3_pin(o[dt]);
        asm volatile("; pin" ::"v"(l_run), "v"(m_run));
    };
    // Every MFMA phase issues the DMAs of K block kb + 2 and V block kb + 1: the
    // tiles are loaded cooperatively, so each wavefront issues its share of every
    // one, active or not, and passes the same barriers.
    auto dma = [&](int kb) {
        issue_k(kb + 2);
        issue_v(kb + 1);
    };
    auto vb = [&](int kb) { return &vbuf[(kb + F3_STAGES - 1) % F3_STAGES][0]; };   // V of block kb - 1
    auto kbuf_of = [&](int kb) { return &kbuf[kb % F3_STAGES][0]; };
    // this wavefront's last block with an unmasked key
    const int last = CAUSAL ? min(nkb - 1, (q0 + 31) / F3_BK) : nkb - 1;

    // iteration 0: S only
    dma(0);
    mfma_phase(f3_tag<false>{}, f3_tag<true>{}, vb(0), kbuf_of(0));
    f3_phase_end<DPP>();
    softmax(0);
    f3_phase_end<DPP>();
    // iterations 1 .. last: O += V^T P^T for block kb - 1, then S for block kb
    for (int kb = 1; kb <= last; ++kb) {
        dma(kb);
        mfma_phase(f3_tag<true>{}, f3_tag<true>{}, vb(kb), kbuf_of(kb));
        f3_phase_end<DPP>();
        softmax(kb);
        f3_phase_end<DPP>();
    }
    // iteration last + 1: the final O update
    dma(last + 1);
    mfma_phase(f3_tag<true>{}, f3_tag<false>{}, vb(last + 1), kbuf_of(last + 1));
    f3_phase_end<DPP>();
    f3_phase_end<DPP>();
    // remaining iterations (causal: blocks past this wavefront's queries)
    for (int kb = last + 2; kb <= nkb; ++kb) {
        dma(kb);
        f3_phase_end<DPP>();
        f3_phase_end<DPP>();
    }
    if (!late) __builtin_amdgcn_s_barrier();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- O / L, fp16.  o[dt] register r: d = 32 dt + 8 (r / 4) + 4 h + r % 4 of query my_q.
    const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
    const float inv = 1.f / l_tot;
    if (my_q >= p.S) return;
    f16* orow = Ob + (int64_t)my_q * p.osl;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
            const int d = 32 * dt + 8 * g4 + 4 * h;
            f16x4 v = {(f16)(o[dt][4 * g4 + 0] * inv), (f16)(o[dt][4 * g4 + 1] * inv),
                       (f16)(o[dt][4 * g4 + 2] * inv), (f16)(o[dt][4 * g4 + 3] * inv)};
            if (DQK != 256 || d < p.dv) __builtin_nontemporal_store(v, reinterpret_cast<f16x4*>(orow + d));
        }
}

// ---- flash_fwd5_kernel: score and output wavefronts ----
//
// Same transposed formulation (S^T = K Q^T, O^T = V^T P^T on 32x32x16 f16 MFMAs, a
// lane owns one query per 32-query half), with the work of 64 queries split between
// the two wavefronts that share a SIMD (w and w + 4):
//  * score wavefront w (0-3): Q^T of its 64 queries in registers; per key block it
//    computes S^T = K Q^T (32 MFMAs), the online softmax (lazy rescale), and writes
//    P^T as MFMA B-operand fragments (8 KB) and the rescale factors to workgroup
//    memory;
//  * output wavefront w + 4: O^T of the same 64 queries in registers; per key block
//    it rescales O when told to and adds V^T P^T (32 MFMAs).
// Every K or V fragment read from LDS feeds two MFMAs (two 32-query halves), and the
// score wavefront's softmax VALU runs beside the output wavefront's MFMAs on the same
// SIMD -- no phase barrier between them, one workgroup barrier per key block.
// Score wavefronts compute S for block j + 1 while output wavefronts add P V of block
// j; P is double-buffered.  One workgroup = 8 wavefronts = 256 queries; K in a
// three-stage LDS ring, V in two stages.  The output wavefronts, which wait for the
// score wavefronts, also issue every K and V load and sum the rows of P (from the
// fp16 fragments they read, in fp32) -- the score wavefront does only the scores and
// the softmax.
// QH = 1 gives each pair one 32-query half (128 queries per workgroup): a fragment then feeds one MFMA
// and a key block takes 0.70 of the time for half the queries, for grids that 256-query workgroups
// leave uneven or short of the 256 CUs (fa_cost).
constexpr int F5_PAIRS = 4;
constexpr int F5_BK = 64;
constexpr int F5_KST = 3, F5_VST = 2;
constexpr int F5_PFK = 4;              // K fragments read ahead of the MFMA that uses them
constexpr int F5_PFV = 5;              // V fragments read ahead

typedef _Float16 f5_h2 __attribute__((ext_vector_type(2)));
typedef uint32_t f5_u32x4 __attribute__((ext_vector_type(4)));

// x in lanes 0-31 and 32-63 as two registers: one v_permlane32_swap between two
// distinct copies of x (the builtin with one value twice may be given one register,
// and a register swapped with itself does not produce both halves)
__device__ __forceinline__ void f5_xor32_pair(float x, float& a, float& b) {
    a = x;
    b = x;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}

// q = fp16(q * c) in place, two elements per instruction: the mixed-precision FMA takes an fp16
// half of q (op_sel picks which), fp32 c and a zero addend, and rounds the exact product once to
// fp16 (measured over all 65536 fp16 values at four scales: the correctly rounded product in every
// case, except that -0 comes out +0, which adds nothing to a dot product; (f16)((float)q * c),
// rounded twice, differs in up to 3 % of them) -- one instruction instead of two converts, a
// multiply and a pack.  The trailing s_nop gives a following MFMA that reads q the wait states a
// VALU write needs before it (this is asm, so the compiler does not count it as a VALU write).
__device__ __forceinline__ void fa_scale_f16(f16x8& q, float c) {
    uint4 u = __builtin_bit_cast(uint4, q);
    asm("v_fma_mixlo_f16 %0, %0, %4, 0 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixhi_f16 %0, %0, %4, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixlo_f16 %1, %1, %4, 0 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixhi_f16 %1, %1, %4, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixlo_f16 %2, %2, %4, 0 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixhi_f16 %2, %2, %4, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixlo_f16 %3, %3, %4, 0 op_sel_hi:[1,0,0]\n\t"
        "v_fma_mixhi_f16 %3, %3, %4, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n\t"
        "s_nop 1"
        : "+v"(u.x), "+v"(u.y), "+v"(u.z), "+v"(u.w)
        : "v"(c));
    q = __builtin_bit_cast(f16x8, u);
}

// DE: the head dimension the MFMAs cover, 64, 96 or 128 (D rounded up to a multiple of 32).  K, V
// and Q are staged 128 wide whatever DE is (the chunks past D are DMA-ed as zeros, so the LDS
// layout, its swizzles and the DMA map stay those of D = 128); a smaller DE only drops the S^T
// k-steps and the O^T row tiles that would multiply those zero columns.
template <bool CAUSAL, int DE, int QH>
__global__ void __launch_bounds__(128 * F5_PAIRS, 1) flash_fwd5_kernel(FaParams p) {
    static_assert(DE == 64 || DE == 96 || DE == 128, "the MFMAs cover 64, 96 or 128 of the head dimension");
    constexpr int PQ = 32 * QH;                // queries per pair
    constexpr int BQ = PQ * F5_PAIRS;          // queries per workgroup
    constexpr int DH = 128;                    // staged width
    constexpr int RB = DH * 2;                 // 256 bytes per K / V row
    constexpr int CH = RB / 16;                // 16 chunks
    constexpr int TILE = F5_BK * RB;           // 16 KB
    constexpr int NKS = DE / 16;               // k-steps of S^T (8 at DE = 128)
    constexpr int NDT = DE / 32;               // O^T row tiles (4 at DE = 128)
    constexpr int NSF = 2 * NKS;               // K fragments per block: (ks, kt)
    constexpr int NVF = 4 * NDT;               // V fragments per block: (key step kk, dt)
    constexpr int DPT = TILE / (1024 * F5_PAIRS);   // 4 DMA instructions per wavefront per tile
    constexpr int PBUF = QH * 4 * 1024;             // one pair's P^T fragments for one block
    static_assert(DPT == 4, "4 DMA instructions per tile and wavefront");
    __shared__ __attribute__((aligned(1024))) uint8_t kbuf[F5_KST][TILE];   // [key][RB], chunk ^ key % 16
    __shared__ __attribute__((aligned(1024))) uint8_t vbuf[F5_VST][TILE];   // [key][RB], chunk ^ 4 (key % 4)
    __shared__ __attribute__((aligned(1024))) uint8_t pbuf[2][F5_PAIRS][PBUF];
    __shared__ float abuf[2][F5_PAIRS][PQ];    // rescale factor per query of the next block
    __shared__ int fbuf[2][F5_PAIRS];          // whether that block rescales
    // Q on its way in, O on its way out, 32 rows of 256 bytes at xst[qh]: two halves use the pair's P
    // buffers; one half's would not hold them, so it has room of its own
    __shared__ __attribute__((aligned(1024))) uint8_t xbuf[QH == 1 ? F5_PAIRS : 1][QH == 1 ? 32 * RB : 16];

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool is_s = w < F5_PAIRS;
    const int pr = w & (F5_PAIRS - 1);         // the pair: queries q0 .. q0 + PQ - 1
    const int nqb = (p.S + BQ - 1) / BQ;
    const int nbh = p.H * p.B;
    int bh, qb;
    fa_order(nqb, nbh, CAUSAL, bh, qb);
    const int hh = bh % p.H, bb = bh / p.H;
    const int64_t head = (int64_t)hh * p.sh + (int64_t)bb * p.sb;
    f16* Ob = p.O + (int64_t)hh * p.osh + (int64_t)bb * p.osb;
    const int q0 = qb * BQ + pr * PQ;
    const int r32 = lane & 31, h = lane >> 5;
    const int nkb_s = (p.S + F5_BK - 1) / F5_BK;
    const int nkb = CAUSAL ? min((qb + 1) * (BQ / F5_BK), nkb_s) : nkb_s;
    const int last = CAUSAL ? min(nkb - 1, (q0 + PQ - 1) / F5_BK) : nkb - 1;   // this pair's last key block

    // LDS-DMA of K and V (issued by the output wavefronts): wavefront pr moves rows
    // 16 pr + 4 i + lane / 16 of a tile, physical chunk lane % 16 (K chunk ^ key % 16, V
    // chunk ^ 4 (key % 4)).  The lane offsets are the same for every block; the buffer
    // resource of a block starts at its first row and ends at the sequence's end, so rows
    // at or past S read zero.  Blocks past the end re-read the last one (every iteration
    // issues the same DMAs).
    // A head dimension D < 128 (a multiple of 8) runs zero-padded to 128: a lane whose logical
    // chunk lies at or past D / 8 takes an offset beyond every buffer resource's range, so its
    // DMA writes zero into LDS -- zero Q and K columns add nothing to the scores, and the O
    // columns that the zero V columns produce are not stored.
    const uint32_t row_bytes = (uint32_t)(p.sl * 2);
    const int dch = p.D >> 3;                  // 16-byte chunks of a row that hold data
    auto chunk_ofs = [&](int row, int c) -> uint32_t {
        return c < dch ? (uint32_t)row * row_bytes + 16u * (uint32_t)c : 0x80000000u;
    };
    uint32_t dv_k[DPT], dv_v[DPT];
#pragma unroll
    for (int i = 0; i < DPT; ++i) {
        const int row = 16 * pr + 4 * i + lane / CH;
        dv_k[i] = chunk_ofs(row, (lane % CH) ^ (row & 15));
        dv_v[i] = chunk_ofs(row, (lane % CH) ^ (4 * (row & 3)));
    }
    auto dma_tile = [&](bool is_k, int j) __attribute__((always_inline)) {
        const int src = j < nkb ? j : nkb - 1;
        const f16* base = (is_k ? p.K : p.V) + head + (int64_t)src * F5_BK * p.sl;
        const uint32_t rows = (uint32_t)min(F5_BK, p.S - src * F5_BK);
        const v4i rs = make_rsrc(base, rows * row_bytes);
        const uint32_t dst = lds_addr(is_k ? &kbuf[0][0] : &vbuf[0][0]) + (uint32_t)pr * 16 * RB +
                             (uint32_t)(j % (is_k ? F5_KST : F5_VST)) * TILE;
#pragma unroll
        for (int i = 0; i < DPT; ++i)
            dma16(rs, is_k ? dv_k[i] : dv_v[i], 0u, __builtin_amdgcn_readfirstlane(dst + 1024u * i));
    };
    typedef __attribute__((address_space(3))) f16x8 lds_f16x8;
    typedef __attribute__((address_space(3))) f3_s16x4 lds_s16x4;
    // P^T fragment (kt, ks, qh) of pair pr in buffer b: 1 KB, lane l at 16 l
    const uint32_t p_lane = lds_addr(&pbuf[0][0][0]) + (uint32_t)pr * PBUF + 16u * lane;
    auto paddr = [&](int b, int kt, int ks, int qh) __attribute__((always_inline)) -> uint32_t {
        return p_lane + (uint32_t)(b * F5_PAIRS * PBUF + ((kt * 2 + ks) * QH + qh) * 1024);
    };

    uint32_t xst[QH];
#pragma unroll
    for (int qh = 0; qh < QH; ++qh) xst[qh] = QH == 1 ? lds_addr(&xbuf[pr][0]) : lds_addr(&pbuf[qh][pr][0]);

    // prologue DMAs (output wavefronts): K_0, K_1, K_2, V_0
    if (!is_s) {
#pragma unroll
        for (int t = 0; t < 3; ++t) dma_tile(true, t);
        dma_tile(false, 0);
    }

    if (is_s) {
        // ================= score wavefront =================
        // The pair's Q rows go to LDS first (two halves: this pair's P buffers, free until the
        // first block's P is written), in the K tile's layout -- LDS-DMA of 4 whole rows per
        // instruction, chunk ^ row % 16, rows at or past S read zero -- and the Q^T
        // fragments are read from there: whole-row reads instead of 32 rows x 32 bytes per
        // load instruction.
        {
            const uint32_t rows = (uint32_t)max(0, min(PQ, p.S - q0));
            const v4i rs = make_rsrc(p.Q + head + (int64_t)q0 * p.sl, rows * row_bytes);
#pragma unroll
            for (int i = 0; i < 8 * QH; ++i) {
                const int row = 4 * i + lane / CH;
                const uint32_t v = chunk_ofs(row, (lane % CH) ^ (row & 15));
                dma16(rs, v, 0u, __builtin_amdgcn_readfirstlane(xst[i / 8] + (uint32_t)((4 * i) % 32) * RB));
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        f16x8 qf[QH][NKS];   // Q^T B operands: query q0 + 32 qh + r32, d = 16 ks + 8 h + [0, 8)
#pragma unroll
        for (int qh = 0; qh < QH; ++qh)
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks)
                qf[qh][ks] = *(const lds_f16x8*)(uintptr_t)(xst[qh] + (uint32_t)(r32 * RB + (((2 * ks + h) ^ (r32 & 15)) << 4)));
#pragma unroll
        for (int qh = 0; qh < QH; ++qh)
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                const uint4 u = __builtin_bit_cast(uint4, qf[qh][ks]);
                asm volatile("" ::"v"(u.x), "v"(u.y), "v"(u.z), "v"(u.w));
            }
        // The base-2 softmax scale c is folded into Q^T (one fp16 rounding of q * c) when
        // that cannot overflow (c <= 1), and the running maximum enters the product as a
        // bias k-step: ones (key rows, k = 0) times -m (query columns, k = 0).  The
        // accumulator then holds S' = c q.k - m directly and P = exp2(S') needs no
        // per-score multiply-add.  m is kept fp16-representable for that; a rescaled block,
        // c > 1, or a maximum beyond +-32768 (after which the wavefront stays on this path)
        // take P = exp2(fma(S, c', -m')) in fp32 instead.  (Up to there m is off by at most 8, and P
        // at most 2^8; beyond it by up to 16, and P = 2^16 is infinite in fp16.)
        const float c = p.scale_log2;
        bool fast = c <= 1.f;                    // wavefront-uniform
        if (fast) {
#pragma unroll
            for (int qh = 0; qh < QH; ++qh)
#pragma unroll
                for (int ks = 0; ks < NKS; ++ks) fa_scale_f16(qf[qh][ks], c);
        }
        const float c_raw = fast ? 1.f : c;      // the multiplier S needs on the fp32 path
        f16x8 ones{};                            // bias A operand: 1 at k = 0 of every key row
        ones[0] = h == 0 ? (f16)1.f : (f16)0.f;
        f16x8 qm[QH] = {};                       // bias B operand: -m at k = 0 of each query
        // K fragment (kt, ks): row 32 kt + r32, chunk (2 ks + h) ^ (r32 % 16)
        uint32_t kb0[NKS];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks)
            kb0[ks] = lds_addr(&kbuf[0][0]) + (uint32_t)(r32 * RB + (((2 * ks + h) ^ (r32 & 15)) << 4));
        f32x16 st[2][QH];          // st[kt][qh] register r: key 32 kt + 8 (r / 4) + 4 h + r % 4
        float m_run[QH] = {};

        // S_kb = K_kb Q^T (minus m), the softmax, P^T and the rescale factors into buffer b
        auto block = [&](int kb, int b, bool first) __attribute__((always_inline)) {
            uint32_t ka[NKS];
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                ka[ks] = kb0[ks] + (uint32_t)((kb % F5_KST) * TILE);
                asm("; lds address" : "+v"(ka[ks]));
            }
            auto kread = [&](int f) __attribute__((always_inline)) -> f16x8 {   // f = 2 ks + kt
                return *(const lds_f16x8*)(uintptr_t)(ka[f >> 1] + (uint32_t)((f & 1) * 32 * RB));
            };
            // reads F5_PFK fragments ahead of their MFMAs; sched_barrier keeps this order
            // (the scheduler otherwise moves each read next to its use)
            f16x8 fr[F5_PFK];
#pragma unroll
            for (int f = 0; f < F5_PFK; ++f) fr[f] = kread(f);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int qh = 0; qh < QH; ++qh)
                    st[kt][qh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ones, qm[qh], f32x16{}, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < QH * NSF; ++i) {   // MFMA i: fragment f = i / QH (ks = f / 2, kt = f % 2), qh = i % QH
                const int f = i / QH, qh = i % QH, ks = f >> 1, kt = f & 1;
                st[kt][qh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[f % F5_PFK], qf[qh][ks], st[kt][qh], 0, 0, 0);
                if (qh == QH - 1 && f + F5_PFK < NSF) fr[f % F5_PFK] = kread(f + F5_PFK);
                __builtin_amdgcn_sched_barrier(0);
            }
            // mask: causal key > query; else keys >= S.  A pair's causal last block is its diagonal
            // block (it starts at the pair's first query, kb * 64 = q0, for every pair with a query
            // below S; the others are never stored), where key tile 1 lies wholly above query half
            // 0 and key tile 0 wholly below query half 1: only the two diagonal 32 x 32 tiles compare.
            // (A pair of one half starts at the block's first or 32nd key: every tile compares.)
            if (CAUSAL ? kb == last : (kb + 1) * F5_BK > p.S) {
                int dv = CAUSAL ? 4 * h - r32 - (QH == 1 ? q0 & 32 : 0) : kb * F5_BK + 4 * h - p.S;
                asm volatile("; mask" : "+v"(dv));
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int qh = 0; qh < QH; ++qh)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int kr = 32 * kt + 8 * (r >> 2) + (r & 3);
                            if (QH == 2 && CAUSAL && kt != qh) {
                                if (kt > qh) st[kt][qh][r] = -INFINITY;
                                continue;
                            }
                            const bool off = CAUSAL ? dv > 32 * qh - kr : dv >= -kr;
                            st[kt][qh][r] = off ? -INFINITY : st[kt][qh][r];
                        }
            }
            // t = how far this block's largest exponent lies above the running maximum
            const bool fast_blk = fast;           // st holds S' (fast) or S (fp32 path)
            float vl[QH];   // this lane's largest score per query half
#pragma unroll
            for (int qh = 0; qh < QH; ++qh) {
                float v = -INFINITY;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) v = fmaxf(v, st[kt][qh][r]);
                vl[qh] = fast_blk ? v : fmaf(v, c_raw, -m_run[qh]);
            }
            const bool rescale = first || __builtin_amdgcn_ballot_w64(vl[0] > F3_RESCALE || vl[QH - 1] > F3_RESCALE) != 0;
            float sub[QH] = {};
            if (rescale) {
                float t[QH];
#pragma unroll
                for (int qh = 0; qh < QH; ++qh) {
                    float a, bb2;
                    f5_xor32_pair(vl[qh], a, bb2);
                    t[qh] = fmaxf(a, bb2);
                }
                float mn[QH];
                bool ovf = false;
#pragma unroll
                for (int qh = 0; qh < QH; ++qh) {
                    // the first block sets m to its maximum (it always holds key 0, so it
                    // is never fully masked); later ones only raise it
                    mn[qh] = m_run[qh] + (first ? t[qh] : fmaxf(t[qh], 0.f));
                    ovf = ovf || !(fabsf(mn[qh]) <= 32768.f);
                }
                if (fast && __builtin_amdgcn_ballot_w64(ovf) != 0) fast = false;
                float alpha[QH];
#pragma unroll
                for (int qh = 0; qh < QH; ++qh) {
                    if (fast) mn[qh] = (float)(f16)mn[qh];
                    alpha[qh] = __builtin_amdgcn_exp2f(m_run[qh] - mn[qh]);
                    sub[qh] = fast_blk ? mn[qh] - m_run[qh] : mn[qh];
                    m_run[qh] = mn[qh];
                    qm[qh][0] = (fast && h == 0) ? (f16)(-mn[qh]) : (f16)0.f;
                }
                if (h == 0) {
#pragma unroll
                    for (int qh = 0; qh < QH; ++qh) abuf[b][pr][32 * qh + r32] = alpha[qh];
                }
            } else if (!fast_blk) {
#pragma unroll
                for (int qh = 0; qh < QH; ++qh) sub[qh] = m_run[qh];
            }
            if (lane == 0) fbuf[b][pr] = rescale ? 1 : 0;
            // P = exp2(S') (or exp2(S c' - m')) in fp16 (RNE), stored as the output wavefront's B operands
            auto pstore = [&](auto plain) __attribute__((always_inline)) {
                const float cb = fast_blk ? 1.f : c_raw;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                        for (int qh = 0; qh < QH; ++qh) {
                            f5_u32x4 u;
                            const float msub = -sub[qh];
#pragma unroll
                            for (int k = 0; k < 4; ++k) {
                                const int r0 = 8 * ks + 2 * k;
                                float x0 = st[kt][qh][r0], x1 = st[kt][qh][r0 + 1];
                                if constexpr (!decltype(plain)::value) {
                                    x0 = fmaf(x0, cb, msub);
                                    x1 = fmaf(x1, cb, msub);
                                }
                                const f5_h2 hv = {(_Float16)__builtin_amdgcn_exp2f(x0), (_Float16)__builtin_amdgcn_exp2f(x1)};
                                u[k] = __builtin_bit_cast(uint32_t, hv);
                            }
                            *(__attribute__((address_space(3))) f5_u32x4*)(uintptr_t)paddr(b, kt, ks, qh) = u;
                        }
            };
            if (fast_blk && !rescale)
                pstore(f3_tag<true>{});
            else
                pstore(f3_tag<false>{});
        };

        __syncthreads();                         // K_0 .. K_2, V_0 in LDS
        block(0, 0, true);
        __syncthreads();                         // P_0 published
        for (int j = 0; j < nkb; ++j) {
            if (j + 1 <= last) block(j + 1, (j + 1) & 1, false);
            __syncthreads();
        }
    } else {
        // ================= output wavefront =================
        // V^T fragment (dt, kk): two transposing reads at keys kk + 4 h + jj and + 8
        uint32_t vb0[NDT];
        {
            const int jj = (lane & 15) >> 2, q = lane & 3, dh = (lane >> 4) & 1;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
                vb0[dt] = lds_addr(&vbuf[0][0]) +
                          (uint32_t)((4 * h + jj) * RB + (((4 * dt + 2 * dh + (q >> 1)) ^ (4 * jj)) << 4) + ((q & 1) << 3));
        }
        f32x16 o[NDT][QH];
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
            for (int qh = 0; qh < QH; ++qh)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[dt][qh][r] = 0.f;
        float l_run[QH] = {};                    // this lane's partial row sums of P
        const f5_h2 ones = {(_Float16)1.f, (_Float16)1.f};

        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();                         // K_0 .. K_2, V_0 in LDS
        __syncthreads();                         // P_0 published
        for (int j = 0; j < nkb; ++j) {
            const int b = j & 1;
            // K_{j+3} into K_j's stage and V_{j+1} into V_{j-1}'s (both read in iteration j - 1)
            dma_tile(true, j + 3);
            dma_tile(false, j + 1);
            if (j <= last) {
                if (j > 0 && fbuf[b][pr] != 0) {   // the maximum moved at block j: O *= alpha
                    float al[QH];
#pragma unroll
                    for (int qh = 0; qh < QH; ++qh) al[qh] = abuf[b][pr][32 * qh + r32];
#pragma unroll
                    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
#pragma unroll
                            for (int qh = 0; qh < QH; ++qh) o[dt][qh][r] *= al[qh];
#pragma unroll
                    for (int qh = 0; qh < QH; ++qh) l_run[qh] *= al[qh];
                }
                uint32_t va[NDT];
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt) {
                    va[dt] = vb0[dt] + (uint32_t)((j % F5_VST) * TILE);
                    asm("; lds address" : "+v"(va[dt]));
                }
                auto vread = [&](int f) __attribute__((always_inline)) -> f16x8 {   // f = NDT kk + dt
                    const int kk = 16 * (f / NDT), dt = f % NDT;
                    const f3_s16x4 lo =
                        __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(va[dt] + (uint32_t)(kk * RB)));
                    const f3_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (lds_s16x4*)(uintptr_t)(va[dt] + (uint32_t)((kk + 8) * RB)));
                    return __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                };
                auto pread = [&](int kk, int qh) __attribute__((always_inline)) -> f16x8 {
                    return *(const lds_f16x8*)(uintptr_t)paddr(b, kk >> 1, kk & 1, qh);
                };
                // V fragments F5_PFV ahead, P one key step ahead; sched_barrier keeps the order
                f16x8 fr[F5_PFV];
                f16x8 pp[2][QH];   // [kk % 2][qh]
#pragma unroll
                for (int qh = 0; qh < QH; ++qh) pp[0][qh] = pread(0, qh);
#pragma unroll
                for (int f = 0; f < F5_PFV; ++f) fr[f] = vread(f);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < QH * NVF; ++i) {   // MFMA i: V fragment f = i / QH (kk = f / NDT, dt = f % NDT), qh = i % QH
                    const int f = i / QH, qh = i % QH, kk = f / NDT, dt = f % NDT;
                    if (i % (QH * NDT) == 0 && kk < 3) {   // the next key step's P fragments
#pragma unroll
                        for (int qq = 0; qq < QH; ++qq) pp[(kk + 1) & 1][qq] = pread(kk + 1, qq);
                    }
                    if (i % (QH * NDT) == QH * NDT / 2) {   // row sums of this key step's P (fp16 values, fp32 sum)
#pragma unroll
                        for (int qq = 0; qq < QH; ++qq)
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                l_run[qq] = __builtin_amdgcn_fdot2(f5_h2{pp[kk & 1][qq][2 * e], pp[kk & 1][qq][2 * e + 1]},
                                                                   ones, l_run[qq], false);
                    }
                    o[dt][qh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[f % F5_PFV], pp[kk & 1][qh], o[dt][qh], 0, 0,
                                                                       0);
                    if (qh == QH - 1 && f + F5_PFV < NVF) fr[f % F5_PFV] = vread(f + F5_PFV);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // K_{j+3}, V_{j+1} landed
            __syncthreads();
        }
        // ---- O / L, fp16.  o[dt][qh] register r: d = 32 dt + 8 (r / 4) + 4 h + r % 4 of query q0 + 32 qh + r32.
        float inv[QH];
#pragma unroll
        for (int qh = 0; qh < QH; ++qh) {
            float la, lb;
            f5_xor32_pair(l_run[qh], la, lb);
            inv[qh] = 1.f / (la + lb);
        }
        if (p.o16) {
            // Staged through the Q rows' place (no wavefront reads it after the last barrier) as
            // rows of 256 bytes, chunk ^ row % 16, then stored 4 whole rows per
            // instruction (16 bytes per lane) instead of 32 rows x 16 bytes.
            typedef __attribute__((address_space(3))) f16x4 lds_f16x4;
#pragma unroll
            for (int qh = 0; qh < QH; ++qh)
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4) {
                        const f16x4 v = {(f16)(o[dt][qh][4 * g4 + 0] * inv[qh]), (f16)(o[dt][qh][4 * g4 + 1] * inv[qh]),
                                         (f16)(o[dt][qh][4 * g4 + 2] * inv[qh]), (f16)(o[dt][qh][4 * g4 + 3] * inv[qh])};
                        *(lds_f16x4*)(uintptr_t)(xst[qh] + (uint32_t)(r32 * RB + (((4 * dt + g4) ^ (r32 & 15)) << 4) + 8 * h)) = v;
                    }
            // all 16 rows of a lane group read before the first store (one LDS round trip), one
            // 64-bit base per lane and a row stride
            const int lrow = lane / CH, cc = lane % CH;
            f16x8 rv[8 * QH];
#pragma unroll
            for (int i = 0; i < 8 * QH; ++i) {
                const int row = 4 * i + lrow;
                rv[i] = *(const lds_f16x8*)(uintptr_t)(xst[i / 8] + (uint32_t)((row % 32) * RB + ((cc ^ (row & 15)) << 4)));
            }
            f16* obase = Ob + (int64_t)(q0 + lrow) * p.osl + 8 * cc;
#pragma unroll
            for (int i = 0; i < 8 * QH; ++i)
                if (q0 + 4 * i + lrow < p.S && cc < dch)
                    __builtin_nontemporal_store(rv[i], reinterpret_cast<f16x8*>(obase + (int64_t)(4 * i) * p.osl));
        } else {
#pragma unroll
            for (int qh = 0; qh < QH; ++qh) {
                const int q = q0 + 32 * qh + r32;
                if (q >= p.S) continue;
                f16* orow = Ob + (int64_t)q * p.osl;
#pragma unroll
                for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4) {
                        const int d = 32 * dt + 8 * g4 + 4 * h;
                        f16x4 v = {(f16)(o[dt][qh][4 * g4 + 0] * inv[qh]), (f16)(o[dt][qh][4 * g4 + 1] * inv[qh]),
                                   (f16)(o[dt][qh][4 * g4 + 2] * inv[qh]), (f16)(o[dt][qh][4 * g4 + 3] * inv[qh])};
                        if (d < p.D) __builtin_nontemporal_store(v, reinterpret_cast<f16x4*>(orow + d));
                    }
            }
        }
    }
}

// ---- flash_fwd6_kernel: head dimensions 56 and 64, both products in one wavefront ----
//
// At D = 64 a 64-key block has half the MFMAs of D = 128 and the same softmax.  O^T (64 registers), the
// scores (64), Q^T (32) and -m (32) of 64 queries fit one wavefront at two per SIMD, so each wavefront
// does both products and the softmax and P stays in registers (the score accumulator converts in
// place to the second product's operand) instead of crossing LDS between a score and an output
// wavefront:
//  * 8 wavefronts: 4 groups of 32 QH queries, each by two wavefronts (w and w + 4, one SIMD) that take
//    the even and the odd key blocks and merge their sums at the end through LDS, so a workgroup's
//    chain is half its key blocks;
//  * a step is two key blocks: K and V of both, 32 KB (128-byte rows, not padded to 256), by LDS-DMA
//    in a ring of four; one barrier a step, a request has two steps to land;
//  * -m is the score product's initial accumulator, so P = exp2 of the scores as they come (the base-2
//    scale is folded into Q^T); each 16-key step's exponentials sit between the second product's MFMAs
//    of the step before;
//  * lazy rescaling as in the other kernels.
// What bounds it is issue: 208 VALU instructions and 32 MFMAs per 64-query block take about 2250 cycles
// of a SIMD (MFMA busy 0.43), and taking out the exponentials, the maximum or the row sums (timing
// copies) gained 4, 3 and 3 %; half a step's offset between a SIMD's wavefronts, four 32-query
// wavefronts a SIMD, and the scale and maximum as a multiply-add per score all ran within 5 % of it.
// B = 4, H = 32, S = 4096 343 -> 323 us causal, 625 -> 573 not; with 32-query groups (QH = 1) H = 4, S =
// 4096 not causal 47.7 -> 37.6, B = 2, H = 12, S = 1500 causal 22.6 -> 18.3 (fa_cost has the rule).
// D = 56 runs zero-padded to 64 (chunks past D read zero).
constexpr int F6_GROUPS = 4;
constexpr int F6_TILE = F5_BK * 128;        // 64 keys of 128 bytes
constexpr int F6_STEP = 4 * F6_TILE;        // K, K, V, V of two blocks
constexpr int F6_RING = 4;

template <bool CAUSAL, int QH>
__global__ void __launch_bounds__(512, 1) flash_fwd6_kernel(FaParams p) {
    constexpr int RB = 128, PQ = 32 * QH, BQ = PQ * F6_GROUPS;
    __shared__ __attribute__((aligned(1024))) uint8_t ring[F6_RING][F6_STEP];
    __shared__ float2 stat[8][QH][32];

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int gq = w & 3, kh = w >> 2;         // query group, key half
    const int r32 = lane & 31, h = lane >> 5;
    const int nqb = (p.S + BQ - 1) / BQ;
    int bh, qb;
    fa_order(nqb, p.H * p.B, CAUSAL, bh, qb);
    const int hh = bh % p.H, bb = bh / p.H;
    const int64_t head = (int64_t)hh * p.sh + (int64_t)bb * p.sb;
    f16* Ob = p.O + (int64_t)hh * p.osh + (int64_t)bb * p.osb;
    const int q0 = qb * BQ + gq * PQ;
    const int nkb_s = (p.S + F5_BK - 1) / F5_BK;
    const int nkb = CAUSAL ? min((qb * BQ + BQ - 1) / F5_BK + 1, nkb_s) : nkb_s;
    const int last = CAUSAL ? min(nkb - 1, (q0 + PQ - 1) / F5_BK) : nkb - 1;   // this group's last key block
    const int steps = (nkb + 1) / 2;

    // LDS-DMA: wavefront w moves rows 8 w + lane / 8 of each of a step's four tiles, slot lane % 8
    // (K chunk ^ row % 8 ^ row / 8 % 2, V chunk ^ 2 (row % 4)); rows at or past S and chunks at or past
    // D read zero
    const uint32_t row_bytes = (uint32_t)(p.sl * 2);
    const int dch = p.D >> 3;
    const int lr = lane >> 3, slot = lane & 7;
    auto chunk_ofs = [&](int row, int c) -> uint32_t {
        return c < dch ? (uint32_t)row * row_bytes + 16u * (uint32_t)c : 0x80000000u;
    };
    const uint32_t ofs_k = chunk_ofs(8 * w + lr, slot ^ lr ^ (w & 1)), ofs_v = chunk_ofs(8 * w + lr, slot ^ (2 * (lr & 3)));
    const uint32_t lds_w = lds_addr(&ring[0][0]) + 1024u * w;
    auto dma_step = [&](int j, int st) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int kb = 2 * j + (t & 1);
            const int first = min(kb, nkb - 1) * F5_BK;
            const uint32_t rows = kb < nkb ? (uint32_t)min(F5_BK, p.S - first) : 0u;
            const v4i rs = make_rsrc((t < 2 ? p.K : p.V) + head + (int64_t)first * p.sl, rows * row_bytes);
            dma16(rs, t < 2 ? ofs_k : ofs_v, 0u, __builtin_amdgcn_readfirstlane(lds_w + (uint32_t)(st * F6_STEP + t * F6_TILE)));
        }
    };
    typedef __attribute__((address_space(3))) f16x8 lds_f16x8;
    typedef __attribute__((address_space(3))) f3_s16x4 lds_s16x4;
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

    // Q of the group: PQ rows, half by each of its wavefronts, in the K tile's layout, through the
    // ring's last place (free until the first step)
    const uint32_t lds_q = lds_addr(&ring[F6_RING - 1][0]) + (uint32_t)(gq * PQ * RB);
    {
        const uint32_t rows = (uint32_t)max(0, min(PQ, p.S - q0));
        const v4i rs = make_rsrc(p.Q + head + (int64_t)q0 * p.sl, rows * row_bytes);
#pragma unroll
        for (int i = 0; i < PQ / 16; ++i) {
            const int i8 = kh * (PQ / 16) + i;   // 8 rows per instruction
            dma16(rs, chunk_ofs(8 * i8 + lr, slot ^ lr ^ (i8 & 1)), 0u,
                  __builtin_amdgcn_readfirstlane(lds_q + 1024u * i8));
        }
    }
    dma_step(0, 0);
    dma_step(1, 1);
    asm volatile("s_waitcnt vmcnt(4)" ::: "memory");   // Q and step 0
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);

    // (the first request into Q's place is step 3's, after the first step's barrier)
    const int ksw = (r32 & 7) ^ ((r32 >> 3) & 1);
    f16x8 qf[QH][4];   // Q^T B operands: query q0 + 32 qh + r32, d = 16 ks + 8 h + [0, 8)
#pragma unroll
    for (int qh = 0; qh < QH; ++qh)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            qf[qh][ks] = *(const lds_f16x8*)(uintptr_t)(lds_q + (uint32_t)((32 * qh + r32) * RB + (((2 * ks + h) ^ ksw) << 4)));
    uint32_t k_rd[4], v_rd[2];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) k_rd[ks] = lds_addr(&ring[0][0]) + (uint32_t)(kh * F6_TILE + r32 * RB + (((2 * ks + h) ^ ksw) << 4));
    {
        const int jj = (lane & 15) >> 2, q = lane & 3, dh = (lane >> 4) & 1;
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
            v_rd[dt] = lds_addr(&ring[0][0]) + (uint32_t)((2 + kh) * F6_TILE + (4 * h + jj) * RB +
                                                          (((4 * dt + 2 * dh + (q >> 1)) ^ (2 * jj)) << 4) + ((q & 1) << 3));
    }
    f32x16 o[2][QH];
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int qh = 0; qh < QH; ++qh)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[dt][qh][r] = 0.f;
    // m is unset (-inf, and 0 taken off the scores) until a block holds a score above -inf; up_at: a score above
    // it moves m
    float m_run[QH], l_run[QH], up_at[QH];
#pragma unroll
    for (int qh = 0; qh < QH; ++qh) {
        m_run[qh] = up_at[qh] = -INFINITY;
        l_run[qh] = 0.f;
    }
    const f5_h2 ones = {(_Float16)1.f, (_Float16)1.f};
    f32x16 neg_m[QH];   // -m of the lane's query: the score product's initial accumulator
#pragma unroll
    for (int qh = 0; qh < QH; ++qh)
#pragma unroll
        for (int r = 0; r < 16; ++r) neg_m[qh][r] = 0.f;
    // the base-2 scale folded into Q^T (c <= 1, so the product cannot overflow; one rounding of q c)
#pragma unroll
    for (int qh = 0; qh < QH; ++qh)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) fa_scale_f16(qf[qh][ks], p.scale_log2);

    auto block = [&](int kb, uint32_t st_ofs) __attribute__((always_inline)) {
        f32x16 st[2][QH];   // S' = c q.k - m; st[kt][qh] register r: key 32 kt + 8 (r / 4) + 4 h + r % 4
        auto kread = [&](int f) __attribute__((always_inline)) -> f16x8 {   // f = 2 ks + kt
            return *(const lds_f16x8*)(uintptr_t)(k_rd[f >> 1] + st_ofs + (uint32_t)((f & 1) * 32 * RB));
        };
        f16x8 fr[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) fr[f] = kread(f);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8 * QH; ++i) {   // fragment f = i / QH, qh = i % QH
            const int f = i / QH, qh = i % QH, ks = f >> 1, kt = f & 1;
            st[kt][qh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fr[f & 3], qf[qh][ks], ks == 0 ? neg_m[qh] : st[kt][qh], 0, 0, 0);
            if (qh == QH - 1 && f + 4 < 8) fr[f & 3] = kread(f + 4);
            __builtin_amdgcn_sched_barrier(0);
        }
        auto vread = [&](int f) __attribute__((always_inline)) -> f16x8 {   // f = 2 kk + dt, keys 16 kk ..
            const int kk = 16 * (f >> 1), dt = f & 1;
            const f3_s16x4 lo =
                __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(v_rd[dt] + st_ofs + (uint32_t)(kk * RB)));
            const f3_s16x4 hi =
                __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)(v_rd[dt] + st_ofs + (uint32_t)((kk + 8) * RB)));
            return __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        };
        f16x8 vf[4];
#pragma unroll
        for (int f = 0; f < 4; ++f) vf[f] = vread(f);
        // mask: causal key > query (the group's last block holds its diagonal); else keys >= S
        if (CAUSAL ? kb == last : (kb + 1) * F5_BK > p.S) {
            int dv = CAUSAL ? kb * F5_BK + 4 * h - r32 - q0 : kb * F5_BK + 4 * h - p.S;
            asm volatile("; mask" : "+v"(dv));
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int qh = 0; qh < QH; ++qh)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int kr = 32 * kt + 8 * (r >> 2) + (r & 3);
                        const bool off = CAUSAL ? dv > 32 * qh - kr : dv >= -kr;
                        st[kt][qh][r] = off ? -INFINITY : st[kt][qh][r];
                    }
        }
        float vl[QH];   // this lane's largest S' per query half
        bool up = false;
#pragma unroll
        for (int qh = 0; qh < QH; ++qh) {
            float v = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int r = 0; r < 16; ++r) v = fmaxf(v, st[kt][qh][r]);
            vl[qh] = v;
            up = up || v > up_at[qh];
        }
        if (__builtin_amdgcn_ballot_w64(up) != 0) {
#pragma unroll
            for (int qh = 0; qh < QH; ++qh) {
                float a, b;
                f5_xor32_pair(vl[qh], a, b);
                // a query's first block with a score above -inf sets m to its maximum, later ones only raise
                // it; a block of -inf before that (keys masked by infinite operands) leaves it unset
                const bool set = m_run[qh] != -INFINITY;
                const float t = fmaxf(a, b), d = set ? fmaxf(t, 0.f) : (t == -INFINITY ? 0.f : t);
                const float alpha = set ? __builtin_amdgcn_exp2f(-d) : 1.f;
                m_run[qh] = set ? m_run[qh] + d : t;
                const bool now_set = m_run[qh] != -INFINITY;
                up_at[qh] = now_set ? F3_RESCALE : -INFINITY;
                l_run[qh] *= alpha;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    neg_m[qh][r] = now_set ? -m_run[qh] : 0.f;
                    st[0][qh][r] -= d;
                    st[1][qh][r] -= d;
                    o[0][qh][r] *= alpha;
                    o[1][qh][r] *= alpha;
                }
            }
        }
        // P of key step kk (16 keys) and its row sums
        f5_u32x4 pf[2][QH];
        auto probs = [&](int kk, int qh) __attribute__((always_inline)) {
            f5_u32x4 u;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int r0 = 8 * (kk & 1) + 2 * k;
                const f5_h2 hv = {(_Float16)__builtin_amdgcn_exp2f(st[kk >> 1][qh][r0]),
                                  (_Float16)__builtin_amdgcn_exp2f(st[kk >> 1][qh][r0 + 1])};
                l_run[qh] = __builtin_amdgcn_fdot2(hv, ones, l_run[qh], false);
                u[k] = __builtin_bit_cast(uint32_t, hv);
            }
            pf[kk & 1][qh] = u;
        };
#pragma unroll
        for (int qh = 0; qh < QH; ++qh) probs(0, qh);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
            for (int qh = 0; qh < QH; ++qh) {
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
                    o[dt][qh] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                        vf[(2 * kk + dt) & 3], __builtin_bit_cast(f16x8, pf[kk & 1][qh]), o[dt][qh], 0, 0, 0);
                if (kk < 3) probs(kk + 1, qh);
            }
            if (kk < 2) {
                vf[(2 * kk) & 3] = vread(2 * kk + 4);
                vf[(2 * kk + 1) & 3] = vread(2 * kk + 5);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    for (int j = 0; j < steps; ++j) {
        const uint32_t now = (uint32_t)((j & (F6_RING - 1)) * F6_STEP);
        dma_step(j + 2, (j + 2) & (F6_RING - 1));
        const int kb = 2 * j + kh;
        if (kb <= last) block(kb, now);
        asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)" ::: "memory");   // this wavefront's part of step j + 1 landed
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    // ---- merge.  Of its two partial results a group's wavefront kh finishes query half kh (QH = 2) or
    // columns 32 kh .. + 31 (QH = 1) and hands over the rest; a wavefront with no block or no
    // finite score has m = -inf and weighs nothing.
    constexpr int ND = QH == 2 ? 2 : 1;   // 32-column tiles this wavefront finishes
    f32x16 keep[ND];
    const int peer = w ^ 4;
    auto box = [&](int wave) { return lds_addr(&ring[0][0]) + (uint32_t)(wave * ND * 4096 + lane * 16); };
#pragma unroll
    for (int t = 0; t < ND; ++t) {
        f32x16 give;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float lo = QH == 2 ? o[t][0][r] : o[0][0][r], hi = QH == 2 ? o[t][QH - 1][r] : o[1][0][r];
            keep[t][r] = kh ? hi : lo;
            give[r] = kh ? lo : hi;
        }
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4)
            *(lds_f32x4*)(uintptr_t)(box(w) + (uint32_t)(t * 4 + g4) * 1024u) =
                f32x4{give[4 * g4], give[4 * g4 + 1], give[4 * g4 + 2], give[4 * g4 + 3]};
    }
    float l_all[QH];
#pragma unroll
    for (int qh = 0; qh < QH; ++qh) {
        float a, b;
        f5_xor32_pair(l_run[qh], a, b);
        l_all[qh] = a + b;
        if (h == 0) stat[w][qh][r32] = make_float2(m_run[qh], l_all[qh]);
    }
    __syncthreads();
    const int mq = QH == 2 ? kh : 0;
    const float m_own = QH == 2 && kh ? m_run[QH - 1] : m_run[0], l_own = QH == 2 && kh ? l_all[QH - 1] : l_all[0];
    const float2 ot = stat[peer][mq][r32];
    const float m_all = fmaxf(m_own, ot.x);
    const float a_own = __builtin_amdgcn_exp2f(m_own - m_all), a_ot = __builtin_amdgcn_exp2f(ot.x - m_all);
    const float inv = 1.f / (a_own * l_own + a_ot * ot.y);
    const float f_own = a_own * inv, f_ot = a_ot * inv;
#pragma unroll
    for (int t = 0; t < ND; ++t)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
            const f32x4 x = *(const lds_f32x4*)(uintptr_t)(box(peer) + (uint32_t)(t * 4 + g4) * 1024u);
#pragma unroll
            for (int r = 0; r < 4; ++r) keep[t][4 * g4 + r] = keep[t][4 * g4 + r] * f_own + x[r] * f_ot;
        }
    const int qs = q0 + (QH == 2 ? 32 * kh : 0), c0 = QH == 2 ? 0 : 4 * kh;   // first query, first 16-byte chunk
    if (p.o16) {
        // rows of 16 ND x 4 bytes staged behind the boxes, chunk ^ row % (4 ND), then stored whole
        constexpr int NC = 4 * ND;
        const uint32_t ep = lds_addr(&ring[0][0]) + (uint32_t)(8 * ND * 4096 + w * 32 * NC * 16);
        typedef __attribute__((address_space(3))) f16x4 lds_f16x4;
#pragma unroll
        for (int t = 0; t < ND; ++t)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const f16x4 v = {(f16)keep[t][4 * g4], (f16)keep[t][4 * g4 + 1], (f16)keep[t][4 * g4 + 2], (f16)keep[t][4 * g4 + 3]};
                *(lds_f16x4*)(uintptr_t)(ep + (uint32_t)((r32 * NC + ((4 * t + g4) ^ (r32 & (NC - 1)))) * 16 + 8 * h)) = v;
            }
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
        __builtin_amdgcn_wave_barrier();
        constexpr int RPI = 64 / NC;
        const int row = lane / NC, cc = lane % NC;
        f16x8 rv[32 / RPI];
#pragma unroll
        for (int i = 0; i < 32 / RPI; ++i)
            rv[i] = *(const lds_f16x8*)(uintptr_t)(ep + (uint32_t)(((RPI * i + row) * NC + (cc ^ ((RPI * i + row) & (NC - 1)))) * 16));
        f16* obase = Ob + (int64_t)(qs + row) * p.osl + 8 * (c0 + cc);
#pragma unroll
        for (int i = 0; i < 32 / RPI; ++i)
            if (qs + RPI * i + row < p.S && c0 + cc < dch)
                __builtin_nontemporal_store(rv[i], reinterpret_cast<f16x8*>(obase + (int64_t)(RPI * i) * p.osl));
    } else if (qs + r32 < p.S) {
        f16* orow = Ob + (int64_t)(qs + r32) * p.osl;
#pragma unroll
        for (int t = 0; t < ND; ++t)
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                const int d = 8 * (c0 + 4 * t + g4) + 4 * h;
                const f16x4 v = {(f16)keep[t][4 * g4], (f16)keep[t][4 * g4 + 1], (f16)keep[t][4 * g4 + 2], (f16)keep[t][4 * g4 + 3]};
                if (d < p.D) __builtin_nontemporal_store(v, reinterpret_cast<f16x4*>(orow + d));
            }
    }
}

// Any D <= 256, any S: one thread per query row, online softmax in fp32 over every
// key (the clamped/ragged path; not the fast one).
__global__ void flash_generic_kernel(FaParams p, int D) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t total = (int64_t)p.S * p.H * p.B;
    if (t >= total) return;
    const int qrow = (int)(t % p.S);
    const int64_t bh = t / p.S;
    const int h = (int)(bh % p.H), b = (int)(bh / p.H);
    const f16* q = p.Q + h * p.sh + b * p.sb + (int64_t)qrow * p.sl;
    const f16* Kb = p.K + h * p.sh + b * p.sb;
    const f16* Vb = p.V + h * p.sh + b * p.sb;
    float acc[256];
    for (int e = 0; e < D; ++e) acc[e] = 0.f;
    float m = -3.0e38f, l = 0.f;
    const int nk = p.causal ? qrow + 1 : p.S;
    for (int j = 0; j < nk; ++j) {
        const f16* k = Kb + (int64_t)j * p.sl;
        float s = 0.f;
        for (int e = 0; e < D; ++e) s = fmaf((float)q[e], (float)k[e], s);
        s *= p.scale_log2;
        const float mn = fmaxf(m, s);
        const float a = exp2f(m - mn), e1 = exp2f(s - mn);
        const f16* v = Vb + (int64_t)j * p.sl;
        for (int e = 0; e < D; ++e) acc[e] = acc[e] * a + e1 * (float)v[e];
        l = l * a + e1;
        m = mn;
    }
    f16* o = p.O + h * p.osh + b * p.osb + (int64_t)qrow * p.osl;
    for (int e = 0; e < D; ++e) o[e] = (f16)(acc[e] / l);
}

// The score/output kernel runs 32-query pairs (128 queries a workgroup) or 64-query ones.  A 64-key
// block costs a workgroup of 32-query pairs about 0.70 (D > 96) or 0.75
// of what it costs one of 64-query pairs, and a workgroup's start and end about 1.5 such blocks, so
// twice the workgroups pay where the wide ones leave CUs idle or, causal, the longest of them (its
// last query block's ceil(S / 64) key blocks) outlasts the rest.  Measured (us, 64- / 32-query pairs;
// causal but for the last two): B = 1, H = 32, S = 1537, D = 128 37.8 / 29.4; S = 2048 49.3 / 41.3;
// H = 8, S = 2048 44.0 / 30.1; B = 2, H = 16, S = 512 16.3 / 11.6; but B = 4, H = 32, S = 512 19.2 /
// 21.4, 1024 54.8 / 58.2, 4096 504 / 598; H = 4, S = 4096, D = 64 64.0 / 48.0; B = 4, H = 12, S = 777,
// D = 64 18.1 / 25.9.  Over 800 drawn calls the narrow pairs took 0.62 to 1.03 of the wide ones' time where they
// are estimated below 0.95 of it, 1.00 to 1.10 from there to 1 (B = 3, H = 16, S = 1300, D = 32 26.0 / 28.6; H = 32, B = 4,
// S = 380, D = 128 16.2 / 17.3), 0.93 to 1.49 above: so they need an estimate below 0.95.
//
// flash_fwd6_kernel (D = 56 and 64) takes 0.93 of that block with 64-query groups and 0.58 with 32-query
// ones, two blocks at a time, and 2.3 and 2.1 for its start and merge: (64-query pairs / 32-query pairs /
// its two widths) H = 32, B = 4, S = 4096 causal 343 / 445 / 323 / 374; B = 1, H = 32, S = 2500 not causal
// 87 / 94 / 84 / 77; B = 4, H = 12, S = 777 not causal 18.2 / 26 / 18.7 / 23.1; B = 4, H = 16, S = 300 causal
// 9.7 / 7.5 / 10.4 / 7.8.
//
// The key blocks' time on the busiest CU plus its workgroups' starts and ends, in 64-query-pair blocks;
// step: key blocks taken at a time.
static double fa_cost(int64_t S, int64_t heads, bool causal, int64_t bq, double block, double start, int64_t step) {
    const double nqb = (double)((S + bq - 1) / bq);
    const double nkb = (double)(((S + F5_BK - 1) / F5_BK + step - 1) / step * step);
    const double wgs = nqb * (double)heads, per = (double)bq / F5_BK, rounds = std::ceil(wgs / 256);
    // causal: a head's sum spread over the CUs, or its longest workgroup
    const double sum = per * nqb * (nqb + 1) / 2 - std::max(0.0, nqb * per - nkb);
    const double blocks = causal ? std::max(nkb, sum * (double)heads / 256) : rounds * nkb;
    return block * blocks + start * rounds;
}

}  // namespace lava

using namespace lava;

extern "C" int lava_hip_flash_attn_fwd_f16(const void* Q, const void* K, const void* V, void* O, int64_t B, int64_t H,
                                           int64_t S, int64_t D, const int64_t* strides, const int64_t* ostrides,
                                           float scale, int causal, void* stream) {
    LAVA_ARG(B >= 0 && H >= 0 && S >= 0 && D >= 0, "flash_attn_fwd_f16: negative extent");
    if (B == 0 || H == 0 || S == 0) return LAVA_HIP_OK;
    LAVA_ARG(D >= 1, "flash_attn_fwd_f16: D = 0 with S > 0");
    LAVA_ARG(Q && K && V && O && strides, "flash_attn_fwd_f16: null pointer");
    LAVA_ARG(scale == scale && scale != INFINITY && scale != -INFINITY, "flash_attn_fwd_f16: scale is not finite");
    const int64_t* os = ostrides ? ostrides : strides;
    LAVA_ARG(strides[0] == 1 && os[0] == 1, "flash_attn_fwd_f16: the head dimension (E) must be contiguous");
    for (int i = 1; i < 4; ++i)
        LAVA_ARG(strides[i] >= 0 && os[i] >= 0, "flash_attn_fwd_f16: negative stride %d", i);
    LAVA_ARG(strides[1] >= D && os[1] >= D, "flash_attn_fwd_f16: sequence stride smaller than D");
    LAVA_ARG(S <= 0x7fffffff && H <= 0x7fffffff && B <= 0x7fffffff, "flash_attn_fwd_f16: extent too large");
    LAVA_ARG(aligned(Q, 2) && aligned(K, 2) && aligned(V, 2) && aligned(O, 2), "flash_attn_fwd_f16: misaligned");
    LAVA_REQUIRE(D <= 256, LAVA_HIP_ERR_UNSUPPORTED, "flash_attn_fwd_f16: D = %lld > 256 is not supported",
                 (long long)D);
    int rc = lava_hip_init();
    if (rc != LAVA_HIP_OK) return rc;

    FaParams p;
    p.Q = (const f16*)Q;
    p.K = (const f16*)K;
    p.V = (const f16*)V;
    p.O = (f16*)O;
    p.sl = strides[1];
    p.sh = strides[2];
    p.sb = strides[3];
    p.osl = os[1];
    p.osh = os[2];
    p.osb = os[3];
    p.S = (int)S;
    p.H = (int)H;
    p.B = (int)B;
    p.scale_log2 = scale * 1.4426950408889634f;
    p.causal = causal != 0;
    p.o16 = aligned(O, 16) && os[1] % 8 == 0 && os[2] % 8 == 0 && os[3] % 8 == 0;
    p.D = (int)D;
    p.dv = (int)D;
    hipStream_t s = as_stream(stream);

    // D <= 128 (a multiple of 8) with 16-byte rows, and D = 256: the MFMA kernels.  D <= 128 runs
    // on flash_fwd5_kernel (score/output wavefront pairs, rows staged zero-padded to 128, MFMAs over
    // D rounded up to 64, 96 or 128; the scale folds into Q^T, so any sign; at D = 64 it runs
    // 1.2x flash_fwd3_kernel, 837 against 682 TFLOP/s causal at B=4 H=32 S=4096), D = 256 with a
    // positive scale on flash_fwd3_kernel (ping-pong wavefront pairs; its base-2 running maximum
    // assumes one); all take any S (a ragged last block of queries or keys is zero-filled and
    // masked).  lava_hip_set_kernel_override(LAVA_HIP_FAMILY_ATTN, 3) pins flash_fwd3_kernel for
    // D = 64 and 128 with a positive scale (tests and A/B timing).  Everything else runs on
    // flash_generic_kernel.
    bool lay_ok = D >= 8 && D <= FA_D && D % 8 == 0 && strides[0] == 1 && os[0] == 1;
    for (int i = 1; i < 4; ++i) lay_ok = lay_ok && strides[i] % 8 == 0 && os[i] % 4 == 0;
    lay_ok = lay_ok && aligned(Q, 16) && aligned(K, 16) && aligned(V, 16) && aligned(O, 8) &&
             S * strides[1] * 2 < ((int64_t)1 << 31);
    const int64_t blocks3 = ((S + F3_BQ - 1) / F3_BQ) * H * B;
    const int64_t blocks5 = ((S + 32 * F5_PAIRS - 1) / (32 * F5_PAIRS)) * H * B;   // with 32-query pairs, the most
    const int pin = kernel_override(LAVA_HIP_FAMILY_ATTN);
    const bool fast3 = lay_ok && scale > 0.f && (D == 64 || D == FA_D) && pin == 3 && blocks3 <= 0x7fffffff;
    const bool fast5 = lay_ok && !fast3 && blocks5 <= 0x7fffffff;
    // 128 < D <= 256 (a multiple of 8) with a positive scale: the ping-pong kernel over Q/K rows
    // zero-padded to 256, once per 128-column half of V and O (the scores are computed twice)
    bool fast256 = D > FA_D && D <= 256 && D % 8 == 0 && scale > 0.f && strides[0] == 1 && os[0] == 1 &&
                   blocks3 <= 0x7fffffff &&
                   aligned(Q, 16) && aligned(K, 16) && aligned(V, 16) && aligned(O, 8) &&
                   S * strides[1] * 2 < ((int64_t)1 << 31);
    for (int i = 1; i < 4; ++i) fast256 = fast256 && strides[i] % 8 == 0 && os[i] % 4 == 0;
    const double cost5w = fa_cost(S, H * B, p.causal, 64 * F5_PAIRS, 1.0, 1.5, 1);
    const double cost5n = fa_cost(S, H * B, p.causal, 32 * F5_PAIRS, D > 96 ? 0.70 : 0.75, 1.5, 1);
    if (fast5 && pin == 0 && D > 48 && D <= 64 && scale > 0.f && p.scale_log2 <= 1.f) {
        const double cost6w = fa_cost(S, H * B, p.causal, 64 * F6_GROUPS, 0.93, 2.3, 2);
        const double cost6n = fa_cost(S, H * B, p.causal, 32 * F6_GROUPS, 0.58, 2.1, 2);
        if (std::min(cost6w, cost6n) < 0.96 * std::min(cost5w, cost5n)) {   // (the estimates hold to a few percent)
            auto go = [&](auto kernel, int64_t bq) {
                hipLaunchKernelGGL(kernel, dim3((unsigned)(((S + bq - 1) / bq) * H * B)), dim3(128 * F6_GROUPS), 0, s, p);
            };
            if (cost6n < cost6w)
                p.causal ? go(flash_fwd6_kernel<true, 1>, 32 * F6_GROUPS) : go(flash_fwd6_kernel<false, 1>, 32 * F6_GROUPS);
            else
                p.causal ? go(flash_fwd6_kernel<true, 2>, 64 * F6_GROUPS) : go(flash_fwd6_kernel<false, 2>, 64 * F6_GROUPS);
            LAVA_LAUNCH_CHECK(cost6n < cost6w ? "flash_fwd6_kernel+flash_fwd6_kernel<32>" : "flash_fwd6_kernel");
            return LAVA_HIP_OK;
        }
    }
    if (fast5) {   // any D <= 128, a multiple of 8 (staged zero-padded to 128; MFMAs over D rounded up to 64, 96, 128)
        auto go = [&](auto kernel, int64_t blocks) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(128 * F5_PAIRS), 0, s, p);
        };
        auto by_d = [&](auto causal_tag, auto qh_tag) {
            constexpr bool C = decltype(causal_tag)::value;
            constexpr int QH = decltype(qh_tag)::value;
            const int64_t blocks = ((S + 32 * QH * F5_PAIRS - 1) / (32 * QH * F5_PAIRS)) * H * B;
            if (D <= 64) go(flash_fwd5_kernel<C, 64, QH>, blocks);
            else if (D <= 96) go(flash_fwd5_kernel<C, 96, QH>, blocks);
            else go(flash_fwd5_kernel<C, 128, QH>, blocks);
        };
        const bool narrow = cost5n < 0.95 * cost5w;
        typedef std::integral_constant<int, 1> Q1;
        typedef std::integral_constant<int, 2> Q2;
        if (p.causal)
            narrow ? by_d(f3_tag<true>{}, Q1{}) : by_d(f3_tag<true>{}, Q2{});
        else
            narrow ? by_d(f3_tag<false>{}, Q1{}) : by_d(f3_tag<false>{}, Q2{});
        LAVA_LAUNCH_CHECK(narrow ? "flash_fwd5_kernel+flash_fwd5_kernel<32>" : "flash_fwd5_kernel");
        return LAVA_HIP_OK;
    }
    if (fast3) {
        const dim3 grid((unsigned)blocks3);
        if (D == 64) {
            if (p.causal)
                hipLaunchKernelGGL((flash_fwd3_kernel<true, 64, 64>), grid, dim3(64 * F3_WAVES), 0, s, p);
            else
                hipLaunchKernelGGL((flash_fwd3_kernel<false, 64, 64>), grid, dim3(64 * F3_WAVES), 0, s, p);
        } else if (p.causal) {
            hipLaunchKernelGGL((flash_fwd3_kernel<true, 128, 128>), grid, dim3(64 * F3_WAVES), 0, s, p);
        } else {
            hipLaunchKernelGGL((flash_fwd3_kernel<false, 128, 128>), grid, dim3(64 * F3_WAVES), 0, s, p);
        }
        LAVA_LAUNCH_CHECK("flash_fwd3_kernel");
        return LAVA_HIP_OK;
    }
    if (fast256) {
        // two launches, each over the full 256-wide scores and one 128-column half of V and O
        const dim3 grid((unsigned)blocks3);
        for (int half = 0; half < 2; ++half) {
            FaParams ph = p;
            ph.V = p.V + 128 * half;
            ph.O = p.O + 128 * half;
            ph.dv = (int)(D - 128 * half < 128 ? D - 128 * half : 128);
            if (p.causal)
                hipLaunchKernelGGL((flash_fwd3_kernel<true, 256, 128>), grid, dim3(64 * F3_WAVES), 0, s, ph);
            else
                hipLaunchKernelGGL((flash_fwd3_kernel<false, 256, 128>), grid, dim3(64 * F3_WAVES), 0, s, ph);
            LAVA_LAUNCH_CHECK("flash_fwd3_kernel");
        }
        return LAVA_HIP_OK;
    }
    const int64_t rows = S * H * B;
    LAVA_REQUIRE((rows + 63) / 64 <= 0x7fffffff, LAVA_HIP_ERR_UNSUPPORTED, "flash_attn_fwd_f16: problem too large");
    hipLaunchKernelGGL(flash_generic_kernel, dim3((unsigned)((rows + 63) / 64)), dim3(64), 0, s, p, (int)D);
    LAVA_LAUNCH_CHECK("flash_generic_kernel");
    return LAVA_HIP_OK;
}
