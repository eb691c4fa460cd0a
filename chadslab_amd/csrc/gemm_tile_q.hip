// Dequant-GEMM for many activation rows:  y[m,n] = sum_k x[m,k] * w[n,k],  x bf16 [M,K], int4 group-32 or int8 per-row
// weights, fp32 accumulation on v_mfma_f32_32x32x16_bf16.
//
// What bounds it: the matrix cores, at the clock the power of all the work leaves (1.8-1.9 GHz here, 2.4 idle), and the
// work beside them.  One wave alone on a SIMD issues a vector instruction every eight cycles or so and stalls at every
// wait; two hide up to six vector instructions behind each 32-cycle MFMA (measured).  Hence eight waves per workgroup,
// two per SIMD, each with a column block of 32 weight rows and all activation rows of the tile:
//
//   256 x 256 tile   eight waves side by side (WN = 8), 128 accumulators each; every weight is dequantised once per
//                    256 activation rows.
//   128 x 128 tile   four waves side by side, twice (WN = 4, WK = 2): the two halves of the workgroup take alternate
//                    64-k blocks and meet in LDS at the end.  For grids that would leave the chip empty with the large one.
//   64 x 64 tile     two waves side by side, four times (WN = 2, WK = 4); 32 x 64 for at most 32 rows.  For few rows and for
//                    grids of one round (gemm_q_bf16.hip: takes_small_tile).
//   exact weights    (HILO) 128, 64 or 32 rows x 128 weight rows, WN = 4, WK = 2, K possibly split over workgroups.
//
//   * A (activations): global -> LDS by DMA, three stages of 64 * WK k, read back as fragments one or two slices (16 k)
//     ahead of their MFMAs.  16-byte pieces of a 128-byte row segment are XOR-swizzled by row / 2: LDS has 64 banks, two
//     segments cover them, so the key changes every second row (588 B/ns per compute unit; keyed by the row itself, 294).
//   * B (weights): the packed bytes take the same road; lane (n, kq) reads back 32 k of its row and dequantises them one
//     slice ahead into the MFMA operand: 17 vector instructions per 8 weights (int4) or 12 (int8).
//   * int4 scales: 16 bytes (8 groups = 256 k) per row by DMA into an area of the wave's own, or, where K is no multiple
//     of 256, two bytes per lane and step.
//   * One barrier per step, in front of the last slices, whose fragments are in registers by then.
// The order inside a slice is given to the compiler's scheduler: left alone it issues all MFMAs of a slice, then all of
// the dequantisation, and the two waves of a SIMD, which the barrier keeps in step, do the same thing at the same time.
//
// Measured (us; the one-wave-per-SIMD tile and the 128 x 64 kernel this replaced at these sizes in brackets):
//   int4 4096 x 14336 x 4096: 409 (486)   4096^3: 113 (129)   1000 x 4096 x 14336: 116 (143)   256 x 14336 x 4096: 33 (44)
//   int8 4096^3: 110 (191)   1000 x 4096 x 14336: 111 (160)   512 x 4096 x 4096: 26.5 (27.4)
// (the vendor's GEMM on bf16 weights: 328, 87, 113, 40; 88, 112, 25).  Tried and not kept: waves of 128 x 64 (every weight
// dequantised by two waves), four-wave workgroups of 128 x 256, two per compute unit (both 2-4 % slower), waves that
// alternate between a phase of MFMAs and one of LDS reads and dequantisation, the two of a SIMD in opposite phases (the
// same time: what is left is power, not order - fed zeros, the same kernel takes 95 us at 4096^3).
//
// HILO: the dequantised weight is kept exactly, as the sum of two bf16 operands (a 4-bit integer times an fp16 scale has
// at most 15 significant bits), for callers that must not round weights; twice the matrix work.
// The MFMA k-slot of a lane is free as long as A and B agree: slot group kq of slice t holds k = 32 kq + 8 t .. +7.
#include <type_traits>

#include "chadq_common.h"
#include "gemm_tile_q.h"

namespace chadq {
namespace tileq {

constexpr int kStages = 3;

template <bool I4, int WN, int WK, int WMB, bool GUARD>
struct Cfg {
    static constexpr int NW = WN * WK, T = 64 * NW;
    static constexpr int BM = 32 * WMB, BN = 32 * WN, KS = 64 * WK;  // tile, k per step
    static constexpr int BB = (I4 ? 32 : 64) * WK;                   // packed bytes of a weight row per step
    static constexpr int A_STAGE = BM * 128 * WK, B_STAGE = BN * BB, STAGE = A_STAGE + B_STAGE;
    static constexpr int A_DMA = A_STAGE / (NW * 1024), B_DMA = B_STAGE / (NW * 1024);  // instructions per wave and step
    static_assert(A_DMA * NW * 1024 == A_STAGE && B_DMA * NW * 1024 == B_STAGE, "whole DMA instructions per wave");
    static constexpr int S_OFF = kStages * STAGE;
    // scales of a wave, two buffers: 256 k (32 rows x 16 B, fetched twice), or (GUARD) one step (64 lanes x 4 B)
    static constexpr int S_BUF = !I4 ? 0 : GUARD ? 256 : 1024, S_WAVE = 2 * S_BUF;
    static constexpr int SPB = 4 / WK;                               // steps per 256 k
    static constexpr int EP_PITCH = BN * 2 + 16;                     // result tile in LDS: bf16 rows, padded
    static constexpr int OPER = S_OFF + NW * S_WAVE, EPI = BM * EP_PITCH, RED = WK == 4 ? BM * BN * 16 : WK > 1 ? BM * BN * 4 : 0;
    static constexpr int LDS0 = OPER > EPI ? OPER : EPI, LDS = LDS0 > RED ? LDS0 : RED;
    static constexpr int AHEAD = WMB > 4 ? 1 : 2;  // slices between a fragment's request and its MFMAs (what the registers allow)
    static_assert(LDS <= 163840, "one workgroup per compute unit");
};

// The bare barrier instruction (__syncthreads() would also wait for every outstanding request); the empty asm statements
// keep the compiler from moving LDS accesses across it.
__device__ __forceinline__ void wg_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// 8 signed bytes (two words) -> 8 bf16, exact: an integer up to 127 has its low 16 fp32 bits zero
__device__ __forceinline__ bf16x8 dequant8_i8(uint32_t a, uint32_t b) {
    float f[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        f[e] = (float)(int8_t)(a >> (8 * e));
        f[4 + e] = (float)(int8_t)(b >> (8 * e));
    }
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = __builtin_amdgcn_perm(__float_as_uint(f[2 * e + 1]), __float_as_uint(f[2 * e]), 0x07060302u);
    bf16x8 o;
    __builtin_memcpy(&o, &r, 16);
    return o;
}

// dequant8_i4 with nothing rounded: hi = the value cut off after 16 bits, lo = the rest (at most 8 bits)
__device__ __forceinline__ void dequant8_i4_exact(uint32_t w, const float (&cs)[4], uint32_t mlo, uint32_t mhi, uint32_t magic, bf16x8 &hi,
                                                  bf16x8 &lo) {
    const f16x2 h0 = as_f16x2(and_or(w, mlo, magic)), h1 = as_f16x2(and_or(w, mhi, magic));
    const uint32_t w8 = w >> 8;
    const f16x2 h2 = as_f16x2(and_or(w8, mlo, magic)), h3 = as_f16x2(and_or(w8, mhi, magic));
    float f[8];
    f[0] = __builtin_fmaf((float)h0.x, cs[0], cs[2]), f[4] = __builtin_fmaf((float)h0.y, cs[0], cs[2]);
    f[1] = __builtin_fmaf((float)h1.x, cs[1], cs[3]), f[5] = __builtin_fmaf((float)h1.y, cs[1], cs[3]);
    f[2] = __builtin_fmaf((float)h2.x, cs[0], cs[2]), f[6] = __builtin_fmaf((float)h2.y, cs[0], cs[2]);
    f[3] = __builtin_fmaf((float)h3.x, cs[1], cs[3]), f[7] = __builtin_fmaf((float)h3.y, cs[1], cs[3]);
    uint32_t h[4], l[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t u0 = __float_as_uint(f[2 * e]), u1 = __float_as_uint(f[2 * e + 1]);
        h[e] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
        const float r0 = f[2 * e] - __uint_as_float(u0 & 0xFFFF0000u), r1 = f[2 * e + 1] - __uint_as_float(u1 & 0xFFFF0000u);
        l[e] = __builtin_amdgcn_perm(__float_as_uint(r1), __float_as_uint(r0), 0x07060302u);
    }
    __builtin_memcpy(&hi, h, 16);
    __builtin_memcpy(&lo, l, 16);
}

// EPI (what becomes of the sums): EPI_BF16 y bf16 [M,N], times the row scale for int8; EPI_F32 y fp32 [gridDim.y][M,N],
// part blockIdx.y holding the sum over its kspan k; EPI_GEGLU the weight rows come in pairs (gate, up) of a feature and
// h = bf16(gelu_tanh(gate) * up) goes to y as bf16 [M, N/2].
template <bool I4, int WN, int WK, int WMB, bool GUARD, bool HILO, int EPI>
__global__ __launch_bounds__(64 * WN * WK) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_tile_q_kernel(
    const uint16_t *__restrict__ x, const uint8_t *__restrict__ wq, const void *__restrict__ scv, void *__restrict__ yv, int M, int N,
    int K, int kspan) {
    typedef Cfg<I4, WN, WK, WMB, GUARD> C;
    constexpr int BM = C::BM, BN = C::BN, BB = C::BB, AHEAD = C::AHEAD;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 31, kq = lane >> 5;
    const int wk = wave / WN, wn = wave % WN;
    // workgroup i runs on XCD i % 8: deal the tiles so that one XCD walks consecutive n-tiles of the same m-panel
    const int tiles_n = (N + BN - 1) / BN, tiles = tiles_n * ((M + BM - 1) / BM);
    const int per_xcd = (tiles + 7) / 8;
    const int tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (tile >= tiles) return;
    const int m0 = (tile / tiles_n) * BM, n0 = (tile % tiles_n) * BN;
    const int kbeg = EPI == EPI_BF16 ? 0 : blockIdx.y * kspan;                                        // a multiple of 256
    const int kn = EPI == EPI_BF16 ? K : (K - kbeg < kspan ? K - kbeg : kspan);                       // k of this workgroup
    const int G = K >> 5, steps = (kn + C::KS - 1) / C::KS;
    const int wrow = I4 ? K >> 1 : K;  // bytes of a weight row

    // ---- requests.  Buffer form of the DMA: the tile's first row in a resource descriptor, the lane's place in a 32-bit
    // offset that never changes, the step in the scalar offset.  A row past the matrix is requested beyond the
    // descriptor's range and arrives as zeros (its products are not stored; multipliers fed zeros draw less power).
    const int mrows = M - m0 < BM ? M - m0 : BM, nrows = N - n0 < BN ? N - n0 : BN;
    const __amdgpu_buffer_rsrc_t arsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(x) + (size_t)m0 * K, 0, mrows * K * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t brsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(wq) + (size_t)n0 * wrow, 0, nrows * wrow, 0x00020000);
    constexpr uint32_t kOut = 0x80000000u;
    uint32_t aoff[C::A_DMA], boff[C::B_DMA];
    int apc[C::A_DMA], bpc[C::B_DMA];
    constexpr int BPR = BB / 16;  // 16-byte pieces per weight row and step
    // WK = 4: a row's 128 or 256 bytes span half or all of the banks, so its pieces are XOR-swizzled by the row as A's are
    auto bkey = [](int r) { return WK < 4 ? 0 : BPR == 8 ? (r >> 1) & 7 : r & 15; };
#pragma unroll
    for (int q = 0; q < C::A_DMA; ++q) {  // 8 row segments of 128 B per instruction, [k half][row][128 B]
        const int e = (q * C::NW + wave) * 8 + (lane >> 3), r = e % BM;
        apc[q] = e / BM * 128 + 16 * ((lane & 7) ^ ((r >> 1) & 7));
        aoff[q] = r < mrows ? (uint32_t)r * (uint32_t)(K * 2) + (uint32_t)apc[q] : kOut;
    }
#pragma unroll
    for (int q = 0; q < C::B_DMA; ++q) {  // 64 / BPR rows per instruction
        const int r = (q * C::NW + wave) * (64 / BPR) + lane / BPR;
        bpc[q] = 16 * ((lane % BPR) ^ bkey(r));
        boff[q] = r < nrows ? (uint32_t)r * (uint32_t)wrow + (uint32_t)bpc[q] : kOut;
    }
    const uint16_t *srow = nullptr;
    if constexpr (I4) {
        const int n = n0 + wn * 32 + nl;
        srow = reinterpret_cast<const uint16_t *>(scv) + (size_t)(n < N ? n : N - 1) * G + (kbeg >> 5);
    }
    uint8_t *const slds = lds + C::S_OFF + wave * C::S_WAVE;

    auto dma = [&](const __amdgpu_buffer_rsrc_t &rsrc, uint32_t voff, int soff, uint8_t *dst) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)dst, 16, voff, soff, 0, 0);
    };
    // GUARD: a piece past the end of its row is not fetched (zeros); whole pieces: K % 32 == 0 (int4), K % 16 == 0 (int8)
    auto issue_a = [&](int step, int q0, int q1, uint8_t *stage) {
#pragma unroll
        for (int q = 0; q < C::A_DMA; ++q)
            if (q >= q0 && q < q1) {
                const int soff = kbeg * 2 + step * (2 * C::KS);
                dma(arsrc, GUARD && soff + apc[q] >= K * 2 ? kOut : aoff[q], soff, stage + (q * C::NW + wave) * 1024);
            }
    };
    auto issue_b = [&](int step, uint8_t *stage) {
#pragma unroll
        for (int q = 0; q < C::B_DMA; ++q) {
            const int soff = (I4 ? kbeg >> 1 : kbeg) + step * BB;
            dma(brsrc, GUARD && soff + bpc[q] >= wrow ? kOut : boff[q], soff, stage + C::A_STAGE + (q * C::NW + wave) * 1024);
        }
    };
    auto issue_s = [&](int blk) {  // blk: 256-k block, or (GUARD) step
        if constexpr (I4 && GUARD) {
            const int g = 2 * (blk * WK + wk) + kq;
            dma2_to_lds(srow + (g < G ? g : 0), slds + (blk & 1) * C::S_BUF);
        } else if constexpr (I4) {
            dma16_to_lds(srow + blk * 8, slds + (blk & 1) * C::S_BUF);
        }
    };

    // ---- fragment read offsets: row nl of a 32-row block, piece 4 kq + t; the lane's packed weights
    uint32_t foff[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) foff[t] = (uint32_t)(wk * BM * 128 + nl * 128 + (((4 * kq + t) ^ ((nl >> 1) & 7)) << 4));
    constexpr int BQ = I4 ? 1 : 2;  // 16-byte pieces of a lane's 32 k
    uint32_t woff[BQ];
#pragma unroll
    for (int e = 0; e < BQ; ++e) woff[e] = (uint32_t)(C::A_STAGE + (wn * 32 + nl) * BB + 16 * (((2 * wk + kq) * BQ + e) ^ bkey(wn * 32 + nl)));

    const uint32_t c_mlo = vgpr_const(0x000F000Fu), c_mhi = vgpr_const(0x00F000F0u), c_magic = vgpr_const(0x64006400u);

    f32x16 acc[WMB];
#pragma unroll
    for (int a = 0; a < WMB; ++a)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[a][v] = 0.f;

    u32x4 bq[BQ];  // the lane's packed weights of a step: 32 k
    uint16_t sraw = 0;
    float cs[4];
    auto fetch = [&](int step, const uint8_t *stage) {
#pragma unroll
        for (int e = 0; e < BQ; ++e) bq[e] = *reinterpret_cast<const u32x4 *>(stage + woff[e]);
        if constexpr (I4) {
            if (GUARD) sraw = *reinterpret_cast<const uint16_t *>(slds + (step & 1) * C::S_BUF + lane * 4);
            else sraw = *reinterpret_cast<const uint16_t *>(slds + (step / C::SPB & 1) * C::S_BUF + nl * 16 + (((step * WK + wk) & 3) * 2 + kq) * 2);
        }
    };
    auto prep = [&](int step) {  // scale -> FMA constants; int4 weights past the row's end read as u = 0 and get the scale 0
        if constexpr (I4) {
            const float s = (GUARD && kbeg + step * C::KS + wk * 64 + kq * 32 >= K) ? 0.f : f16_bits_to_f32(sraw);
            cs[0] = s;
            cs[1] = s * 0.0625f;
            cs[2] = -1032.f * s;
            cs[3] = -72.f * s;
        }
    };
    bf16x8 bf[2], bl[2];
    auto deq = [&](int t) {
        if constexpr (I4 && HILO) dequant8_i4_exact(bq[0][t], cs, c_mlo, c_mhi, c_magic, bf[t & 1], bl[t & 1]);
        else if constexpr (I4) bf[t & 1] = dequant8_i4(bq[0][t], cs[0], cs[1], cs[2], cs[3], c_mlo, c_mhi, c_magic);
        else bf[t & 1] = dequant8_i8(bq[t >> 1][2 * (t & 1)], bq[t >> 1][2 * (t & 1) + 1]);
    };
    bf16x8 af[2 * AHEAD][WMB];
    auto frags = [&](int t, const uint8_t *stage) {
#pragma unroll
        for (int mb = 0; mb < WMB; ++mb) af[t % (2 * AHEAD)][mb] = *reinterpret_cast<const bf16x8 *>(stage + mb * 4096 + foff[t]);
    };

    // ---- prologue: two stages and the scales they need
    uint8_t *cur = lds, *nxt = lds + C::STAGE, *far = lds + 2 * C::STAGE;
    issue_s(0);
    if (GUARD || C::SPB == 1 ? steps > 1 : C::SPB == 2 && steps > 2) issue_s(1);
    issue_b(0, cur);
    issue_a(0, 0, C::A_DMA, cur);
    if (steps > 1) {
        issue_b(1, nxt);
        issue_a(1, 0, C::A_DMA, nxt);
        wait_vmcnt<C::A_DMA + C::B_DMA>();  // everything of step 0
    } else {
        wait_vmcnt<0>();
    }
    wg_barrier();
    fetch(0, cur);
    frags(0, cur);
    if (AHEAD == 2) frags(1, cur);
    prep(0);
    deq(0);

    // Step i works on stage `cur` = i % 3 and requests step i+2 into `far`, which held step i-1: everybody has left that
    // stage before the barrier of step i-1.  In front of the barrier a wave waits until no more than what it has
    // requested during this step is outstanding: its part of stage i+1 and of the scales is then in LDS.
    auto mfmas = [&](int t) {
#pragma unroll
        for (int mb = 0; mb < WMB; ++mb) {
            acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[t % (2 * AHEAD)][mb], bf[t & 1], acc[mb], 0, 0, 0);
            if (HILO) acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[t % (2 * AHEAD)][mb], bl[t & 1], acc[mb], 0, 0, 0);
        }
    };
    // The order inside a slice: LDS reads with the first MFMAs, memory requests and the dequantisation spread over all of
    // them (mask 8: MFMA, 2: vector ALU, 0x100: LDS read, 0x20: vector memory).
    constexpr int NM = WMB * (HILO ? 2 : 1), DQ = I4 ? (HILO ? 37 : 17) : 12;
    auto order = [&]() {
#pragma unroll
        for (int e = 0; e < NM; ++e) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (e < WMB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (e % 2 == 1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, (DQ + NM - 1) / NM, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](int i, auto more1_c, auto more2_c) {
        constexpr bool more1 = decltype(more1_c)::value, more2 = decltype(more2_c)::value;  // steps i+1, i+2 exist
        constexpr int H = (C::A_DMA + C::B_DMA + 1) / 2 - C::B_DMA;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (t == 4 - AHEAD && more1) {
                if (more2) wait_vmcnt<C::A_DMA + C::B_DMA>();
                else wait_vmcnt<0>();
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this stage has been read
                wg_barrier();
                if (GUARD || C::SPB == 1) {
                    if (more2) issue_s(i + 2);
                } else if (I4 && (i + 3) % C::SPB == 0 && i + 3 < steps) {
                    issue_s((i + 3) / C::SPB);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (t < 4 - AHEAD) frags(t + AHEAD, cur);
            if (t == 0 && more2) {
                issue_b(i + 2, far);
                issue_a(i + 2, 0, H, far);
            }
            if (t == 1 && more2) issue_a(i + 2, H < 0 ? 0 : H, C::A_DMA, far);
            mfmas(t);
            if (t < 3) deq(t + 1);
            if (t == 4 - AHEAD && more1) fetch(i + 1, nxt);
            if (t >= 4 - AHEAD && more1) frags(t + AHEAD - 4, nxt);
            if (t == 3 && more1) {
                prep(i + 1);
                deq(0);
            }
            order();
        }
        uint8_t *const r = cur;
        cur = nxt;
        nxt = far;
        far = r;
    };
    using T = std::true_type;
    using F = std::false_type;
    int i = 0;
    for (; i + 2 < steps; ++i) step(i, T{}, T{});
    if (steps > 1) step(i++, T{}, F{});
    step(i, F{}, F{});

    // ---- epilogue.  The lane holds, for every mb, column nl of rows 8*(v/4) + 4*kq + v%4 of a 32 x 32 block.
    wg_barrier();  // every wave is done with the stages, which everything below reuses
    // WK = 2: the two waves that hold the k halves of one result exchange halves of it through LDS and each finishes one:
    // lower row blocks by the first, upper ones by the second.  (A tile of one row block: its upper eight values.)
    // WK = 4: every wave leaves all of its values and finishes a quarter of the sums, added in the order of the k.
    constexpr int PARTS = WK == 4 ? 4 : WMB == 1 ? 2 : WMB;    // units of exchange: row blocks, halves of the only one, quarters
    constexpr int UV = WK == 4 ? WMB * 4 : WMB == 1 ? 8 : 16, PE = PARTS / WK;  // values per unit, units a wave finishes
    auto val = [&](int u, int v) { return WMB == 1 ? acc[0][u * 8 + v] : acc[WMB == 1 ? 0 : u][v]; };
    float res[PE][UV];
    if constexpr (WK == 2) {
        float *const red = reinterpret_cast<float *>(lds) + wn * (WMB * 1024) + lane * 4;
#pragma unroll
        for (int u = 0; u < PE; ++u)
#pragma unroll
            for (int q = 0; q < UV / 4; ++q) {
                f32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = wk ? val(u, 4 * q + e) : val(PE + u, 4 * q + e);
                *reinterpret_cast<f32x4 *>(red + ((wk * PE + u) * (UV / 4) + q) * 256) = o;
            }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < PE; ++u)
#pragma unroll
            for (int q = 0; q < UV / 4; ++q) {
                const f32x4 o = *reinterpret_cast<const f32x4 *>(red + (((1 - wk) * PE + u) * (UV / 4) + q) * 256);
#pragma unroll
                for (int e = 0; e < 4; ++e) res[u][4 * q + e] = (wk ? val(PE + u, 4 * q + e) : val(u, 4 * q + e)) + o[e];
            }
        __syncthreads();
    } else if constexpr (WK == 4) {
        float *const red = reinterpret_cast<float *>(lds) + lane * 4;
#pragma unroll
        for (int q = 0; q < WMB * 4; ++q) {
            const f32x4 o = {acc[q / 4][q % 4 * 4], acc[q / 4][q % 4 * 4 + 1], acc[q / 4][q % 4 * 4 + 2], acc[q / 4][q % 4 * 4 + 3]};
            *reinterpret_cast<f32x4 *>(red + (wave * WMB * 4 + q) * 256) = o;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < UV / 4; ++q) {
            f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < WK; ++w) o += *reinterpret_cast<const f32x4 *>(red + ((w * WN + wn) * WMB * 4 + wk * (UV / 4) + q) * 256);
#pragma unroll
            for (int e = 0; e < 4; ++e) res[0][4 * q + e] = o[e];
        }
        __syncthreads();
    } else {
#pragma unroll
        for (int u = 0; u < PE; ++u)
#pragma unroll
            for (int v = 0; v < UV; ++v) res[u][v] = val(u, v);
    }
    const int u0 = wk * PE;  // the wave's first unit
    auto row_of = [&](int u, int v) {
        if (WK == 4) {
            const int f = u0 * UV + v, vv = f & 15;
            return (f >> 4) * 32 + 8 * (vv >> 2) + 4 * kq + (vv & 3);
        }
        const int vv = WMB == 1 ? (u0 + u) * 8 + v : v;
        return (WMB == 1 ? 0 : (u0 + u) * 32) + 8 * (vv >> 2) + 4 * kq + (vv & 3);
    };
    if constexpr (EPI == EPI_F32) {  // 128 contiguous bytes per row straight from the registers
        float *const y = reinterpret_cast<float *>(yv) + (size_t)blockIdx.y * M * N;
        const int n = n0 + wn * 32 + nl;
#pragma unroll
        for (int u = 0; u < PE; ++u)
#pragma unroll
            for (int v = 0; v < UV; ++v) {
                const int m = m0 + row_of(u, v);
                if (m < M && n < N) y[(size_t)m * N + n] = res[u][v];
            }
        return;
    }
    // bf16 results leave through a tile in LDS, as whole rows: neighbouring lanes first swap one value of each row pair
    // (one DPP move), so that a lane writes two adjacent columns of one row as a 32-bit word - or forms the gated value
    // of one feature of one row - and the tile is then read back 16 bytes per thread.
    constexpr bool GE = EPI == EPI_GEGLU;
    constexpr int EP = C::EP_PITCH;
    const bool odd = lane & 1;
    float colscale = 1.f;
    if constexpr (!I4) {
        const int n = n0 + wn * 32 + nl;
        colscale = reinterpret_cast<const float *>(scv)[n < N ? n : N - 1];
    }
#pragma unroll
    for (int u = 0; u < PE; ++u)
#pragma unroll
        for (int v = 0; v < UV; v += 2) {
            float a0 = res[u][v], a1 = res[u][v + 1];  // rows r and r+1, column nl
            if constexpr (!I4) {
                a0 *= colscale;
                a1 *= colscale;
            }
            const float send = odd ? a0 : a1;
            const float recv = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(send), 0xB1, 0xF, 0xF, false));  // lane ^ 1
            const int row = row_of(u, v) + (odd ? 1 : 0);
            // even lane: row r, columns (nl, nl+1) = (own a0, neighbour's a0); odd lane: row r+1, columns (nl-1, nl)
            if constexpr (GE)
                *reinterpret_cast<uint16_t *>(lds + row * EP + (wn * 16 + (nl >> 1)) * 2) =
                    (uint16_t)f32_to_bf16_bits(gelu_tanh_dev(odd ? recv : a0) * (odd ? a1 : recv));
            else
                *reinterpret_cast<uint32_t *>(lds + row * EP + (wn * 32 + (nl & ~1)) * 2) = odd ? pack_bf16_rne(recv, a1) : pack_bf16_rne(a0, recv);
        }
    __syncthreads();
    uint16_t *const y = reinterpret_cast<uint16_t *>(yv);
    constexpr int COLS = GE ? BN / 2 : BN, LPR = COLS / 8;  // 16-byte pieces (lanes) per tile row
    const int NO = GE ? N >> 1 : N, c0 = GE ? n0 >> 1 : n0;
    const bool y_vec = ((NO & 7) == 0) && ((reinterpret_cast<uintptr_t>(y) & 15u) == 0);
    for (int p = tid; p < BM * LPR; p += C::T) {
        const int row = p / LPR, c8 = (p % LPR) * 8, m = m0 + row, n = c0 + c8;
        if (m >= M) continue;
        const u32x4 o = *reinterpret_cast<const u32x4 *>(lds + row * EP + c8 * 2);
        uint16_t *const yp = y + (size_t)m * NO + n;
        if (y_vec && n + 8 <= NO) {
            *reinterpret_cast<u32x4 *>(yp) = o;
        } else {
            for (int e = 0; e < 8; ++e)
                if (n + e < NO) yp[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
        }
    }
}

template <bool I4, int WN, int WK, int WMB, bool GUARD, bool HILO = false, int EPI = EPI_BF16>
static int launch(const uint16_t *x, const uint8_t *wq, const void *sc, void *y, int M, int N, int K, int ksplit, hipStream_t st) {
    typedef Cfg<I4, WN, WK, WMB, GUARD> C;
    static std::atomic<bool> attr_set{false};  // setting it twice from two threads is harmless
    if (!attr_set.load(std::memory_order_acquire)) {
        CHADQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_tile_q_kernel<I4, WN, WK, WMB, GUARD, HILO, EPI>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS));
        attr_set.store(true, std::memory_order_release);
    }
    const int tiles = ((N + C::BN - 1) / C::BN) * ((M + C::BM - 1) / C::BM);
    hipLaunchKernelGGL((gemm_tile_q_kernel<I4, WN, WK, WMB, GUARD, HILO, EPI>), dim3((tiles + 7) / 8 * 8, ksplit), dim3(C::T), C::LDS, st, x,
                       wq, sc, y, M, N, K, K / ksplit);
    return hip_check(hipGetLastError(), "gemm_tile_q launch");
}

}  // namespace tileq

// A tile's byte offsets are signed 32-bit in the descriptor: 256 rows of the wider matrix stay below 2 GiB.
bool gemm_tile_q_ok(int K) { return K < (1 << 22); }

int gemm_tile_i4g32_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, uint16_t *y, int M, int N, int K, bool big,
                           hipStream_t st) {
    const bool guard = K % 256 != 0 || !aligned16(sc);  // 16 bytes of scales at a time want aligned rows of them
    if (big)
        return guard ? tileq::launch<true, 8, 1, 8, true>(x, wp, sc, y, M, N, K, 1, st) : tileq::launch<true, 8, 1, 8, false>(x, wp, sc, y, M, N, K, 1, st);
    return guard ? tileq::launch<true, 4, 2, 4, true>(x, wp, sc, y, M, N, K, 1, st) : tileq::launch<true, 4, 2, 4, false>(x, wp, sc, y, M, N, K, 1, st);
}

int gemm_tile_i8row_launch(const uint16_t *x, const int8_t *w8, const float *sc, uint16_t *y, int M, int N, int K, bool big, hipStream_t st) {
    const uint8_t *w = reinterpret_cast<const uint8_t *>(w8);
    if (big)
        return K % 64 ? tileq::launch<false, 8, 1, 8, true>(x, w, sc, y, M, N, K, 1, st) : tileq::launch<false, 8, 1, 8, false>(x, w, sc, y, M, N, K, 1, st);
    return K % 128 ? tileq::launch<false, 4, 2, 4, true>(x, w, sc, y, M, N, K, 1, st) : tileq::launch<false, 4, 2, 4, false>(x, w, sc, y, M, N, K, 1, st);
}

// At most 64 rows, or few enough tiles for one round: 32 or 64 rows x 64 weight rows, the eight waves two side by side and
// four along K (256 k per step).
// What bounds it is the operands' way into the compute unit: at 48 x 14336 x 4096 a workgroup pulls 393 KB of activations and
// 147 KB of weights and scales, and these requests alone, nothing computed, take 10.1 of its 13.5 us in a queue of launches
// (2.2 of them the launch; the weights alone 6.2).  As many weight rows per workgroup as the 128 x 64 kernel has (one
// round of the chip up to 16384 of them), but twice the waves, a quarter of the steps and no padding to 128 rows.
// us (the 128 x 64 kernel in brackets): int4 48 x 14336 x 4096 13.5 (21.0), 17 x 4096 x 4096 9.7 (18.1), 64 x 2048 x 14336
// 36 (52), 64 x 32768 x 4096 28 (42), 64 x 1024 x 1024 5.5 (8.6); int8 48 x 14336 x 4096 13.6 (21.7).
int gemm_tile_small_i4g32_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, uint16_t *y, int M, int N, int K, hipStream_t st) {
    const bool guard = K % 256 != 0 || !aligned16(sc);
    if (M <= 32)
        return guard ? tileq::launch<true, 2, 4, 1, true>(x, wp, sc, y, M, N, K, 1, st) : tileq::launch<true, 2, 4, 1, false>(x, wp, sc, y, M, N, K, 1, st);
    return guard ? tileq::launch<true, 2, 4, 2, true>(x, wp, sc, y, M, N, K, 1, st) : tileq::launch<true, 2, 4, 2, false>(x, wp, sc, y, M, N, K, 1, st);
}

int gemm_tile_small_i8row_launch(const uint16_t *x, const int8_t *w8, const float *sc, uint16_t *y, int M, int N, int K, hipStream_t st) {
    const uint8_t *w = reinterpret_cast<const uint8_t *>(w8);
    if (M <= 32)
        return K % 256 ? tileq::launch<false, 2, 4, 1, true>(x, w, sc, y, M, N, K, 1, st) : tileq::launch<false, 2, 4, 1, false>(x, w, sc, y, M, N, K, 1, st);
    return K % 256 ? tileq::launch<false, 2, 4, 2, true>(x, w, sc, y, M, N, K, 1, st) : tileq::launch<false, 2, 4, 2, false>(x, w, sc, y, M, N, K, 1, st);
}

// ---- exact weights (HILO), K % 256 == 0: the projections of a prompt, whose tokens must come out as the decode step's do.
// Tiles of 32, 64 or 128 rows x 128 weight rows; with few rows the weight stream decides, not the padding.
template <int EPI>
static int launch_exact(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, void *y, int M, int N, int K, int ksplit, hipStream_t st) {
    if (M <= 32) return tileq::launch<true, 4, 2, 1, false, true, EPI>(x, wp, sc, y, M, N, K, ksplit, st);
    if (M <= 64) return tileq::launch<true, 4, 2, 2, false, true, EPI>(x, wp, sc, y, M, N, K, ksplit, st);
    return tileq::launch<true, 4, 2, 4, false, true, EPI>(x, wp, sc, y, M, N, K, ksplit, st);
}

// K splits that make the launch shortest: rounds of 256 workgroups times the k of each (and what a workgroup costs
// besides, about 256 k worth).  At most kExactMaxSplits parts, each a multiple of 256 k.
int gemm_exact_splits(int M, int N, int K) {
    const int bm = M <= 32 ? 32 : M <= 64 ? 64 : 128;
    const int64_t tiles = (int64_t)((M + bm - 1) / bm) * ((N + 127) / 128);
    int best = 1;
    int64_t best_cost = 0;
    for (int s = 1; s <= kExactMaxSplits; s *= 2) {
        if (K % (s * 256) != 0) break;
        const int64_t cost = (tiles * s + 255) / 256 * (K / s + 256);
        if (s == 1 || cost < best_cost) {
            best = s;
            best_cost = cost;
        }
    }
    return best;
}

int gemm_exact_f32_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, float *y_parts, int M, int N, int K, int ksplit,
                          hipStream_t st) {
    return launch_exact<tileq::EPI_F32>(x, wp, sc, y_parts, M, N, K, ksplit, st);
}

int gemm_exact_geglu_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, uint16_t *h, int M, int N, int K, hipStream_t st) {
    return launch_exact<tileq::EPI_GEGLU>(x, wp, sc, h, M, N, K, 1, st);
}

}  // namespace chadq
