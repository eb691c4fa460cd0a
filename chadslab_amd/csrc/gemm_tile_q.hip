// Dequant-GEMM for many activation rows:  y[m,n] = sum_k x[m,k] * w[n,k],  x bf16 [M,K], int4 group-32 or int8 per-row
// weights, fp32 accumulation on v_mfma_f32_32x32x16_bf16.
//
// A workgroup's WM x WN x WK waves share a tile; a wave sums MB x NB blocks of 32 x 32, so that every weight it dequantises meets
// 32 * MB activation rows; the WK waves of one result take KW (64 or 32) of a step's k each and meet in LDS at the end.
//
//   256 x 256        WN = 8, MB = 8: eight waves side by side (or, exact weights and fewer rows, see the end of the file)
//   256, 192 x 128   WM = WN = WK = 2, MB = 4 or 3, NB = 2
//   128 x 128        int4: WN = 4, WK = 2, MB = 4; int8: WN = 2, WK = 4, MB = 4, NB = 2.   96 x 128: the latter with MB = 3
//   128, 96 x 64     WN = 2, WK = 4, MB = 4 or 3, 32 k per wave and step.   64, 32 x 64: MB = 2 or 1, 64 k
//   exact weights    256, 128 x 128: WN = 4, WK = 2, MB = 8 or 4.  128, 64, 32 x 64: WN = 2, WK = 4; K possibly split over workgroups
//   SHORT            32, 64 x 64, 128 x 128 (WN = 4, WK = 2, MB = 4) and, int4, 256 x 256 with another loop, for few steps (short_k)
//
//   * A (activations): global -> LDS by DMA, ST stages of a step each, read back as fragments one or two slices (16 k)
//     ahead of their MFMAs.  16-byte pieces of a 128-byte row segment are XOR-swizzled by row / 2: LDS has 64 banks, two
//     segments cover them, so the key changes every second row (600 B/ns per compute unit; keyed by the row itself, 300).
//   * B (weights): the packed bytes take the same road, one step further ahead; a lane reads the k of its row for the next step at
//     the beginning of this one and dequantises them one slice ahead into the MFMA operand: 17 vector instructions per 8
//     weights (int4) or 12 (int8).  int4 scales travel with them, the 16 bytes (256 k) that hold the step's, or, where K is no
//     multiple of 256, two bytes per lane.
//   * One barrier per step, in front of the last slices, whose fragments are in registers by then.
//
// What bounds it.  Large products: the matrix cores at the clock the power of all the work leaves (1.7 GHz; the counters have the
// 256 x 256 tile at 68 % of its cycles in MFMAs; fed zeros 4096^3 takes 84 us, with data 113).  One round or less of small tiles: the
// order of a wave's own instructions.  A wave issues one every four cycles at best, two of them on a SIMD run in step because of the
// barrier, and whatever stands between two MFMAs stops both.  Hence a loop body without a branch (every wave requests the same
// number of pieces, surplus ones into a place nobody reads), the requests dealt out one behind each MFMA (forty in a row behind the
// barrier: +3 us of 24 at 512 x 4096 x 4096), the packed weights a step ahead (their LDS latency stood in front of the
// dequantisation), stages as constants in an unrolled loop.  128 x 4096 x 4096, one tile on a quarter of the chip: 20.9 -> 17.1 us.
// The requests alone take 13.8 us of the 22 at 512 rows; starting each workgroup at another k (16.4 -> 13.8 for them) gives the
// whole kernel nothing.
// The order inside a slice is given to the compiler's scheduler: left alone it issues all MFMAs of a slice, then all of
// the dequantisation, and the two waves of a SIMD do the same thing at the same time.
//
// Measured (us; the same tiles with the requests behind the barrier, or the 128 x 64 kernel of gemm_q_bf16.hip, in brackets):
//   int4 512 x 4096 x 4096 22.2 (23.7)   1000 x 4096 x 14336 112 (118)   48 x 14336 x 4096 14.5 (15.8)   968 x 3200 x 7552 55 (55)
//   3318 x 1792 x 3328 44 (54)   265 x 12544 x 1536 20 (28)   4096^3 114 (116)   4096 x 14336 x 4096 425 (420)
//   int8 512 x 4096 x 4096 21.4 (28.0)   1000 x 4096 x 14336 107 (115)   858 x 6656 x 13408 174 (202)   1800 x 1664 x 15360 85 (101)
// (the vendor's GEMM on bf16 weights: 512 x 4096 x 4096 25, 1000 x 4096 x 14336 112, 4096^3 88, 4096 x 14336 x 4096 328).
// Tried and not kept: NB = 2 for the 256 x 256 tile (half the fragment reads, twice the dequantisation: 117-118 us at 4096^3), four
// waves of 256 x 64 with 512 registers (115 there, but 10 % slower in a round that is not full), 64 x 128 tiles (25 us at 512 rows),
// four-wave workgroups for the 128-row tiles (the same time), a stage more (the same), a stage less (28 us)  For few steps:
// one body for all of them with its conditions at run time (24 x 1024 x 1120 6.5 us, five bodies 5.8, SHORT 5.2), no unrolled loop, no
// second request of the last step's weights (both nothing from two steps on).
//
// EXACT: no weight is rounded, for callers whose sums must be those of the decode step.  The operands are integers: (u - 8) / 2^4 in products of whole
// steps, whose activations carry the factor 2^-5 (kExactX), (u - 8) / 2^9 in guarded ones, whose activations are plain; the scale of a group of 32 k
// is applied to its sum, one fp32 FMA per value.
// Unpacking takes 14 instructions per 8 weights in the former (signed nibbles to fp32, the upper halves paired), 19
// in the latter (by way of e4m3): gate/up of a 2048 x 16384 layer, 24 / 100 / 256 tokens 16.6 -> 15 / 30.2 -> 29 / 50.4 -> 43-46 us in a stream of that
// product alone.  What bounds it is everything together, at the clock its power leaves (1.8 GHz): of 42 us at 256 tokens the FMAs taken out
// leave 34, the LDS reads of the activations 33, their requests 37, the unpacking 42; reading three or four row blocks ahead, other
// orders of a pair's instructions and waves of 128 x 64 (half the LDS reads, twice the unpacking: 48) give nothing.
// (An earlier form kept a weight as the sum of two bf16 operands: twice the matrix work, 63.7 us.)  A group's sum is finite for all finite
// activations (32 x 8 < 2^9), and a weight of 0 is the operand 0: a large activation beside it leaves the other products their low bits.
// The MFMA k-slot of a lane is free as long as A and B agree: slot group kq of slice t holds k = (KW / 2) kq + 8 t .. +7
// (EXACT: 16 t + 8 kq .. +7).
#include <type_traits>

#include "chadq_common.h"
#include "gemm_tile_q.h"

namespace chadq {
namespace tileq {

#ifndef CHADQ_GEMM_ABLATE
#define CHADQ_GEMM_ABLATE 0  // measurement builds only: 1 = the dequantisation compiled out (packed words go to the matrix core as they are)
#endif

// WM waves along the rows, WN along the columns, WK along k; MB x NB blocks of 32 x 32 per wave; KW k per wave and step; ST stages
// SHORT: the loop for few steps
template <bool I4, int WM, int WN, int WK, int MB, int NB, int KW, int ST, bool GUARD, bool SHORT>
struct Cfg {
    static constexpr int NW = WM * WN * WK, T = 64 * NW;
    static constexpr int BM = 32 * MB * WM, BN = 32 * NB * WN, KS = KW * WK;  // tile, k per step
    static constexpr int SL = KW / 16;                                        // slices of 16 k (one MFMA) per step
    static constexpr int BB = (I4 ? KW / 2 : KW) * WK;                        // packed bytes of a weight row per step
    static constexpr int A_STAGE = BM * KS * 2, B_STAGE = BN * BB;
    // int4 scales of a step: the 16 bytes (256 k) of every column that hold it, or (GUARD) 4 bytes per lane and block of each wave
    static constexpr int S_STAGE = !I4 || SHORT ? 0 : GUARD ? 256 * NB * NW : BN * 16;
    static constexpr int STAGE = A_STAGE + B_STAGE + S_STAGE;
    // DMA instructions per step: A_DMA of each wave for the activations; the BI of the weights and the SI of the scales are dealt
    // to the waves, as many to each (BS_DMA; what is left over fetches nothing, into a place nobody reads: every wave has the
    // same number of requests in flight, so the waits and the loop need no branch)
    static constexpr int A_DMA = A_STAGE / (NW * 1024), BI = B_STAGE / 1024, SI = GUARD ? 0 : S_STAGE / 1024;
    static constexpr int BS_DMA = (BI + SI + NW - 1) / NW, G_DMA = I4 && GUARD ? NB : 0, REQ = A_DMA + BS_DMA + G_DMA;
    static_assert(A_DMA * NW * 1024 == A_STAGE && BI * 1024 == B_STAGE, "whole DMA instructions");
    static constexpr bool DUMP = (BI + SI) % NW != 0;
    static constexpr int DUMP_OFF = ST * STAGE;
    // SHORT: the scales of a wave behind the stages, two buffers: 256 k (32 rows x 16 B, fetched twice), or (GUARD) one step (64 lanes x 4 B)
    static constexpr int S_BUF = !I4 || !SHORT ? 0 : GUARD ? 256 : 1024, S_OFF = ST * STAGE;
    static_assert(!SHORT || (!DUMP && WM == 1 && NB == 1 && KW == 64 && ST == 3), "what that loop knows");
    static constexpr int SPB = 256 / KS;                                      // steps per 256 k
    static constexpr int EP_PITCH = BN * 2 + 16;                              // result tile in LDS: bf16 rows, padded
    static constexpr int OPER = ST * STAGE + (DUMP ? 1024 : 0) + 2 * NW * S_BUF, EPI = BM * EP_PITCH;
    static constexpr int RED = WK == 4 ? NW * MB * 4096 : WK == 2 ? WM * WN * MB * 4096 : 0;  // one column block at a time
    static constexpr int LDS0 = OPER > EPI ? OPER : EPI, LDS = LDS0 > RED ? LDS0 : RED;
    static constexpr int AHEAD = MB * NB > 4 || SL == 2 ? 1 : 2;  // slices between a fragment's request and its MFMAs (what the registers allow)
    static_assert(LDS <= 163840, "one workgroup per compute unit");
    static_assert(ST >= 3 && ST <= 6, "the stages that the last steps know");
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

// 8 nibbles -> 8 bf16 (u - 8) / 2^9 in k order, exact: |u - 8| in a byte of its own is the e4m3 number |u - 8| / 2^9 (its low eight
// values are the subnormals, the others the next binade, with the same spacing), the sign goes above it.  19 instructions.
__device__ __forceinline__ bf16x8 signed8_i4(uint32_t w) {
    uint32_t b[2];  // bytes of u0 u2 u4 u6, of u1 u3 u5 u7
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t v = h ? w >> 4 : w, u = v & 0x0F0F0F0Fu, n = ~v & 0x08080808u, m = n >> 3;  // n: 8 where u < 8
        b[h] = ((u ^ (0x08080808u - m)) + m) | (n << 4);                                           // u - 8, or 7 - u + 1 and the sign
    }
    const uint32_t lo = __builtin_amdgcn_perm(b[1], b[0], 0x05010400u), hi = __builtin_amdgcn_perm(b[1], b[0], 0x07030602u);
    const u32x4 r = {__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, false)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, true)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, false)),
                     __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, true))};
    bf16x8 o;
    __builtin_memcpy(&o, &r, 16);
    return o;
}

// The same as (u - 8) / 2^4, for activations that carry the factor 2^-5: v_cvt_off_f32_i4 takes a signed nibble, u ^ 8, of any byte.  14
// instructions.
__device__ __forceinline__ bf16x8 signed8_i4_16th(uint32_t w) {
    const uint32_t lo = w ^ 0x88888888u;
    uint32_t hi = lo >> 4;
    asm("" : "+v"(hi));  // (else the shift is merged with that of each byte, and no byte select of the conversion is left)
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        r[e] = __builtin_amdgcn_perm(__float_as_uint(__builtin_amdgcn_cvt_off_f32_i4((hi >> (8 * e)) & 255u)),
                                     __float_as_uint(__builtin_amdgcn_cvt_off_f32_i4((lo >> (8 * e)) & 255u)), 0x07060302u);
    bf16x8 o;
    __builtin_memcpy(&o, &r, 16);
    return o;
}

// EPI (what becomes of the sums): EPI_BF16 y bf16 [M,N], times the row scale for int8; EPI_F32 y fp32 [gridDim.y][M,N],
// part blockIdx.y holding the sum over its kspan k; EPI_GEGLU the weight rows come in pairs (gate, up) of a feature and
// h = bf16(gelu_tanh(gate) * up) goes to y as bf16 [M, N/2], times the factor that the activations carry (kExactX).  EPI_QKV (WN = 2, WK = 4): as
// QkvOut says; a tile's columns are 32 of a head's first half and the 32 of its second half that they are rotated with.
// (A type of its own per epilogue: a name formed from the unnamed enumeration would not be the same for the host's and the device's compiler.)
template <int EPI>
struct MoreOut {};
template <>
struct MoreOut<EPI_QKV> : QkvOut {};
template <bool I4, int WM, int WN, int WK, int MB, int NB, int KW, int ST, bool GUARD, bool EXACT, int EPI, bool SHORT>
__global__ __launch_bounds__(64 * WM * WN * WK) __attribute__((amdgpu_waves_per_eu(WM * WN * WK / 4, WM * WN * WK / 4))) void gemm_tile_q_kernel(
    const uint16_t *__restrict__ x, const uint8_t *__restrict__ wq, const void *__restrict__ scv, void *__restrict__ yv, int M, int N,
    int K, int kspan, MoreOut<EPI> qkv) {
    typedef Cfg<I4, WM, WN, WK, MB, NB, KW, ST, GUARD, SHORT> C;
    constexpr int BM = C::BM, BN = C::BN, BB = C::BB, AHEAD = C::AHEAD, SL = C::SL;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nl = lane & 31, kq = lane >> 5;
    const int wn = wave % WN, wm = wave / WN % WM, wk = wave / (WN * WM);
    // workgroup i runs on XCD i % 8: deal the tiles so that one XCD walks consecutive n-tiles of the same m-panel
    const int tiles_n = (N + BN - 1) / BN, tiles = tiles_n * ((M + BM - 1) / BM);
    const int per_xcd = (tiles + 7) / 8;
    const int tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (tile >= tiles) return;
    const int m0 = (tile / tiles_n) * BM;
    int n0 = (tile % tiles_n) * BN, half = 32;  // the tile's first weight row; (EPI_QKV) how far its second 32 are from there
    if constexpr (EPI == EPI_QKV) {
        static_assert(WM == 1 && WN == 2 && WK == 4 && NB == 1 && !GUARD, "what the rotation knows");
        half = qkv.dh >> 1;
        const int per_head = half >> 5, tn = tile % tiles_n;
        n0 = tn / per_head * qkv.dh + tn % per_head * 32;
    }
    const int kbeg = EPI == EPI_BF16 ? 0 : blockIdx.y * kspan;                                        // a multiple of 256
    const int kn = EPI == EPI_BF16 ? K : (K - kbeg < kspan ? K - kbeg : kspan);                       // k of this workgroup
    const int G = K >> 5, steps = (kn + C::KS - 1) / C::KS;
    const int wrow = I4 ? K >> 1 : K;  // bytes of a weight row

    // ---- requests.  Buffer form of the DMA: the tile's first row in a resource descriptor, the lane's place in a 32-bit
    // offset that never changes, the step in the scalar offset.  A row past the matrix is requested beyond the
    // descriptor's range and arrives as zeros (its products are not stored; multipliers fed zeros draw less power).
    const int mrows = M - m0 < BM ? M - m0 : BM, nrows = EPI == EPI_QKV ? half + 32 : N - n0 < BN ? N - n0 : BN;
    auto wrow_at = [&](int r) { return EPI == EPI_QKV ? (r & 31) + (r >> 5) * half : r; };  // of the tile's column r, behind n0
    const __amdgpu_buffer_rsrc_t arsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(x) + (size_t)m0 * K, 0, mrows * K * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t brsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(wq) + (size_t)n0 * wrow, 0, nrows * wrow, 0x00020000);
    constexpr uint32_t kOut = 0x80000000u;
    const __amdgpu_buffer_rsrc_t srsrc = __builtin_amdgcn_make_buffer_rsrc(
        I4 ? const_cast<uint16_t *>(reinterpret_cast<const uint16_t *>(scv)) + (size_t)n0 * G : nullptr, 0, I4 ? nrows * G * 2 : 0, 0x00020000);
    uint32_t aoff[C::A_DMA], boff[C::BS_DMA];
    int apc[C::A_DMA], bpc[C::BS_DMA];
    constexpr int BPR = BB / 16;  // 16-byte pieces per weight row and step
    // WK = 4: a row's 64 to 256 bytes span a quarter to all of the banks, so its pieces are XOR-swizzled by the row as A's are
    auto bkey = [](int r) { return WK < 4 ? 0 : BPR == 4 ? (r >> 2) & 3 : BPR == 8 ? (r >> 1) & 7 : r & 15; };
#pragma unroll
    for (int q = 0; q < C::A_DMA; ++q) {  // 8 row segments of 128 B per instruction, [64 k][row][128 B]
        const int e = (q * C::NW + wave) * 8 + (lane >> 3), r = e % BM;
        apc[q] = e / BM * 128 + 16 * ((lane & 7) ^ ((r >> 1) & 7));
        aoff[q] = r < mrows ? (uint32_t)r * (uint32_t)(K * 2) + (uint32_t)apc[q] : kOut;
    }
#pragma unroll
    for (int q = 0; q < C::BS_DMA; ++q) {  // 64 / BPR weight rows, or the scales of 64, per instruction
        const int e = q * C::NW + wave, r = e * (64 / BPR) + lane / BPR, c = (e - C::BI) * 64 + lane, rw = wrow_at(r), cw = wrow_at(c);
        bpc[q] = 16 * ((lane % BPR) ^ bkey(r));
        if (SHORT || e < C::BI) boff[q] = rw < nrows ? (uint32_t)rw * (uint32_t)wrow + (uint32_t)bpc[q] : kOut;
        else boff[q] = e < C::BI + C::SI && cw < nrows ? (uint32_t)cw * (uint32_t)(G * 2) : kOut;
    }
    const uint16_t *srow[NB];  // GUARD: the scale rows of the lane's columns
    if constexpr (I4 && GUARD) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int n = n0 + (wn * NB + nb) * 32 + nl;
            srow[nb] = reinterpret_cast<const uint16_t *>(scv) + (size_t)(n < N ? n : N - 1) * G + (kbeg >> 5);
        }
    }

    auto dma = [&](const __amdgpu_buffer_rsrc_t &rsrc, uint32_t voff, int soff, uint8_t *dst) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)dst, 16, voff, soff, 0, 0);
    };
    // GUARD: a piece past the end of its row is not fetched (zeros); whole pieces: K % 32 == 0 (int4), K % 16 == 0 (int8).
    // `whole`: the step is not the last one, so there is none.
    auto issue_a = [&](int q, int step, uint8_t *stage, bool whole) {
        const int soff = kbeg * 2 + step * (2 * C::KS);
        dma(arsrc, GUARD && !whole && soff + apc[q] >= K * 2 ? kOut : aoff[q], soff, stage + (q * C::NW + wave) * 1024);
    };
    auto issue_b = [&](int q, int step, uint8_t *stage, bool whole) {
        const int boffs = (I4 ? kbeg >> 1 : kbeg) + step * BB, soffs = (kbeg >> 4) + step / C::SPB * 16;
        const int e = q * C::NW + wave;
        if (q >= C::BS_DMA) {  // GUARD, int4: scales
            const int nb = q - C::BS_DMA, g = KW == 64 ? 2 * (step * WK + wk) + kq : step * WK + wk;
            dma2_to_lds(srow[nb] + (g < G - (kbeg >> 5) ? g : 0), stage + C::A_STAGE + C::B_STAGE + (wave * NB + nb) * 256);
        } else if ((q + 1) * C::NW <= C::BI) {
            dma(brsrc, GUARD && !whole && boffs + bpc[q] >= wrow ? kOut : boff[q], boffs, stage + C::A_STAGE + e * 1024);
        } else {
            const bool isb = e < C::BI, none = C::DUMP && e >= C::BI + C::SI;
            const __amdgpu_buffer_rsrc_t rs = q * C::NW >= C::BI ? srsrc : isb ? brsrc : srsrc;
            dma(rs, GUARD && !whole && isb && boffs + bpc[q] >= wrow ? kOut : boff[q], isb ? boffs : soffs,
                none ? lds + C::DUMP_OFF : stage + C::A_STAGE + e * 1024);
        }
    };
    // The requests of a step: the weights and scales of step j+1 (the last step has none: its own once more, read by nobody), the
    // activations of step j
    auto request = [&](int r, int j, uint8_t *stage_b, uint8_t *stage_a, bool whole) {
        if (r < C::REQ - C::A_DMA) issue_b(r, whole || j + 1 < steps ? j + 1 : j, stage_b, whole);
        else issue_a(r - (C::REQ - C::A_DMA), j, stage_a, whole);
    };

    // ---- fragment read offsets: row nl of a 32-row block, the wave's pieces SL kq + t (EXACT: 2 t + kq, so that two slices are one
    // scale group); the lane's packed weights
    static_assert(!EXACT || (I4 && NB == 1 && (!GUARD || KW == 64)), "exact weights: int4, one column block");
    uint32_t foff[SL];
#pragma unroll
    for (int t = 0; t < SL; ++t)
        foff[t] = (uint32_t)(wk * KW / 64 * BM * 128 + (wm * MB * 32 + nl) * 128 +
                             (((wk * KW % 64 / 8 + (EXACT ? 2 * t + kq : SL * kq + t)) ^ ((nl >> 1) & 7)) << 4));
    constexpr int LB = I4 ? KW / 4 : KW / 2, BQ = EXACT ? KW / 32 : LB > 16 ? LB / 16 : 1;  // bytes of a lane's k, 16-byte pieces of them
    uint32_t woff[BQ];
#pragma unroll
    for (int e = 0; e < BQ; ++e) {  // (a block of 32 rows further on has the same key)
        const int b = (2 * wk + (EXACT ? 0 : kq)) * LB + 16 * e, r = wn * 32 * NB + nl;
        woff[e] = (uint32_t)(C::A_STAGE + r * BB + 16 * (b / 16 ^ bkey(r)) + b % 16);
    }

    const uint32_t c_mlo = vgpr_const(0x000F000Fu), c_mhi = vgpr_const(0x00F000F0u), c_magic = vgpr_const(0x64006400u);

    f32x16 acc[MB][NB];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.f;

    // Requests are spread over the MFMAs of a step, from the barrier on.  (A compute unit takes one in
    // 16 cycles; forty of them behind a barrier keep every wave from its next MFMA for as long as a step should take.)
    constexpr int NE = MB * NB, BAR = SL - AHEAD;          // MFMAs of a slice; the slice in front of which the barrier stands
    constexpr int GR = KW / 32, Q = GR * MB, LOOK = 2;     // EXACT: scale groups of a step, pairs of MFMAs, pairs from the barrier on
    static_assert(!EXACT || (Q >= LOOK && Q % 2 == 0), "the pairs behind the barrier are of the same step; two sums in turn");
    constexpr bool UNROLL = !EXACT || MB > 2;
    constexpr int NP = EXACT ? Q : SL * NE, AFTER = EXACT ? LOOK : AHEAD * NE;  // positions of a step, those behind its barrier
    auto first = [](int p) { return (p * C::REQ + NP - 1) / NP; };  // the first request at position p or later

    using T = std::true_type;
    using F = std::false_type;
    // ---- prologue
    if constexpr (!SHORT) {
#pragma unroll
        for (int r = 0; r < C::REQ - C::A_DMA; ++r) issue_b(r, 0, lds, false);
#pragma unroll
        for (int j = 0; j < ST - 1; ++j)
            if (j < steps)
#pragma unroll
                for (int r = 0; r < C::REQ; ++r) request(r, j, lds + (j + 1) * C::STAGE, lds + j * C::STAGE, false);
        if (steps >= ST - 1) wait_vmcnt<(ST - 2) * C::REQ>();  // the activations of step 0, the weights of steps 0 and 1
        else wait_vmcnt<0>();
        wg_barrier();
    }
    auto run = [&](auto &step) {
        // (stages as constants in the loop: their addresses cost nothing there; not worth the code for few rows, whose workgroups
        // take a few steps each)
        int i = 0;
        for (; UNROLL && i + 2 * ST + 1 < steps; i += ST) {
#pragma unroll
            for (int u = 0; u < ST; ++u) step(i + u, u, std::integral_constant<int, ST - 2>{}, T{}, T{}, T{});
        }
        int slot = 0;
        auto next = [&]() {
            ++i;
            slot = slot + 1 == ST ? 0 : slot + 1;
        };
        for (; i + ST < steps; next()) step(i, slot, std::integral_constant<int, ST - 2>{}, T{}, T{}, F{});
        if (ST <= steps) step(i, slot, std::integral_constant<int, ST - 2>{}, T{}, F{}, F{}), next();
        if (ST >= 6 && i + 4 < steps) step(i, slot, std::integral_constant<int, 3>{}, F{}, F{}, F{}), next();
        if (ST >= 5 && i + 3 < steps) step(i, slot, std::integral_constant<int, 2>{}, F{}, F{}, F{}), next();
        if (ST >= 4 && i + 2 < steps) step(i, slot, std::integral_constant<int, 1>{}, F{}, F{}, F{}), next();
        if (i + 1 < steps) step(i, slot, std::integral_constant<int, 0>{}, F{}, F{}, F{}), next();
        step(i, slot, std::integral_constant<int, -1>{}, F{}, F{}, F{});
    };

    if constexpr (EXACT) {
    // Exact weights: integers as operands, two MFMAs from zero on per scale group and row block, and one fp32 FMA per
    // value that applies the scale.  A pair of MFMAs runs beside the FMAs of the pair before it.
    constexpr int RING = Q >= 4 ? 4 : 2;
    // The row block beside whose MFMAs the next group's words are taken over (a step of one group: when they have arrived) and the one, not
    // before it, beside which the first half of their operands is made
    constexpr int PREP = GR > 1 || MB <= 2 ? 0 : MB > 4 ? 2 : 1, HALF = MB <= 2 ? 0 : MB > 4 ? MB / 2 - 1 : GR > 1 ? 1 : 2;
    static_assert(MB <= 4 || MB == 8, "the row blocks these are right for");
    uint32_t wv[GR][2], wnx[GR][2];  // the lane's packed words of a step [group][slice], of the next one
    uint32_t sraw[GR];               // its scales
    float sc2[GR], s_last = 0.f;     // ... as floats, that of the group whose sums are next
    constexpr float undo = 512.f;    // what the operands leave out, or (whole steps) they and the activations
    static_assert(16.f / kExactX == undo, "operands of (u - 8) / 2^4 for activations that carry the factor");
    auto fetch = [&](int step, const uint8_t *stage) {
#pragma unroll
        for (int g = 0; g < GR; ++g)
#pragma unroll
            for (int e = 0; e < 2; ++e) wnx[g][e] = *reinterpret_cast<const uint32_t *>(stage + woff[g] + e * 8 + kq * 4);
        const uint8_t *const sp = stage + C::A_STAGE + C::B_STAGE;
#pragma unroll
        for (int g = 0; g < GR; ++g)
            sraw[g] = *reinterpret_cast<const uint16_t *>(GUARD ? sp + wave * 256 + (nl + 32 * g) * 4
                                                                : sp + (wn * 32 + nl) * 16 + ((step * WK + wk) * GR + g & 7) * 2);
    };
    auto prep = [&](int step) {
#pragma unroll
        for (int g = 0; g < GR; ++g) {
            wv[g][0] = wnx[g][0];
            wv[g][1] = wnx[g][1];
            sc2[g] = (GUARD && kbeg + step * C::KS + wk * KW + 32 * g >= K) ? 0.f : undo * f16_bits_to_f32((uint16_t)sraw[g]);
        }
    };
    bf16x8 bo[2], bnx[2];  // operands of the present group, of the next one
    auto operand = [](uint32_t w) { return GUARD ? signed8_i4(w) : signed8_i4_16th(w); };
    bf16x8 af[RING][2];
    auto frag = [&](int q, const uint8_t *stage) {  // of pair q: group q / MB, row block q % MB
#pragma unroll
        for (int e = 0; e < 2; ++e) af[q % RING][e] = *reinterpret_cast<const bf16x8 *>(stage + (q % MB) * 4096 + foff[2 * (q / MB) + e]);
    };
    f32x16 tmp[2];
#pragma unroll
    for (int v = 0; v < 16; ++v) tmp[1][v] = 0.f;

    fetch(0, lds);
#pragma unroll
    for (int q = 0; q < LOOK; ++q) frag(q, lds);
    if (ST <= steps) {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        wg_barrier();                        // step 0's weights have been read
#pragma unroll
        for (int r = 0; r < first(AFTER); ++r) request(r, ST - 1, lds, lds + (ST - 1) * C::STAGE, false);
    }
    prep(0);
    bo[0] = operand(wv[0][0]);
    bo[1] = operand(wv[0][1]);
    auto step = [&](int i, int slot, auto pending_c, auto before_c, auto more_c, auto whole_c) {
        constexpr bool whole = decltype(whole_c)::value, before = decltype(before_c)::value, more = decltype(more_c)::value;  // as below
        constexpr int pending = decltype(pending_c)::value;
        uint8_t *const cur = lds + slot * C::STAGE, *const nxt = lds + (slot + 1 == ST ? 0 : slot + 1) * C::STAGE;
        uint8_t *const prv = lds + (slot == 0 ? ST - 1 : slot - 1) * C::STAGE;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int g = q / MB, mb = q % MB;
            if (q == 0 && pending >= 0) fetch(i + 1, nxt);  // (in front of the barrier also where that is the first thing: MB = 1)
            if (q == Q - LOOK && pending >= 0) {
                wait_vmcnt<(pending > 0 ? pending * C::REQ : 0)>();
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
                wg_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
            const int p = q < Q - LOOK ? q + LOOK : q - (Q - LOOK);
#pragma unroll
            for (int r = first(p); r < first(p + 1); ++r) {
                if (before && q < Q - LOOK) request(r, i + ST - 1, cur, prv, whole);
                if (more && q >= Q - LOOK) request(r, i + ST, nxt, cur, whole);
            }
            f32x16 zero;
#pragma unroll
            for (int v = 0; v < 16; ++v) zero[v] = 0.f;
            tmp[q & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[q % RING][0], bo[0], zero, 0, 0, 0);
            tmp[q & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[q % RING][1], bo[1], tmp[q & 1], 0, 0, 0);
            if (q < Q - LOOK) frag(q + LOOK, cur);
            else if (pending >= 0) frag(q - (Q - LOOK), nxt);
            f32x16 &a = acc[(mb + MB - 1) % MB][0];
#pragma unroll
            for (int v = 0; v < 16; ++v) a[v] = __builtin_fmaf(tmp[(q + 1) & 1][v], s_last, a[v]);
            if (mb == 0) s_last = sc2[g];
            // the next group's operands, a share beside each pair
            if (g + 1 < GR || pending >= 0) {
                if (g + 1 == GR && mb == PREP) prep(i + 1);
                if (mb == HALF) bnx[0] = operand(wv[(g + 1) % GR][0]);
                if (mb == MB - 1) bnx[1] = operand(wv[(g + 1) % GR][1]);
            }
            if (mb == MB - 1) {
                bo[0] = bnx[0];
                bo[1] = bnx[1];
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 5, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 60, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    run(step);
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[MB - 1][0][v] = __builtin_fmaf(tmp[(Q - 1) & 1][v], s_last, acc[MB - 1][0][v]);
    } else {
    uint8_t *const slds = lds + C::S_OFF + 2 * wave * C::S_BUF;  // SHORT
    u32x4 bq[NB][BQ], bn[NB][BQ];  // the lane's packed weights of a step (int4 and 32 k: half of one), of the next one
    uint16_t sraw[NB];
    float cs[NB][4];
    auto fetch = [&](int step, const uint8_t *stage) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
            for (int e = 0; e < BQ; ++e) {
                const uint8_t *const p = stage + woff[e] + nb * 32 * BB;
                if constexpr (LB == 8) {
                    const u32x2 v = *reinterpret_cast<const u32x2 *>(p);
                    bn[nb][e] = u32x4{v.x, v.y, 0u, 0u};
                } else {
                    bn[nb][e] = *reinterpret_cast<const u32x4 *>(p);
                }
            }
            const uint8_t *const sp = stage + C::A_STAGE + C::B_STAGE;
            if constexpr (I4 && SHORT)
                sraw[nb] = *reinterpret_cast<const uint16_t *>(
                    slds + (GUARD ? (step & 1) * C::S_BUF + lane * 4 : (step / C::SPB & 1) * C::S_BUF + nl * 16 + (((step * WK + wk) & 3) * 2 + kq) * 2));
            else if constexpr (I4 && GUARD) sraw[nb] = *reinterpret_cast<const uint16_t *>(sp + (wave * NB + nb) * 256 + lane * 4);
            else if constexpr (I4)
                sraw[nb] = *reinterpret_cast<const uint16_t *>(sp + ((wn * NB + nb) * 32 + nl) * 16 +
                                                               (KW == 64 ? ((step * WK + wk) & 3) * 2 + kq : (step * WK + wk) & 7) * 2);
        }
    };
    auto prep = [&](int step) {  // the fetched ones' turn; scale -> FMA constants; int4 weights past the row's end read as u = 0 and get the scale 0
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int e = 0; e < BQ; ++e) bq[nb][e] = bn[nb][e];
        if constexpr (I4) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const float s = (GUARD && kbeg + step * C::KS + wk * KW + kq * (KW / 2) >= K) ? 0.f : f16_bits_to_f32(sraw[nb]);
                cs[nb][0] = s;
                cs[nb][1] = s * 0.0625f;
                cs[nb][2] = -1032.f * s;
                cs[nb][3] = -72.f * s;
            }
        }
    };
    bf16x8 bf[2][NB];
    auto deq = [&](int t) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if constexpr (CHADQ_GEMM_ABLATE == 1) {
                const u32x4 q = bq[nb][(I4 ? 0 : t >> 1) % BQ], raw = {q.x + (uint32_t)t, q.y, q.z, q.w};
                __builtin_memcpy(&bf[t & 1][nb], &raw, 16);
            } else if constexpr (I4) bf[t & 1][nb] = dequant8_i4(bq[nb][0][t], cs[nb][0], cs[nb][1], cs[nb][2], cs[nb][3], c_mlo, c_mhi, c_magic);
            else bf[t & 1][nb] = dequant8_i8(bq[nb][t >> 1][2 * (t & 1)], bq[nb][t >> 1][2 * (t & 1) + 1]);
        }
    };
    bf16x8 af[2 * AHEAD][MB];
    auto frag = [&](int t, int mb, const uint8_t *stage) {
        af[t % (2 * AHEAD)][mb] = *reinterpret_cast<const bf16x8 *>(stage + mb * 4096 + foff[t]);
    };

    auto frags = [&](int t, const uint8_t *stage) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) frag(t, mb, stage);
    };
    auto begin = [&]() {
        fetch(0, lds);
#pragma unroll
        for (int t = 0; t < AHEAD; ++t) frags(t, lds);
        if (!SHORT && ST <= steps) {
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            wg_barrier();                        // step 0's weights have been read
#pragma unroll
            for (int r = 0; r < first(AFTER); ++r) request(r, ST - 1, lds, lds + (ST - 1) * C::STAGE, false);
        }
        prep(0);
        deq(0);
    };

    // Step i works on stage i % ST and reads the packed weights of step i+1 at its beginning.  In front of its last slices, whose
    // fragments are in registers, a wave waits until its part of the activations of step i+1 and of the weights of step i+2 is
    // in LDS; the barrier says so for all of them, and that the activations of stage i and the weights of stage i+1 have been
    // read: step i+ST's and step i+ST+1's are requested into their place, from here to the next barrier.
    auto mfma = [&](int t, int e) {
        const int mb = e / NB, nb = e % NB;
        acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[t % (2 * AHEAD)][mb], bf[t & 1][nb], acc[mb][nb], 0, 0, 0);
    };
    // The order inside a slice: LDS reads with the first MFMAs, memory requests and the dequantisation spread over all of
    // them (mask 8: MFMA, 2: vector ALU, 0x100: LDS read, 0x20: vector memory).
    constexpr int DQ = NB * (I4 ? 17 : 12);
    if constexpr (SHORT) {
        // Few steps: everything of a step is requested together, two steps ahead, half of the activations a slice later, and the packed
        // weights are read with the step's first fragments.  Half the code and no request in front of the first MFMA that
        // it does not wait for: what a product of a few steps takes longest for is its way to the first MFMA and the code that it
        // runs through once.
        const uint16_t *const srow1 = reinterpret_cast<const uint16_t *>(scv) + (size_t)(n0 + wn * 32 + nl < N ? n0 + wn * 32 + nl : N - 1) * G;
        auto issue_s = [&](int blk) {  // blk: 256-k block, or (GUARD) step
            if constexpr (I4 && GUARD) {
                const int g = 2 * (blk * WK + wk) + kq;
                dma2_to_lds(srow1 + (g < G ? g : 0), slds + (blk & 1) * C::S_BUF);
            } else if constexpr (I4) {
                dma16_to_lds(srow1 + blk * 8, slds + (blk & 1) * C::S_BUF);
            }
        };
        auto issue = [&](int step, uint8_t *stage, bool b, int q0, int q1) {
#pragma unroll
            for (int q = 0; q < C::BS_DMA; ++q)
                if (b) issue_b(q, step, stage, false);
#pragma unroll
            for (int q = 0; q < C::A_DMA; ++q)
                if (q >= q0 && q < q1) issue_a(q, step, stage, false);
        };
        constexpr int STEP = C::A_DMA + C::BS_DMA;  // requests of a step, its scales aside
        uint8_t *cur = lds, *nxt = lds + C::STAGE, *far = lds + 2 * C::STAGE;
        issue_s(0);
        if (GUARD || C::SPB == 1 ? steps > 1 : C::SPB == 2 && steps > 2) issue_s(1);
        issue(0, cur, true, 0, C::A_DMA);
        if (steps > 1) {
            issue(1, nxt, true, 0, C::A_DMA);
            wait_vmcnt<STEP>();  // everything of step 0
        } else {
            wait_vmcnt<0>();
        }
        wg_barrier();
        begin();
        auto order = [&]() {
#pragma unroll
            for (int e = 0; e < MB; ++e) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                if (e % 2 == 1) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, (DQ + MB - 1) / MB, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        // Step i works on stage `cur` = i % 3 and requests step i+2 into `far`, which held step i-1: everybody has left that stage before
        // the barrier of step i-1.  In front of the barrier a wave waits until no more than what it has requested during this step is
        // outstanding: its part of stage i+1 and of the scales is then in LDS.
        auto step = [&](int i, auto more1_c, auto more2_c) {
            constexpr bool more1 = decltype(more1_c)::value, more2 = decltype(more2_c)::value;  // steps i+1, i+2 exist
            constexpr int H = (STEP + 1) / 2 - C::BS_DMA < 0 ? 0 : (STEP + 1) / 2 - C::BS_DMA;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t == BAR && more1) {
                    if (more2) wait_vmcnt<STEP>();
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
                if (t < BAR) frags(t + AHEAD, cur);
                if (t == 0 && more2) issue(i + 2, far, true, 0, H);
                if (t == 1 && more2) issue(i + 2, far, false, H, C::A_DMA);
#pragma unroll
                for (int e = 0; e < MB; ++e) mfma(t, e);
                if (t < 3) deq(t + 1);
                if (t == BAR && more1) fetch(i + 1, nxt);
                if (t >= BAR && more1) frags(t - BAR, nxt);
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
        int i = 0;
        for (; i + 2 < steps; ++i) step(i, T{}, T{});
        if (steps > 1) step(i++, T{}, F{});
        step(i, F{}, F{});
    } else {
    begin();
    auto order = [&]() {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, (DQ + NE - 1) / NE, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto step = [&](int i, int slot, auto pending_c, auto before_c, auto more_c, auto whole_c) {
        constexpr bool whole = decltype(whole_c)::value;     // everything it requests lies before the last step
        constexpr int pending = decltype(pending_c)::value;  // further steps whose requests may be outstanding at the barrier; -1: the last step
        constexpr bool before = decltype(before_c)::value;   // step i+ST-1 exists: the rest of its requests
        constexpr bool more = decltype(more_c)::value;       // step i+ST exists
        uint8_t *const cur = lds + slot * C::STAGE, *const nxt = lds + (slot + 1 == ST ? 0 : slot + 1) * C::STAGE;
        uint8_t *const prv = lds + (slot == 0 ? ST - 1 : slot - 1) * C::STAGE;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < SL; ++t) {
            if (t == BAR && pending >= 0) {
                wait_vmcnt<(pending > 0 ? pending * C::REQ : 0)>();
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
                wg_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                if (e < MB && t < BAR) frag(t + AHEAD, e, cur);
                if (e < MB && t >= BAR && pending >= 0) frag(t - BAR, e, nxt);
                if (t == 0 && e == 0 && pending >= 0) fetch(i + 1, nxt);
                const int p = (t < BAR ? t + AHEAD : t - BAR) * NE + e;
#pragma unroll
                for (int r = first(p); r < first(p + 1); ++r) {
                    if (before && t < BAR) request(r, i + ST - 1, cur, prv, whole);
                    if (more && t >= BAR) request(r, i + ST, nxt, cur, whole);
                }
                mfma(t, e);
            }
            if (t < SL - 1) deq(t + 1);
            if (t == SL - 1 && pending >= 0) {
                prep(i + 1);
                deq(0);
            }
            order();
        }
    };
    run(step);
    }
    }

    // ---- epilogue.  The lane holds, for every mb and nb, column nl of rows 8*(v/4) + 4*kq + v%4 of a 32 x 32 block.
    wg_barrier();  // every wave is done with the stages, which everything below reuses
    // A wave finishes 1/WK of its values, MB * 16 of them numbered (row block, v).  WK = 2: the two waves that hold the k halves of
    // one result trade halves of it through LDS.  WK = 4: every wave leaves all of them and adds its quarter in the order of the k.
    constexpr int UV = MB * 16 / WK;
    auto row_of = [&](int v) {
        auto at = [](int f) { return (f >> 4) * 32 + 8 * ((f & 15) >> 2) + (f & 3); };
        // (where no carry goes between the two parts of the number, the second part of the row is a constant)
        return wm * MB * 32 + 4 * kq + (16 % UV == 0 || UV % 16 == 0 ? at(wk * UV) + at(v) : at(wk * UV + v));
    };
    if constexpr (EPI == EPI_QKV) {
        // as WK = 4 below, but a wave adds up both halves of its pairs of columns: each of the two waves of a pair then writes one of them
        const int head = n0 / qkv.dh, j = n0 % qkv.dh + nl;
        float cs[UV], sn[UV];
#pragma unroll
        for (int v = 0; v < UV; ++v) {
            const int m = m0 + row_of(v);
            const float *const t = qkv.table + ((size_t)(qkv.pos + (m < M ? m : M - 1)) * half + j) * 2;
            cs[v] = t[0];
            sn[v] = t[1];
        }
        float *const red = reinterpret_cast<float *>(lds) + lane * 4;
#pragma unroll
        for (int q = 0; q < MB * 4; ++q) {
            auto val = [&](int f) { return acc[f >> 4][0][f & 15]; };
            *reinterpret_cast<f32x4 *>(red + (wave * MB * 4 + q) * 256) = f32x4{val(4 * q), val(4 * q + 1), val(4 * q + 2), val(4 * q + 3)};
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < UV / 4; ++q) {
            f32x4 o[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int w = 0; w < WK; ++w) o[h] += *reinterpret_cast<const f32x4 *>(red + ((w * WN + h) * MB * 4 + wk * (UV / 4) + q) * 256);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int v = 4 * q + e, m = m0 + row_of(v);
                if (m >= M) continue;
                const float a = o[0][e], b = o[1][e];
                const float r = head > qkv.hq ? (wn ? b : a) : wn ? b * cs[v] + a * sn[v] : a * cs[v] - b * sn[v];
                const int at = j + wn * half;
                if (head < qkv.hq) qkv.q[((size_t)m * qkv.hq + head) * qkv.dh + at] = r;
                else (head == qkv.hq ? qkv.kc : qkv.vc)[(size_t)(qkv.pos + m) * qkv.dh + at] = (uint16_t)f32_to_bf16_bits(r);
            }
        }
        return;
    }
    float res[NB][UV];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        auto val = [&](int f) { return acc[f >> 4][nb][f & 15]; };
        if constexpr (WK == 2) {
            float *const red = reinterpret_cast<float *>(lds) + (wm * WN + wn) * (MB * 1024) + lane * 4;
#pragma unroll
            for (int q = 0; q < UV / 4; ++q) {
                f32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = wk ? val(4 * q + e) : val(UV + 4 * q + e);
                *reinterpret_cast<f32x4 *>(red + (wk * (UV / 4) + q) * 256) = o;
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < UV / 4; ++q) {
                const f32x4 o = *reinterpret_cast<const f32x4 *>(red + ((1 - wk) * (UV / 4) + q) * 256);
#pragma unroll
                for (int e = 0; e < 4; ++e) res[nb][4 * q + e] = (wk ? val(UV + 4 * q + e) : val(4 * q + e)) + o[e];
            }
            __syncthreads();
        } else if constexpr (WK == 4) {
            float *const red = reinterpret_cast<float *>(lds) + lane * 4;
#pragma unroll
            for (int q = 0; q < MB * 4; ++q)
                *reinterpret_cast<f32x4 *>(red + (wave * MB * 4 + q) * 256) = f32x4{val(4 * q), val(4 * q + 1), val(4 * q + 2), val(4 * q + 3)};
            __syncthreads();
#pragma unroll
            for (int q = 0; q < UV / 4; ++q) {
                f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int w = 0; w < WK; ++w)
                    o += *reinterpret_cast<const f32x4 *>(red + (((w * WM + wm) * WN + wn) * MB * 4 + wk * (UV / 4) + q) * 256);
#pragma unroll
                for (int e = 0; e < 4; ++e) res[nb][4 * q + e] = o[e];
            }
            __syncthreads();
        } else {
#pragma unroll
            for (int v = 0; v < UV; ++v) res[nb][v] = val(v);
        }
    }
    if constexpr (EPI == EPI_F32) {  // 128 contiguous bytes per row straight from the registers
        float *const y = reinterpret_cast<float *>(yv) + (size_t)blockIdx.y * M * N;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int n = n0 + (wn * NB + nb) * 32 + nl;
#pragma unroll
            for (int v = 0; v < UV; ++v) {
                const int m = m0 + row_of(v);
                if (m < M && n < N) y[(size_t)m * N + n] = res[nb][v];
            }
        }
        return;
    }
    // bf16 results leave through a tile in LDS, as whole rows: neighbouring lanes first swap one value of each row pair
    // (one DPP move), so that a lane writes two adjacent columns of one row as a 32-bit word - or forms the gated value
    // of one feature of one row - and the tile is then read back 16 bytes per thread.
    constexpr bool GE = EPI == EPI_GEGLU;
    constexpr int EP = C::EP_PITCH;
    const bool odd = lane & 1;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int cb = (wn * NB + nb) * 32;  // the block's first column in the tile
        float colscale = 1.f;
        if constexpr (!I4) {
            const int n = n0 + cb + nl;
            colscale = reinterpret_cast<const float *>(scv)[n < N ? n : N - 1];
        }
#pragma unroll
        for (int v = 0; v < UV; v += 2) {
            float a0 = res[nb][v], a1 = res[nb][v + 1];  // rows r and r+1, column nl
            if constexpr (!I4) {
                a0 *= colscale;
                a1 *= colscale;
            }
            const float send = odd ? a0 : a1;
            const float recv = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(send), 0xB1, 0xF, 0xF, false));  // lane ^ 1
            const int row = row_of(v) + (odd ? 1 : 0);
            // even lane: row r, columns (nl, nl+1) = (own a0, neighbour's a0); odd lane: row r+1, columns (nl-1, nl)
            if constexpr (GE)
                *reinterpret_cast<uint16_t *>(lds + row * EP + (cb + nl) / 2 * 2) =
                    (uint16_t)pack_bf16_rne(gelu_tanh_dev(odd ? recv : a0) * (odd ? a1 : recv) * kExactX, 0.f);
            else
                *reinterpret_cast<uint32_t *>(lds + row * EP + (cb + (nl & ~1)) * 2) = odd ? pack_bf16_rne(recv, a1) : pack_bf16_rne(a0, recv);
        }
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

// K in n parts (blockIdx.y) of `span` k each, a multiple of 256, the last one possibly shorter.  Whoever chooses n chooses the span with it: parts
// that end before K would be a wrong sum, a part behind it a sum of nothing.
struct KParts {
    int n = 1, span = 0;
};

template <bool I4, int WM, int WN, int WK, int MB, int NB, int KW, int ST, bool GUARD, bool EXACT = false, int EPI = EPI_BF16, bool SHORT = false>
static int launch(const uint16_t *x, const uint8_t *wq, const void *sc, void *y, int M, int N, int K, KParts kp, hipStream_t st,
                  MoreOut<EPI> qkv = {}) {
    typedef Cfg<I4, WM, WN, WK, MB, NB, KW, ST, GUARD, SHORT> C;
    if (kp.n == 1) kp.span = K;
    else
        CHADQ_REQUIRE(EPI == EPI_F32 && kp.n > 1 && kp.span > 0 && kp.span % 256 == 0 && (int64_t)kp.n * kp.span >= K && (int64_t)(kp.n - 1) * kp.span < K,
                      CHADQ_ERR_SHAPE, "gemm: %d parts of %d k do not make up %d", kp.n, kp.span, K);
    static std::atomic<bool> attr_set{false};  // setting it twice from two threads is harmless
    if (!attr_set.load(std::memory_order_acquire)) {
        CHADQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_tile_q_kernel<I4, WM, WN, WK, MB, NB, KW, ST, GUARD, EXACT, EPI, SHORT>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS));
        attr_set.store(true, std::memory_order_release);
    }
    const int tiles = ((N + C::BN - 1) / C::BN) * ((M + C::BM - 1) / C::BM);
    hipLaunchKernelGGL((gemm_tile_q_kernel<I4, WM, WN, WK, MB, NB, KW, ST, GUARD, EXACT, EPI, SHORT>), dim3((tiles + 7) / 8 * 8, kp.n), dim3(C::T), C::LDS, st,
                       x, wq, sc, y, M, N, K, kp.span, qkv);
    return hip_check(hipGetLastError(), "gemm_tile_q launch");
}

}  // namespace tileq

// A tile's byte offsets are signed 32-bit in the descriptor: 256 rows of the wider matrix stay below 2 GiB.
bool gemm_tile_q_ok(int K) { return K < (1 << 22); }

// Which tile.  A tile takes c0 + c1 * K / 4096 us on a chip full of them and less on one that is not: a round of f * 256 tiles b +
// (1 - b) f of it; s is what a launch takes besides.  Longer launches run at a lower clock, which costs the tiles differently: `a` us of
// work take a (1 + q a / (a + 100)).  The constants are fitted to whole calls, every tile on 4500 random products (65 to 7000 rows, 64 to
// 33000 columns, 32 to 18000 k), for whole and for guarded steps (K no multiple of a step, or int4 scales that are not aligned), whose
// requests cost the tiles of two column blocks per wave more.  The tile picked is 0.2 % slower on average than the best of all, 7 % in
// one case of a hundred.  (With constants of products of 512 k and more only, the picks below that were up to 40 % off: 193 x 12160 x
// 128 int8 6.5 us on 128 x 128 tiles, 8.8 on 128 x 64.)  Up to 64 rows the smallest tiles win in any number of rounds (the others are
// padded to 96 rows and every round of theirs carries the same weights): 33 x 20000 x 2048 15.4 us (128 x 64: 23.7), 64 x 256000 x 2048
// 151 (299), 64 x 16384 x 16384 63 (87).
struct TileCost {
    GemmTile tile;
    int bm, bn, ks;  // ks: k of a step
    float s, c0, c1, b, q;
};
static const TileCost kCost[2][2][8] = {  // [int8, int4][whole steps, guarded]
    {{{TILE_64x64, 64, 64, 256, 1.89f, 2.51f, 10.61f, 0.67f, -0.03f}, {TILE_96x64, 96, 64, 128, 1.88f, 3.11f, 12.80f, 0.72f, 0.18f},
      {TILE_128x64, 128, 64, 128, 0.00f, 5.66f, 15.04f, 0.76f, 0.18f}, {TILE_96x128, 96, 128, 128, 0.00f, 8.21f, 21.96f, 0.51f, -0.02f},
      {TILE_128x128, 128, 128, 128, 0.00f, 7.28f, 28.37f, 0.62f, -0.06f}, {TILE_192x128, 192, 128, 64, 1.36f, 6.81f, 40.17f, 0.62f, 0.00f},
      {TILE_256x128, 256, 128, 64, 2.00f, 7.67f, 53.01f, 0.55f, -0.03f}, {TILE_256x256, 256, 256, 64, 1.77f, 9.47f, 105.38f, 0.53f, -0.11f}},
     {{TILE_64x64, 64, 64, 256, 2.05f, 2.18f, 11.35f, 0.67f, 0.24f}, {TILE_96x64, 96, 64, 128, 1.52f, 3.45f, 14.81f, 0.71f, 0.19f},
      {TILE_128x64, 128, 64, 128, 1.14f, 4.22f, 16.36f, 0.71f, 0.62f}, {TILE_96x128, 96, 128, 128, 0.00f, 7.63f, 24.52f, 0.61f, -0.04f},
      {TILE_128x128, 128, 128, 128, 0.36f, 6.35f, 31.52f, 0.65f, -0.08f}, {TILE_192x128, 192, 128, 64, 1.83f, 5.69f, 44.59f, 0.66f, -0.00f},
      {TILE_256x128, 256, 128, 64, 1.86f, 7.58f, 56.05f, 0.51f, -0.03f}, {TILE_256x256, 256, 256, 64, 1.56f, 9.07f, 119.73f, 0.48f, -0.18f}}},
    {{{TILE_64x64, 64, 64, 256, 1.93f, 2.66f, 10.60f, 0.70f, -0.03f}, {TILE_96x64, 96, 64, 128, 2.47f, 2.71f, 13.49f, 0.70f, 0.26f},
      {TILE_128x64, 128, 64, 128, 0.00f, 5.42f, 16.04f, 0.80f, 0.18f}, {TILE_96x128, 96, 128, 128, 0.00f, 7.28f, 22.22f, 0.66f, 0.06f},
      {TILE_128x128, 128, 128, 128, 2.36f, 3.88f, 30.34f, 0.54f, 0.02f}, {TILE_192x128, 192, 128, 64, 2.96f, 4.86f, 48.02f, 0.48f, 0.01f},
      {TILE_256x128, 256, 128, 64, 2.58f, 5.85f, 62.65f, 0.50f, -0.09f}, {TILE_256x256, 256, 256, 64, 2.21f, 8.13f, 111.38f, 0.50f, -0.07f}},
     {{TILE_64x64, 64, 64, 256, 1.84f, 2.38f, 11.89f, 0.74f, 0.11f}, {TILE_96x64, 96, 64, 128, 0.63f, 4.46f, 15.47f, 0.81f, 0.37f},
      {TILE_128x64, 128, 64, 128, 1.41f, 3.75f, 19.00f, 0.80f, 0.21f}, {TILE_96x128, 96, 128, 128, 0.00f, 6.78f, 27.90f, 0.73f, 0.06f},
      {TILE_128x128, 128, 128, 128, 1.92f, 3.88f, 31.22f, 0.65f, 0.07f}, {TILE_192x128, 192, 128, 64, 0.00f, 8.48f, 47.18f, 0.61f, 0.28f},
      {TILE_256x128, 256, 128, 64, 1.29f, 7.12f, 70.92f, 0.64f, -0.06f}, {TILE_256x256, 256, 256, 64, 2.70f, 7.41f, 114.01f, 0.48f, -0.05f}}},
};

// K up to which the loop for few steps is the faster one (it also is for the first steps of the others, hence no clear line: within 2 %
// of each other for a third of the value on both sides).  us, that loop / the other: 24 x 1024 x 1120 int4 5.2 / 5.8, 48 x 1024 x 512 4.7 / 4.9,
// 24 x 1024 x 512 int8 3.85 / 4.05, 247 x 13952 x 96 int8 6.7 / 7.8; 48 x 4096 x 8192 int4 21.7 / 19.0, 100 x 1024 x 4096 13.0 / 11.8.
static int short_k(GemmTile t, bool int4, bool guard) {
    switch (t) {
        case TILE_32x64: return int4 ? (guard ? 8192 : 3584) : guard ? 2560 : 3584;
        case TILE_64x64: return int4 && guard ? 4096 : 1792;
        case TILE_128x128: return int4 ? (guard ? 1536 : 768) : guard ? 1536 : 1792;
        case TILE_256x256: return int4 ? (guard ? 1280 : 512) : 0;
        default: return 0;
    }
}

// us of `tiles` workgroups of t, `wgs` of them counted for the fill of the last round (the same number where nothing is split), k each
static float tile_us(const TileCost &t, int64_t wgs, int k) {
    const int64_t rounds = (wgs + 255) >> 8;
    const float fill = (float)(wgs - (rounds - 1) * 256) / 256.f, kk = (float)((k + t.ks - 1) & -t.ks);  // (a step is a power of two)
    const float a = t.s + ((float)(rounds - 1) + t.b + (1.f - t.b) * fill) * (t.c0 + t.c1 * kk / 4096.f);
    return a * (1.f + t.q * a / (a + 100.f));
}

static int64_t tiles_of(const TileCost &t, int M, int N) { return (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn); }

GemmTile gemm_tile_pick(int M, int N, int K, bool int4, bool guard) {
    GemmTile best = M <= 32 ? TILE_32x64 : TILE_64x64;
    if (M > 64) {
        float best_cost = 0.f;
        for (const TileCost &t : kCost[int4][guard]) {
            const float cost = tile_us(t, tiles_of(t, M, N), K);
            if (best_cost == 0.f || cost < best_cost) {
                best = t.tile;
                best_cost = cost;
            }
        }
    }
    if (K > short_k(best, int4, guard)) return best;
    switch (best) {
        case TILE_32x64: return SHORT_32x64;
        case TILE_64x64: return SHORT_64x64;
        case TILE_128x128: return SHORT_128x128;
        case TILE_256x256: return SHORT_256x256;
        default: return best;
    }
}

template <bool I4, bool GUARD>
static int launch_tile(const uint16_t *x, const uint8_t *w, const void *sc, uint16_t *y, int M, int N, int K, GemmTile tile, hipStream_t st) {
    switch (tile) {
        case TILE_32x64: return tileq::launch<I4, 1, 2, 4, 1, 1, 64, 3, GUARD>(x, w, sc, y, M, N, K, {}, st);
        case TILE_64x64: return tileq::launch<I4, 1, 2, 4, 2, 1, 64, 3, GUARD>(x, w, sc, y, M, N, K, {}, st);
        case TILE_96x64: return tileq::launch<I4, 1, 2, 4, 3, 1, 32, GUARD ? 3 : 4, GUARD>(x, w, sc, y, M, N, K, {}, st);
        case TILE_128x64: return tileq::launch<I4, 1, 2, 4, 4, 1, 32, GUARD ? 3 : 4, GUARD>(x, w, sc, y, M, N, K, {}, st);
        case TILE_96x128: return tileq::launch<I4, 1, 2, 4, 3, 2, 32, 3, GUARD>(x, w, sc, y, M, N, K, {}, st);
        case TILE_128x128:  // (the other form: int4 36.7 us against 36.3 at 1024 x 4096 x 4096, int8 113 against 107 at 1000 x 4096 x 14336)
            if constexpr (I4) return tileq::launch<I4, 1, 4, 2, 4, 1, 64, 3, GUARD>(x, w, sc, y, M, N, K, {}, st);
            else return tileq::launch<I4, 1, 2, 4, 4, 2, 32, 3, GUARD>(x, w, sc, y, M, N, K, {}, st);
        case TILE_192x128: return tileq::launch<I4, 2, 2, 2, 3, 2, 32, 3, GUARD>(x, w, sc, y, M, N, K, {}, st);
        case TILE_256x128: return tileq::launch<I4, 2, 2, 2, 4, 2, 32, 3, GUARD>(x, w, sc, y, M, N, K, {}, st);
        case TILE_256x256: return tileq::launch<I4, 1, 8, 1, 8, 1, 64, 3, GUARD>(x, w, sc, y, M, N, K, {}, st);
        case SHORT_32x64: return tileq::launch<I4, 1, 2, 4, 1, 1, 64, 3, GUARD, false, tileq::EPI_BF16, true>(x, w, sc, y, M, N, K, {}, st);
        case SHORT_64x64: return tileq::launch<I4, 1, 2, 4, 2, 1, 64, 3, GUARD, false, tileq::EPI_BF16, true>(x, w, sc, y, M, N, K, {}, st);
        case SHORT_128x128: return tileq::launch<I4, 1, 4, 2, 4, 1, 64, 3, GUARD, false, tileq::EPI_BF16, true>(x, w, sc, y, M, N, K, {}, st);
        case SHORT_256x256:
            if constexpr (I4) return tileq::launch<I4, 1, 8, 1, 8, 1, 64, 3, GUARD, false, tileq::EPI_BF16, true>(x, w, sc, y, M, N, K, {}, st);
            break;
    }
    return fail(CHADQ_ERR_SHAPE, "gemm: no tile %d", (int)tile);
}

int gemm_tile_i4g32_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, uint16_t *y, int M, int N, int K, GemmTile tile,
                           hipStream_t st) {
    const bool guard = K % 256 != 0 || !aligned16(sc);  // 16 bytes of scales at a time want aligned rows of them
    return guard ? launch_tile<true, true>(x, wp, sc, y, M, N, K, tile, st) : launch_tile<true, false>(x, wp, sc, y, M, N, K, tile, st);
}

int gemm_tile_i8row_launch(const uint16_t *x, const int8_t *w8, const float *sc, uint16_t *y, int M, int N, int K, GemmTile tile, hipStream_t st) {
    const uint8_t *w = reinterpret_cast<const uint8_t *>(w8);
    const bool k256 = tile == TILE_32x64 || tile == TILE_64x64 || tile == SHORT_32x64 || tile == SHORT_64x64;
    const bool k64 = tile == TILE_256x256 || tile == TILE_192x128 || tile == TILE_256x128;
    const int step = k256 ? 256 : k64 ? 64 : 128;  // k of a step
    return K % step ? launch_tile<false, true>(x, w, sc, y, M, N, K, tile, st) : launch_tile<false, false>(x, w, sc, y, M, N, K, tile, st);
}

// ---- few tiles and a long K: the product in parts of whole 256-k blocks, one fp32 matrix each, added by a second launch.  A workgroup's walk
// through K is what such a product takes: 48 x 4096 x 14336 is 64 workgroups of 56 steps, 29 us.  us, in one part / in parts, the launch that adds
// them included: int4 81 x 1280 x 14080 29.5 / 14.9 (six), 62 x 1536 x 11264 23.6 / 12.7 (eight), 26 x 5542 x 11776 24.6 / 16.6 (two), 46 x 6528 x 4928
// 14.6 / 13.5 (two), 48 x 4096 x 14336 29.0 / 17.9 (four), 219 x 1440 x 10432 28.8 / 20.7 (five); int8 250 x 640 x 9760 25.5 / 13.6 (six), 152 x 1280 x
// 14336 30.1 / 17.9 (four).  A second launch and its scratch cost a call 1.5 us that its kernels' times do not show, and the constants of gemm_tile_pick,
// fitted to fuller grids, give int8 products of few tiles a us too much in one part: both count, so that calls of 7 to 9 us stay in one (calls of
// qlinear in a row, int8: 17 x 512 x 4096 7.9 / 9.0, 65 x 512 x 3584 8.8 / 9.5; int4 49 x 960 x 2816 8.8 / 9.2).  Of 288 random calls in parts the mean
// takes 0.71 of the time in one (waited for one by one: 0.83), the worst 1.04.
static const TileCost kCost32 = {TILE_32x64, 32, 64, 256, 1.9f, 2.2f, 7.6f, 0.75f, 0.f};

int gemm_split_parts(int M, int N, int K, bool int4, GemmTile *tile, int *span) {
    // us of the second launch and its scratch, as far as they are not hidden, less what the model finds too long in one part; of a MB of parts
    const float kSum = int4 ? 4.f : 5.f, kMB = .3f;
    constexpr int kMost = 8;
    *span = K;
    // (below 2304 k the model never finds enough.  Beyond 200 tiles parts fill no idle compute units: of twelve products of 208 to 256 tiles, 4096 to 14336
    // k, two parts take 0.97 to 1.6 of the time in one, 48 x 14336 x 4096 20.4 us against 13.3, 256 x 3584 x 14336 39.6 against 38.5)
    if (M < 17 || K < 2304 || K >= (1 << 22) || (int64_t)((M + 63) / 64) * ((N + 63) / 64) > 200) return 1;
    float whole = 0.f, best = 0.f;
    int parts = 1;
    auto split = [&](const TileCost &t) {
        const int64_t tiles = tiles_of(t, M, N);
        const int blocks = (K + 255) / 256;
        for (int s = 2; s <= kMost && s <= blocks; ++s) {
            const int per = (blocks + s - 1) / s;
            if ((blocks + per - 1) / per != s) continue;
            // (tiles go to the XCDs in turn, each in all its parts)
            const float us = tile_us(t, (tiles + 7) / 8 * 8 * s, per * 256) + kSum + kMB * 4e-6f * (float)M * (float)N * (float)s;
            if (best == 0.f || us < best) {
                best = us;
                parts = s;
                *span = per * 256;
                *tile = t.tile;
            }
        }
    };
    if (M <= 32) {
        whole = tile_us(kCost32, tiles_of(kCost32, M, N), K);
        split(kCost32);
    } else {
        for (const TileCost &t : kCost[int4][K % 256 != 0]) {
            if (M <= 64 && t.tile != TILE_64x64) continue;
            const float us = tile_us(t, tiles_of(t, M, N), K);
            if (whole == 0.f || us < whole) whole = us;
            if (t.tile == TILE_64x64 || t.tile == TILE_128x64) split(t);
        }
    }
    if (best != 0.f && best < .98f * whole) return parts;
    *span = K;
    return 1;
}

// y[m,n] = bf16(sum of the parts, in order, times the row scale of int8 weights); V columns per thread
template <int V>
__global__ __launch_bounds__(256) void gemm_sum_parts_kernel(const float *__restrict__ parts, const float *__restrict__ scale, uint16_t *__restrict__ y, int N,
                                                             int64_t total, int np) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (i >= total) return;
    typedef float vec __attribute__((ext_vector_type(V)));
    vec p[8];
#pragma unroll
    for (int s = 0; s < 8; ++s)
        if (s < np) p[s] = *reinterpret_cast<const vec *>(parts + s * total + i);
    vec a = p[0];
#pragma unroll
    for (int s = 1; s < 8; ++s)
        if (s < np) a += p[s];
    if (scale) a *= *reinterpret_cast<const vec *>(scale + i % N);
    if constexpr (V == 4) *reinterpret_cast<u32x2 *>(y + i) = u32x2{pack_bf16_rne(a[0], a[1]), pack_bf16_rne(a[2], a[3])};
    else y[i] = (uint16_t)pack_bf16_rne(a[0], 0.f);
}

template <bool I4, bool GUARD>
static int launch_parts(const uint16_t *x, const uint8_t *w, const void *sc, float *parts, int M, int N, int K, GemmTile tile, tileq::KParts np,
                        hipStream_t st) {
    switch (tile) {
        case TILE_32x64: return tileq::launch<I4, 1, 2, 4, 1, 1, 64, 3, GUARD, false, tileq::EPI_F32>(x, w, sc, parts, M, N, K, np, st);
        case TILE_64x64: return tileq::launch<I4, 1, 2, 4, 2, 1, 64, 3, GUARD, false, tileq::EPI_F32>(x, w, sc, parts, M, N, K, np, st);
        default: return tileq::launch<I4, 1, 2, 4, 4, 1, 32, GUARD ? 3 : 4, GUARD, false, tileq::EPI_F32>(x, w, sc, parts, M, N, K, np, st);
    }
}

int gemm_tile_parts_launch(const uint16_t *x, const uint8_t *w, const void *sc, uint16_t *y, int M, int N, int K, bool int4, bool guard, GemmTile tile, int np,
                           int span, float *parts, hipStream_t st) {
    const tileq::KParts kp = {np, span};
    const int rc = int4 ? guard ? launch_parts<true, true>(x, w, sc, parts, M, N, K, tile, kp, st) : launch_parts<true, false>(x, w, sc, parts, M, N, K, tile, kp, st)
                        : guard ? launch_parts<false, true>(x, w, sc, parts, M, N, K, tile, kp, st) : launch_parts<false, false>(x, w, sc, parts, M, N, K, tile, kp, st);
    if (rc) return rc;
    const int64_t total = (int64_t)M * N;
    const float *const scale = int4 ? nullptr : reinterpret_cast<const float *>(sc);
    const bool four = N % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 7u) == 0 && (int4 || aligned16(scale));
    if (four) hipLaunchKernelGGL(gemm_sum_parts_kernel<4>, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, st, parts, scale, y, N, total, np);
    else hipLaunchKernelGGL(gemm_sum_parts_kernel<1>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, parts, scale, y, N, total, np);
    return hip_check(hipGetLastError(), "gemm parts launch");
}

// ---- exact weights, K % 256 == 0: the projections of a prompt, whose tokens must come out as the decode step's do.
// Tiles of 128 or 256 rows x 128 weight rows, or of 32 to 128 x 64: in few tiles a workgroup waits for its weights, and what counts is
// how many workgroups and steps wait at once (two workgroups per compute unit for at most 32 rows; the loop is not unrolled: the
// code of a few steps is fetched as often as it is run).  Whole prompts in us, 128 weight rows for every number of tokens in brackets:
// 24 tokens through 18 layers of 2048 x 16384 1152 (1343), 9 through 6 of 1280 x 3840 262 (321), 37 through 4 of 2048 x 8960 282 (311).
struct ExactCost {
    int bm, bn;  // tile
    float s, c0, c1, d0, d1, b, c2;
};
static const ExactCost kExact32 = {32, 64, 4.87f, -1.63f, .694f, 1.42f, .694f, .870f, .216f};
static const ExactCost kExact[3] = {{64, 64, 1.33f, 2.61f, .817f, 2.61f, .817f, .787f, .023f}, {128, 64, 1.66f, 3.52f, 1.144f, 3.52f, 1.144f, .784f, .043f},
                                    {128, 128, 2.75f, 1.75f, 2.64f, 1.75f, 2.64f, .883f, .170f}};
static const ExactCost kGeglu[4] = {{64, 64, 1.10f, 2.61f, .860f, 2.61f, .860f, .801f, 0.f}, {128, 64, 2.f, 3.88f, 1.197f, 3.88f, 1.197f, .808f, 0.f},
                                    {128, 128, .75f, 4.60f, 2.871f, 4.60f, 2.871f, .823f, 0.f}, {256, 128, 1.4f, 7.18f, 3.784f, 7.18f, 3.784f, .798f, 0.f}};

// us that a launch takes in `parts` K splits of `per` 256-k blocks.  Tiles go to the XCDs in turn, each in all its splits, and a round is over
// when the fullest XCD has dealt its workgroups to its 32 compute units: 33 tiles in 7 parts are 231 workgroups, but 35 on one XCD.  A tile
// takes c0 + c1 * per in the first round and d0 + d1 * per in a further one (of the tiles of 32 rows two fit on a compute unit), the last
// round b + (1 - b) f of it if it is full to f; s is what a launch takes besides, c2 what a MB of fp32 parts takes to be written.  The
// constants of 64 rows and more are fitted to 18700 random products in every number of splits (33 to 700 rows, 128 to 8192 weight rows, 256 to
// 16000 k) and 8900 gated ones, 2 to 5 % standard deviation (two numbers of the 128-row tiles and one of the gated 256 moved by 0.1 to 0.9 us
// where tiles are even; 128 x 64, gated, by 0.9: prompts of 70 to 128 tokens took 1 % longer with it where the
// fit has it even with 128 x 128); the tile and splits they pick take 0.2 % more than the best of all on average.  Of 1400 other products, 65 to 600
// rows, half of them gated, more than half of few steps, the tile picked takes 0.06 % more than the quickest on average and 15 % in the worst case.
static float exact_us(const ExactCost &t, int M, int N, int per, int parts) {
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn), fullest = (tiles + 7) / 8 * parts, rounds = (fullest + 31) / 32;
    const float last = t.b + (1.f - t.b) * (float)(fullest - (rounds - 1) * 32) / 32.f, first = t.c0 + t.c1 * (float)per;
    const float mb = 4e-6f * (float)(tiles * parts) * (float)(t.bm * t.bn);
    return t.s + (rounds == 1 ? last * first : first + ((float)(rounds - 2) + last) * (t.d0 + t.d1 * (float)per)) + t.c2 * mb;
}

// The tile (its rows) that takes a product in the shortest time.  64 rows reach the chip's compute units where 128 leave most of them idle, and
// take a third of the time per k; 256 dequantise a weight half as often.  us, 64 / 128 rows: 101 x 128 x 2048 in eight parts 4.7 / 7.6, 158 x 5120 x
// 2304 in one 12.1 / 27.9, 432 x 5120 x 1536 24.4 / 21.8; gate/up, 64 / 128 / 256 rows: 101 x 8192 x 2048 11.7 / 25.9 / 32.7, 237 x 32512 x 1792 71.6 /
// 49.7 / 38.3.  128 x 64 has the unpacking of 128 rows in as many workgroups as half the rows would make: 256 x 2048 x 16384 in four parts 27.2, in 64 x 64
// tiles in two 31.5, in 128 x 128 in eight 30.0; without it the products of more than 64 rows would take 3 % longer on average, gated ones 4 %.
// (Three stages; four are 2 % slower.)  In one to three steps it is up to 1.4 times as fast as the others too (81 x 2560 x 4352 in six parts 8.6, 64 x 64
// 11.9; gated 78 x 13824 x 512 6.9, 9.3; prompts of 115 to 183 tokens, d = 512 or 768: 0.96 to 0.97 of the time).  Only the choice of the parts counts it
// from four steps on (`splitting`): the parts that it would add there cost the next kernel more, prompts of 110 to 240 tokens, d = 1024 to 1536, 2 to 4 %.
// (In few steps the loop of 128 rows also takes 0.6 us more than the one with all requests of a step in a row did.)  A prompt of
// 256 tokens through 18 layers of 2048 x 16384 2518 -> 2320.
static const ExactCost &exact_pick(int M, int N, int per, int parts, bool geglu, float *us, bool splitting = false) {
    const ExactCost *const t = M <= 32 ? &kExact32 : geglu ? kGeglu : kExact;
    int best = 0;
    *us = exact_us(t[0], M, N, per, parts);
    for (int i = 1; i < (M <= 64 ? 1 : geglu ? 4 : 3); ++i) {
        if (i == 1 && per < 4 && splitting) continue;
        const float u = exact_us(t[i], M, N, per, parts);
        if (u < *us) {
            best = i;
            *us = u;
        }
    }
    return t[best];
}

int gemm_exact_tile(int M, int N, int per, int parts, bool geglu, float *us, int *columns) {
    const ExactCost &t = exact_pick(M, N, per, parts, geglu, us);
    *columns = t.bn;
    return t.bm;
}

template <int EPI>
static int launch_exact(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, void *y, int M, int N, int K, int ksplit, hipStream_t st) {
    float us;
    const tileq::KParts kp = {ksplit, (K / 256 + ksplit - 1) / ksplit * 256};  // (K % 256 == 0)
    const ExactCost &t = exact_pick(M, N, (K / 256 + ksplit - 1) / ksplit, ksplit, EPI == tileq::EPI_GEGLU, &us);
    if (t.bm == 32) return tileq::launch<true, 1, 2, 4, 1, 1, 64, 3, false, true, EPI>(x, wp, sc, y, M, N, K, kp, st);
    if (t.bm == 64) return tileq::launch<true, 1, 2, 4, 2, 1, 64, 3, false, true, EPI>(x, wp, sc, y, M, N, K, kp, st);
    if constexpr (EPI == tileq::EPI_GEGLU) {
        if (t.bm == 256) return tileq::launch<true, 1, 4, 2, 8, 1, 32, 3, false, true, EPI>(x, wp, sc, y, M, N, K, kp, st);
    }
    if (t.bn == 64) return tileq::launch<true, 1, 2, 4, 4, 1, 32, 3, false, true, EPI>(x, wp, sc, y, M, N, K, kp, st);
    return tileq::launch<true, 1, 4, 2, 4, 1, 64, 3, false, true, EPI>(x, wp, sc, y, M, N, K, kp, st);
}

// Decode products of at most 32 rows whose K (or scales) the GEMV of gemv_i4g32_mfma.hip does not take: y fp32 or bf16 [M,N] in one
// pass over the weights.
int gemm_exact_few_rows_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, float *y, int M, int N, int K, bool bf16_out,
                               hipStream_t st) {
    return bf16_out ? tileq::launch<true, 1, 2, 4, 1, 1, 64, 3, true, true, tileq::EPI_BF16>(x, wp, sc, y, M, N, K, {}, st)
                    : tileq::launch<true, 1, 2, 4, 1, 1, 64, 3, true, true, tileq::EPI_F32>(x, wp, sc, y, M, N, K, {}, st);
}

// The K splits of a product, whole 256-k blocks each, the last one possibly shorter.  (With equal parts only, a down projection of 8960 k had
// one part, 63 us of the 125 that its layer took for 37 tokens.)  Rounds of 256 workgroups (512 for up to 32 rows) times the k of each, as the
// splits were chosen by before, miss how tiles fall to the XCDs, what half a chip costs and what the parts cost.  us, so chosen / in other
// parts of the same tiles: 265 x 1344 x 7168 in 7 31.6 / in 6 20.5, 552 x 1280 x 5120 in 5 32.1 / in 4 20.7, 22 x 4480 x 1024 in 4 6.4 / in 2
// 4.9.  kRead: what a MB of parts costs the next kernel: with 0.35 us per MB the down product of 128 tokens, 2048 x 16384, is in eight parts of 128 x
// 64 tiles and the prompt of 18 layers takes 1640-1680 us, with 0.7 in four of 64 x 64 1569-1607.  M counts in whole tiles only: prompt_layout asks for every number of them.
int gemm_exact_splits(int M, int N, int K) {
    constexpr float kRead = .7f;
    const int blocks = K / 256, rows = M <= 32 ? 32 : (M + 63) / 64 * 64;
    int best = 1;
    float best_us = 0.f;
    for (int s = 1; s <= kExactMaxSplits; ++s) {
        const int per = (blocks + s - 1) / s, parts = (blocks + per - 1) / per;
        float us;
        exact_pick(M, N, per, parts, false, &us, true);
        us += kRead * 4e-6f * (float)rows * (float)N * (float)parts;
        if (s == 1 || us < best_us) {
            best = parts;
            best_us = us;
        }
    }
    return best;
}

// q, k and v of a prompt with the rotation and the cache rows in the epilogue: tiles of 64 weight rows, K in one part.
static const ExactCost &qkv_pick(int M, int N, int K) {
    return M <= 32 ? kExact32 : M <= 64 || exact_us(kExact[0], M, N, K / 256, 1) <= exact_us(kExact[1], M, N, K / 256, 1) ? kExact[0] : kExact[1];
}

// What the parts bring may be more than the launch that adds and rotates them takes, 1 to 1.9 us in a queue (its own time is 5 us, most of it the
// way of the parts through memory, which the next kernel has to itself otherwise).  us, in the epilogue / in parts and a launch: 18 layers of
// 2048 x 16384, 24 tokens (four parts) 1088 / 1058, 256 (one) 2085 / 2134; 3 layers of 1792 x 10752, 212 tokens 313 / 325; 6 of 1024 x 4864, 35 tokens
// (four) 283 / 277; 4 of 512 x 3840, 4 tokens (two) 203 / 208.
bool gemm_exact_qkv_pays(int M, int N, int K) {
    const int parts = gemm_exact_splits(M, N, K), per = (K / 256 + parts - 1) / parts;
    float us;
    exact_pick(M, N, per, parts, false, &us);
    return exact_us(qkv_pick(M, N, K), M, N, K / 256, 1) <= us + 1.f;
}

int gemm_exact_qkv_tile(int M, int N, int K) { return qkv_pick(M, N, K).bm; }

int gemm_exact_qkv_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, const QkvOut &out, int M, int K, hipStream_t st) {
    const int N = (out.hq + 2) * out.dh, rows = gemm_exact_qkv_tile(M, N, K);
    if (rows == 32) return tileq::launch<true, 1, 2, 4, 1, 1, 64, 3, false, true, tileq::EPI_QKV>(x, wp, sc, nullptr, M, N, K, {}, st, {out});
    if (rows == 64) return tileq::launch<true, 1, 2, 4, 2, 1, 64, 3, false, true, tileq::EPI_QKV>(x, wp, sc, nullptr, M, N, K, {}, st, {out});
    return tileq::launch<true, 1, 2, 4, 4, 1, 32, 3, false, true, tileq::EPI_QKV>(x, wp, sc, nullptr, M, N, K, {}, st, {out});
}

int gemm_exact_scaled_f32_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, float *y_parts, int M, int N, int K, int ksplit,
                                 hipStream_t st) {
    return launch_exact<tileq::EPI_F32>(x, wp, sc, y_parts, M, N, K, ksplit, st);
}

int gemm_exact_scaled_geglu_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, uint16_t *h, int M, int N, int K, hipStream_t st) {
    return launch_exact<tileq::EPI_GEGLU>(x, wp, sc, h, M, N, K, 1, st);
}

}  // namespace chadq
