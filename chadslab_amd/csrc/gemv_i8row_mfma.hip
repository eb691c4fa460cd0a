// Decode GEMV on int8 per-row weights on the int8 matrix core, any 1..16 activation rows in ONE pass over W (the
// per-row kernel in gemv_i8row.hip streams W once per pair of activation rows).
//
// v_mfma_i32_16x16x64_i8 takes the stored weight bytes as they are, so the K loop has no conversion work at all.
// The fp32 activations are what has to change shape: per activation row and per 2048 k, x is written in fixed point
// with a power-of-two scale, X = rint(x * 2^(20 - e)) with 2^e <= max|x| < 2^(e+1) (|X| <= 2^21), and X as three
// balanced base-256 digits, X = a0 * 2^16 + a1 * 2^8 + a2 with -128 <= a <= 127.  Each digit is one int8 operand
// row; the three int32 dot products are exact and meet again in float64: y = s[n] * sum over blocks 2^(e-20) * (D0 *
// 2^16 + D1 * 2^8 + D2).  What is dropped is at most 2^-21 of the block's largest |x| per element, so a result is off by
// at most scale[n] * sum over blocks of 2^-21 * max_block|x| * sum_{k in block} |W[n,k]| (the result is held to a 1e-3
// relative tolerance; one outlier among the activations costs the small elements of its block their low bits, also
// in rows whose weight at the outlier is zero: chadq_gemv_i8row_fp32 is the form without this).  Integer-valued
// activations below 2^20 are represented exactly and the three digit sums are recombined exactly (in float64), so
// integer sums below 2^24 are exact as in the per-row kernel.  A block with a non-finite activation makes its rows'
// results NaN (the fp32 kernels follow IEEE arithmetic element by element).
//
// One MFMA, D[16x16] += A[16x64] * B[64x16]:
//   B = weights.  Column c is weight row n0 + c (16 rows per wave); lane (c, g = lane/16) supplies 16 k-slots.  A
//       wave fetches 128 k of its 16 rows with two loads of 8 rows x 128 B (lane (c, g) loads piece (c >> 3) + 2g of
//       row c & 7, then of row 8 + (c & 7)); two DPP half-row rotations per word hand every lane the 32 consecutive
//       bytes k = 32g .. 32g + 31 of ITS row c: the B operands of two MFMAs.
//   A = activations.  SETS <= 2 (M <= 4, M <= 8): operand row 4q + d of set s is digit d of activation row 4s + q
//       (row 4q + 3 is zero), so the three digit sums of a result sit in one lane's accumulator registers.  SETS = 3
//       (M <= 16): set d holds digit d of all 16 rows.
// Workgroup = 8 waves on RWS = 1, 2 or 4 blocks of 16 weight rows: wave (rw, kh) multiplies block rw with the kh-th of
// 8 / RWS parts of every 2048 k, so at K <= 2048 a wave's loads - all of its weights - are in flight from the start and
// nothing about the activations can stall the stream.  The 512 threads turn 2048 k of all M activation rows into operand
// order in LDS (SETS x 32 KiB); the activation loads are issued before the weight loads because memory returns in
// order.  Longer rows repeat this per 2048 k with the ring refilled as it is consumed (every load unconditional:
// addresses past the end are clamped and their activations staged as zeros).  The K parts meet in LDS at the end.
//
// What bounds it is how fast one CU takes its weights, about 40 bytes per ns: 3.8 us per 64 rows and 2048 k, however
// few the workgroups are.  So the rows are dealt out until the 256 CUs have one workgroup each: 16 to a workgroup up to
// 4096 rows, 32 up to 8192, else 64.  us at 16 / 32 / 64 rows (64 was all there was), 1 and 16 activation rows:
// 2048 x 2048 4.8 / 4.2 / 5.8 and 8.1 / 8.7 / 10.9; 4096 x 4096 6.9 / 7.2 / 10.2 and 16.4 / 17.0 / 21.1; 2048 x 16384
// 14.7 / 19.1 / 32.9 and 47 / 50 / 65; 8192 x 4096 10.8 / 9.0 / 11.0 and 32 / 18 / 21; 16384 x 2048 9.6 / 7.1 / 7.4 and
// 29 / 17 / 12.  Activations requested two 2048-blocks ahead gave nothing (and spilled at 16 rows).  M plays no part in
// the rule: a row's result does not depend on how many rows come with it.
#include <type_traits>

#include "chadq_common.h"

namespace chadq {

constexpr int kGemvMostParts = 8;

typedef __attribute__((ext_vector_type(4))) int i32x4;

// RWS: blocks of 16 weight rows per workgroup (1, 2 or 4), each shared by 8 / RWS waves
template <int SETS, int RWS>
struct GemvI8Cfg {
    static constexpr int PAIRS = 8;                       // 128-k pair-steps per round (1024 k)
    static constexpr int KHS = 8 / RWS, STEPS = 16 / KHS; // waves of a row block, pair-steps of each per 2048 k
    static constexpr int PAIR_BYTES = SETS * 2048;        // A operands of one pair-step: SETS x 2 MFMAs x 1 KiB
    static constexpr int BUF_BYTES = PAIRS * PAIR_BYTES;  // one round's operands: SETS x 16 KiB
    static constexpr int MROWS = SETS == 3 ? 16 : 4 * SETS;  // activation rows the staging covers
    static constexpr int PARTS = 512 / MROWS;             // staging threads per activation row
    static constexpr int XIT = 128 / PARTS;               // 16-k pieces a thread stages per 2048 k: 1 / 2 / 4
    static constexpr int RES = SETS == 3 ? 4 : SETS;      // results per lane
    static constexpr int AMAX_OFF = 2 * BUF_BYTES;        // [MROWS][8 waves] largest |x| bits
    static constexpr int FOLD_OFF = AMAX_OFF + 16 * 8 * 4;  // [waves but the first of each row block][RES][64 lanes] float64
    static constexpr int LDS = FOLD_OFF + (8 - RWS) * RES * 64 * 8;
};

// lanes 8..15 of every row of 16 take src from the lane 8 below, lanes 0..7 keep old (BANKS = 0xC); or lanes 0..7 take
// src from the lane 8 above and lanes 8..15 keep old (BANKS = 0x3)
template <int BANKS>
__device__ __forceinline__ int half_row_merge(uint32_t old, uint32_t src) {
    return __builtin_amdgcn_update_dpp((int)old, (int)src, 0x128, 0xF, BANKS, false);
}

template <int SETS, int RWS>
__global__ __launch_bounds__(512) void gemv_i8row_mfma_kernel(const float *__restrict__ x, const int8_t *w8,
                                                              const float *sc, float *__restrict__ y, int M, int N,
                                                              int K, int bf16_out, int per, double *__restrict__ parts) {
    using C = GemvI8Cfg<SETS, RWS>;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    uint32_t *amax = reinterpret_cast<uint32_t *>(smem + C::AMAX_OFF);

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int rw = wave % RWS, kh = wave / RWS;
    const int c = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (16 * RWS) + rw * 16;
    // the two loads of a pair-step: rows (c & 7) and 8 + (c & 7) of the wave's 16, piece (c >> 3) + 2g of 128 bytes;
    // rows past the end are clamped, computed and never stored
    const int rx = (n0 + (c & 7) < N) ? n0 + (c & 7) : N - 1, ry = (n0 + 8 + (c & 7) < N) ? n0 + 8 + (c & 7) : N - 1;
    const unsigned char *wbase = reinterpret_cast<const unsigned char *>(w8) + 16 * ((c >> 3) + 2 * g);
    const unsigned char *wpx = wbase + (size_t)rx * K, *wpy = wbase + (size_t)ry * K;
    const int pairs = K >> 7, supers = (K + 2047) >> 11;
    const int sr0 = blockIdx.y * per, sr1 = sr0 + per < supers ? sr0 + per : supers;  // the workgroup's blocks of 2048 k
    auto pair_off = [&](int sr, int t) {  // byte offset of pair-step t of this wave in 2048-block sr
        const int p = sr * 16 + kh * C::STEPS + t;
        return (size_t)((p < pairs) ? p : pairs - 1) * 128;
    };

    // staging role of this thread: activation row sm (clamped for the loads), 16-k pieces so, so + PARTS, ... of 2048 k
    const int sm = threadIdx.x % C::MROWS, so = threadIdx.x / C::MROWS;
    const float *xrow = x + (size_t)((sm < M) ? sm : M - 1) * K;
    f32x4 xr[C::XIT][4];
    auto request_x = [&](int sr) {
#pragma unroll
        for (int it = 0; it < C::XIT; ++it) {
            int k = sr * 2048 + 16 * (so + it * C::PARTS);
            k = (k < K) ? k : K - 16;
#pragma unroll
            for (int q = 0; q < 4; ++q) xr[it][q] = *reinterpret_cast<const f32x4 *>(xrow + k + 4 * q);
        }
    };
    // registers -> fixed point with the block's scale -> three digits -> operand order; leaves the block's row scales
    // 2^(e-20) (NaN for a non-finite block) in bscale[] of every lane
    float bscale[C::RES];
    auto stage_x = [&](int sr) {
        float v[C::XIT][16];
        uint32_t big = 0;  // largest exponent field among this thread's values
#pragma unroll
        for (int it = 0; it < C::XIT; ++it) {
            const bool live = sr * 2048 + 16 * (so + it * C::PARTS) < K;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v[it][4 * q + 0] = live ? xr[it][q].x : 0.f;
                v[it][4 * q + 1] = live ? xr[it][q].y : 0.f;
                v[it][4 * q + 2] = live ? xr[it][q].z : 0.f;
                v[it][4 * q + 3] = live ? xr[it][q].w : 0.f;
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint32_t b = __builtin_amdgcn_ubfe(__float_as_uint(v[it][e]), 23, 8);
                big = b > big ? b : big;
            }
        }
        // the row's largest exponent in this block: over the lanes of this wave that stage the row, then over the waves
#pragma unroll
        for (int off = C::MROWS; off < 64; off <<= 1) {
            const uint32_t o = (uint32_t)__shfl_xor((int)big, off);
            big = o > big ? o : big;
        }
        if (lane < C::MROWS) amax[sm * 8 + wave] = big;
        __syncthreads();
        auto row_exp = [&](int m) {  // exponent field of the row's largest |x| (255: non-finite)
            const u32x4 a = *reinterpret_cast<const u32x4 *>(amax + m * 8), b = *reinterpret_cast<const u32x4 *>(amax + m * 8 + 4);
            uint32_t t = a.x > a.y ? a.x : a.y, u = a.z > a.w ? a.z : a.w, p = b.x > b.y ? b.x : b.y, q = b.z > b.w ? b.z : b.w;
            t = t > u ? t : u;
            p = p > q ? p : q;
            return (int)(t > p ? t : p);
        };
#pragma unroll
        for (int r = 0; r < C::RES; ++r) {
            const int m = (SETS == 3) ? 4 * g + r : 4 * r + g;
            const int eb = row_exp(m);
            // 2^(e - 20) as a float built from its exponent field; tiny blocks are scaled as if max|x| were 2^-100
            const int ec = eb < 27 ? 27 : eb;
            bscale[r] = (eb == 255) ? __uint_as_float(0x7FC00000u) : __uint_as_float((uint32_t)(ec - 20) << 23);
        }
        const int ebm = row_exp(sm);
        const int ecm = ebm < 27 ? 27 : (ebm > 254 ? 254 : ebm);
        const float up = __uint_as_float((uint32_t)(274 - ecm) << 23);  // 2^(20 - e)
#pragma unroll
        for (int it = 0; it < C::XIT; ++it) {
            uint32_t d0[4], d1[4], d2[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                // X = rint(x * 2^(20 - e)) sits in the mantissa of x * 2^(20 - e) + 1.5 * 2^23 as 0x400000 + X; the
                // low three bytes of (X + 0x808080) ^ 0x808080 are the balanced base-256 digits a2, a1, a0 of X
                uint32_t z[4];
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    z[b] = (__float_as_uint(__builtin_fmaf(v[it][4 * w + b], up, 12582912.0f)) + 0x408080u) ^ 0x808080u;
                // 4 x 4 byte transpose (three rows of it): digit d of four consecutive k in one word
                const uint32_t l01 = __builtin_amdgcn_perm(z[1], z[0], 0x05010400u), h01 = __builtin_amdgcn_perm(z[1], z[0], 0x07030602u);
                const uint32_t l23 = __builtin_amdgcn_perm(z[3], z[2], 0x05010400u), h23 = __builtin_amdgcn_perm(z[3], z[2], 0x07030602u);
                d2[w] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
                d1[w] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
                d0[w] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
            }
            const int osr = so + it * C::PARTS;  // piece of the 2048-block: round osr >> 6, piece o of the round
            const int o = osr & 63, t8 = o >> 3, gg = (o >> 1) & 3, jj = o & 1;
            unsigned char *blk = smem + (osr >> 6) * C::BUF_BYTES + t8 * C::PAIR_BYTES + jj * 1024;
            if constexpr (SETS == 3) {
                *reinterpret_cast<u32x4 *>(blk + (gg * 16 + sm) * 16) = u32x4{d0[0], d0[1], d0[2], d0[3]};
                *reinterpret_cast<u32x4 *>(blk + 2048 + (gg * 16 + sm) * 16) = u32x4{d1[0], d1[1], d1[2], d1[3]};
                *reinterpret_cast<u32x4 *>(blk + 4096 + (gg * 16 + sm) * 16) = u32x4{d2[0], d2[1], d2[2], d2[3]};
            } else {
                // the four operand rows of activation row (set, q); XOR-ing the low slot bits with (pair-step, MFMA)
                // spreads a wave's 64 pieces over all banks
                const int f = jj + 2 * (t8 & 1), base = (gg * 16 + 4 * (sm & 3)) ^ f;
                blk += (sm >> 2) * 2048;
                *reinterpret_cast<u32x4 *>(blk + (base ^ 0) * 16) = u32x4{d0[0], d0[1], d0[2], d0[3]};
                *reinterpret_cast<u32x4 *>(blk + (base ^ 1) * 16) = u32x4{d1[0], d1[1], d1[2], d1[3]};
                *reinterpret_cast<u32x4 *>(blk + (base ^ 2) * 16) = u32x4{d2[0], d2[1], d2[2], d2[3]};
                *reinterpret_cast<u32x4 *>(blk + (base ^ 3) * 16) = u32x4{0u, 0u, 0u, 0u};
            }
        }
    };

    request_x(sr0);
    u32x4 ring[2 * C::STEPS];
#pragma unroll
    for (int t = 0; t < C::STEPS; ++t) {
        ring[2 * t] = load_nt_b128(wpx + pair_off(sr0, t));
        ring[2 * t + 1] = load_nt_b128(wpy + pair_off(sr0, t));
    }
    // the weight stream starts before the staging below waits for anything (w8 and sc are not declared restrict so
    // that these loads cannot be moved below this point)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    stage_x(sr0);
    if (sr0 + 1 < sr1) request_x(sr0 + 1);
    __syncthreads();

    double yacc[C::RES];
#pragma unroll
    for (int r = 0; r < C::RES; ++r) yacc[r] = 0.;
    const int t0 = kh * C::STEPS % C::PAIRS;  // the wave's first pair-step in its round of 1024 k
    const unsigned char *abuf = smem + kh * C::STEPS / C::PAIRS * C::BUF_BYTES + t0 * C::PAIR_BYTES;
    auto multiply = [&](int sr, auto refill) {  // this wave's part of 2048-block sr; refill: request the next block's
        i32x4 acc[SETS][2];
#pragma unroll
        for (int s = 0; s < SETS; ++s) acc[s][0] = acc[s][1] = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < C::STEPS; ++t) {
            // wait for this pair-step's weights, then put the request for the next 2048-block in the queue
            asm volatile("" : "+v"(ring[2 * t]), "+v"(ring[2 * t + 1]));
            const u32x4 wx = ring[2 * t], wy = ring[2 * t + 1];
            if constexpr (decltype(refill)::value) {
                ring[2 * t] = load_nt_b128(wpx + pair_off(sr + 1, t));
                ring[2 * t + 1] = load_nt_b128(wpy + pair_off(sr + 1, t));
            }
            __builtin_amdgcn_sched_barrier(0);
            // this lane's row, k = 32g .. 32g + 15 and 32g + 16 .. 32g + 31 of the pair-step
            const i32x4 b0 = {half_row_merge<0xC>(wx.x, wy.x), half_row_merge<0xC>(wx.y, wy.y), half_row_merge<0xC>(wx.z, wy.z),
                              half_row_merge<0xC>(wx.w, wy.w)};
            const i32x4 b1 = {half_row_merge<0x3>(wy.x, wx.x), half_row_merge<0x3>(wy.y, wx.y), half_row_merge<0x3>(wy.z, wx.z),
                              half_row_merge<0x3>(wy.w, wx.w)};
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int s = 0; s < SETS; ++s) {
                    const int slot = (SETS == 3) ? lane : (lane ^ (jj + 2 * (t & 1)));  // (t0 is even)
                    const i32x4 av = *reinterpret_cast<const i32x4 *>(abuf + t * C::PAIR_BYTES + (s * 2 + jj) * 1024 + slot * 16);
                    acc[s][jj] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, jj ? b1 : b0, acc[s][jj], 0, 0, 0);
                }
        }
        // the digit sums meet in float64, where D0 * 2^16 + D1 * 2^8 + D2 (more than the 24 bits of a float before its
        // terms cancel) and its product with the block's power of two are exact; the waves' sums are rounded to fp32 once
        auto combine = [](int d0, int d1, int d2) { return __builtin_fma((double)d0, 65536.0, __builtin_fma((double)d1, 256.0, (double)d2)); };
        if constexpr (SETS == 3) {
            const i32x4 e0 = acc[0][0] + acc[0][1], e1 = acc[1][0] + acc[1][1], e2 = acc[2][0] + acc[2][1];
            const int q0[4] = {e0.x, e0.y, e0.z, e0.w}, q1[4] = {e1.x, e1.y, e1.z, e1.w}, q2[4] = {e2.x, e2.y, e2.z, e2.w};
#pragma unroll
            for (int r = 0; r < 4; ++r)
                yacc[r] = __builtin_fma((double)bscale[r], combine(q0[r], q1[r], q2[r]), yacc[r]);
        } else {
#pragma unroll
            for (int s = 0; s < SETS; ++s) {
                const i32x4 e = acc[s][0] + acc[s][1];
                yacc[s] = __builtin_fma((double)bscale[s], combine(e.x, e.y, e.z), yacc[s]);
            }
        }
    };
    for (int sr = sr0; sr + 1 < sr1; ++sr) {
        multiply(sr, std::true_type{});
        __syncthreads();  // every wave is done with this block's operands and row maxima
        stage_x(sr + 1);
        request_x(sr + 2 < sr1 ? sr + 2 : sr1 - 1);
        __syncthreads();
    }
    multiply(sr1 - 1, std::false_type{});

    // the other waves of the row block hand their sums over
    double *const fold = reinterpret_cast<double *>(smem + C::FOLD_OFF) + rw * C::RES * 64 + lane;
    if (kh) {
#pragma unroll
        for (int r = 0; r < C::RES; ++r) fold[((kh - 1) * RWS * C::RES + r) * 64] = yacc[r];
    }
    __syncthreads();
    if (kh) return;
#pragma unroll
    for (int h = 0; h < C::KHS - 1; ++h)
#pragma unroll
        for (int r = 0; r < C::RES; ++r) yacc[r] += fold[(h * RWS * C::RES + r) * 64];
    const int n = n0 + c;
    const float scale = (n < N) ? sc[n] : 0.f;
#pragma unroll
    for (int r = 0; r < C::RES; ++r) {
        const int m = (SETS == 3) ? 4 * g + r : 4 * r + g;
        if (m < M && n < N) {
            if (parts) parts[((size_t)blockIdx.y * M + m) * N + n] = yacc[r];
            else store_sum(y, (size_t)m * N + n, (float)yacc[r] * scale, bf16_out);
        }
    }
}

bool gemv_i8row_mfma_ok(int M, int K) { return M >= 1 && M <= 16 && K % 128 == 0; }

template <int SETS, int RWS>
static int launch_i8_mfma(const float *x, const int8_t *w8, const float *sc, float *y, int M, int N, int K, bool bf16_out, hipStream_t st, int np = 1,
                          double *parts = nullptr) {
    using C = GemvI8Cfg<SETS, RWS>;
    static std::atomic<bool> attr_set{false};  // setting it twice from two threads is harmless
    if (!attr_set.load(std::memory_order_acquire)) {
        CHADQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&gemv_i8row_mfma_kernel<SETS, RWS>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS));
        attr_set.store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL((gemv_i8row_mfma_kernel<SETS, RWS>), dim3((N + 16 * RWS - 1) / (16 * RWS), np), dim3(512), C::LDS, st, x, w8, sc, y, M, N, K,
                       (int)bf16_out, ((K + 2047) / 2048 + np - 1) / np, parts);
    return hip_check(hipGetLastError(), "gemv_i8row_mfma launch");
}

template <int SETS>
static int launch_i8_mfma(const float *x, const int8_t *w8, const float *sc, float *y, int M, int N, int K, bool bf16_out, hipStream_t st) {
    if (N <= 4096) return launch_i8_mfma<SETS, 1>(x, w8, sc, y, M, N, K, bf16_out, st);
    if (N <= 8192) return launch_i8_mfma<SETS, 2>(x, w8, sc, y, M, N, K, bf16_out, st);
    return launch_i8_mfma<SETS, 4>(x, w8, sc, y, M, N, K, bf16_out, st);
}

// 1..16 activation rows, K a multiple of 128 (x and w8 16-byte aligned as for every int8 GEMV)
int gemv_i8row_mfma_launch(const float *x, const int8_t *w8, const float *sc, float *y, int M, int N, int K,
                           bool bf16_out, hipStream_t st) {
    if (M <= 4) return launch_i8_mfma<1>(x, w8, sc, y, M, N, K, bf16_out, st);
    if (M <= 8) return launch_i8_mfma<2>(x, w8, sc, y, M, N, K, bf16_out, st);
    return launch_i8_mfma<3>(x, w8, sc, y, M, N, K, bf16_out, st);
}

// y[m,n] = the parts of an element added in order, times its row's scale if there is one, rounded once
template <typename T>
__global__ __launch_bounds__(256) void gemv_sum_parts_kernel(const T *__restrict__ parts, const float *__restrict__ scale, float *__restrict__ y, int N, int total,
                                                             int np, int bf16_out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    T p[kGemvMostParts];
#pragma unroll
    for (int s = 0; s < kGemvMostParts; ++s)
        if (s < np) p[s] = parts[(size_t)s * total + i];
    T a = p[0];
#pragma unroll
    for (int s = 1; s < kGemvMostParts; ++s)
        if (s < np) a += p[s];
    store_sum(y, i, scale ? (float)a * scale[i % N] : (float)a, bf16_out);
}

int gemv_sum_parts_launch(const float *parts, float *y, int M, int N, int np, bool bf16_out, hipStream_t st) {
    hipLaunchKernelGGL(gemv_sum_parts_kernel<float>, dim3((M * N + 255) / 256), dim3(256), 0, st, parts, nullptr, y, N, M * N, np, (int)bf16_out);
    return hip_check(hipGetLastError(), "gemv parts launch");
}

// Parts of K (float64 sums, so the result is as precise as in one part) and the blocks of 16 weight rows of a workgroup that go with them, where
// workgroups would walk many blocks of 2048 k.  A block takes a workgroup a share for its activations' way to LDS (by rows) and one for its weights (by
// their rows, and less while compute units idle); few weight rows want more workgroups along K, many activation rows also fewer that stage them: 64
// weight rows each instead of 16 or 32.  The second launch and what goes with it take 3.5 us.  us, in one part / in parts: 512 x 16384, 1 row 13.2 /
// 6.9, 4 16.7 / 7.2, 8 25.8 / 8.3, 16 47.2 / 10.2; 2048 x 8192, 8 rows 15.4 / 9.3; 4096 x 16384, 16 48.0 / 29.1; 8192 x 8192, 16 35.3 / 28.3.
// 147 random calls in parts: 0.56 of the time in a row, 0.72 waited for one by one, none slower.
int gemv_i8row_parts(int M, int N, int K, int *rws) {
    if (!gemv_i8row_mfma_ok(M, K) || N < 1 || N > 8192) return 1;
    const float stage = M <= 4 ? .8f : M <= 8 ? 1.9f : 4.2f, rows = M <= 4 ? 1.4f : M <= 8 ? 1.5f : 1.45f;
    const int blocks = (K + 2047) / 2048;
    auto block_us = [&](int r, int wgs) { return stage + rows * (float)r * (.4f + .6f * (float)(wgs < 256 ? wgs : 256) / 256.f); };
    const int now = N <= 4096 ? 1 : 2;
    float best = (float)blocks * block_us(now, (N + 16 * now - 1) / (16 * now)) - 3.5f;
    int parts = 1;
    for (int r = 1; r <= 4; r *= 2) {
        const int wgs = (N + 16 * r - 1) / (16 * r);
        for (int s = 2; s <= kGemvMostParts && s <= blocks && wgs * s <= 256; ++s) {
            const int per = (blocks + s - 1) / s;
            const float us = (float)per * block_us(r, wgs * s);
            if ((blocks + per - 1) / per == s && us < best) {
                best = us;
                parts = s;
                *rws = r;
            }
        }
    }
    return parts;
}

template <int SETS>
static int launch_i8_parts(const float *x, const int8_t *w8, const float *sc, float *y, int M, int N, int K, int np, int rws, double *parts, hipStream_t st) {
    return rws == 1   ? launch_i8_mfma<SETS, 1>(x, w8, sc, y, M, N, K, false, st, np, parts)
           : rws == 2 ? launch_i8_mfma<SETS, 2>(x, w8, sc, y, M, N, K, false, st, np, parts)
                      : launch_i8_mfma<SETS, 4>(x, w8, sc, y, M, N, K, false, st, np, parts);
}

int gemv_i8row_parts_launch(const float *x, const int8_t *w8, const float *sc, float *y, int M, int N, int K, bool bf16_out, int np, int rws,
                            double *parts, hipStream_t st) {
    const int rc = M <= 4   ? launch_i8_parts<1>(x, w8, sc, y, M, N, K, np, rws, parts, st)
                   : M <= 8 ? launch_i8_parts<2>(x, w8, sc, y, M, N, K, np, rws, parts, st)
                            : launch_i8_parts<3>(x, w8, sc, y, M, N, K, np, rws, parts, st);
    if (rc) return rc;
    hipLaunchKernelGGL(gemv_sum_parts_kernel<double>, dim3((M * N + 255) / 256), dim3(256), 0, st, parts, sc, y, N, M * N, np, (int)bf16_out);
    return hip_check(hipGetLastError(), "gemv parts launch");
}

}  // namespace chadq
