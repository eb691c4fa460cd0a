// Expert products of a mixture of experts for at most 16 rows per expert (a few decoding tokens): a stream of the weights.
//
// What bounds it: the weight stream.  A 4096 x 14336 expert holds 99 MB of packed weights and scales for one to sixteen
// rows of activations.  The many-row kernel (gemm_skinny_i4g32.hip) takes 256 weight rows per workgroup: with few experts
// hit that is one and a fraction rounds of the chip, the last one nearly empty.  Here:
//   * An item of work is 32 weight rows (MODE 1: 16 features of gate and up; MODE 0: 32 rows of down) times K, or times a
//     K split.  Three workgroups per compute unit walk the items at a stride of the grid, and the loads of the next item
//     are requested while the present one is summed, so a workgroup's stream has no gap between items.
//   * The four waves of a workgroup take the item's blocks of 256 k in turn; their sums meet in LDS once per item.
//   * Weights and scales go straight to registers, a block (4 KiB of weights) ahead of the one being summed.  Three waves per SIMD with one
//     block ahead measured 4-8 % faster than two with two ahead.
//   * Where an expert's rows of x or h fit into LDS and a workgroup has items enough (few_launch), they are put there once per
//     expert and K split, already in operand order, a workgroup's items are neighbours instead of a grid apart, and, with at most
//     four tokens, two blocks of weights are on their way: a block's activations are 32 registers to its weights' 24, read again for every
//     item.  4 tokens, 8 experts of 4096 x 14336: gate/up 87 -> 77 us, down 50 -> 49; four blocks in flight are no faster than three.
//   * Otherwise the activations come from the caches, into single registers: a piece is requested again for the next block as soon as its MFMAs
//     have been issued (the caches are nearer than the memory the weights come from).
//   * Through LDS with more than four tokens there is one block ahead as well: two of them and a sum per scale group modulo 4 are some ten
//     registers more than there are.  96 whole calls of 5 to 16 tokens against one sum and two blocks ahead: 0.987 of the time on average,
//     1.028 in the worst; with two ahead and the scales requested a block later, which spilled nothing, 1.010 and 1.048; with spills 1.06.
//   * At most four tokens (FEW): the 16 rows of the A operand are four tokens of four scale groups, each lane group's row non-zero only
//     where it meets that group's words, so the weights are used in the registers they arrived in (no exchange between lanes), the
//     sums of four groups come out in one register each and one FMA per four groups and row is left of four: 188 vector instructions per
//     4 KiB instead of 275.  The whole call, us, before in brackets: 4 tokens, 8 experts of 4096 x 14336 119 (134), with `stream` as
//     below; 2 tokens 86 (98); 3 of 16 of 2304 x 12032 69 (78), 3 of 4 of 3328 x 2816 25.6 (27.5).  What is left at 4 tokens is the stream:
//     with the arithmetic taken out the call takes 108.
//   * `stream`: weights are requested non-temporal where all experts together do not fit into the 256 MB memory-side cache by far.  Row order,
//     us, 4 tokens of 8 experts with / without: 4096 x 14336 (793 MB) 117 / 125, 4096 x 8192 (453 MB) 85.1 / 88.2, 2048 x 14336 (396 MB) 70.9 /
//     70.1, 3072 x 7168 (297 MB) 59.4 / 57.8, 1024 x 2048 19.8 / 19.0: the line is at 400 MB.
//   * In row order a load takes whole 128-byte lines of 8 rows, not 64 bytes of 16 (gate/up 97 -> 87 us); two DPP moves
//     per register pair put the halves in place.
// Gate/up | down in us, 8 experts of 4096 x 14336, top 2, the skinny kernel in brackets: 4 tokens 87 | 50 (130 | 72),
// 16 tokens 145 | 81 (191 | 85); 16 experts of 2048 x 4096, top 4, 16 tokens 46 | 27 (47 | 24: the one shape found whose
// down product is slower here; the whole call is the quicker one all the same, 84.6 against 88.5); 1 token of 1024 x 2048
// 5.2 | 4.5 (12.8 | 7.0).
// Arithmetic: v_mfma_f32_16x16x32_bf16 on unscaled weights.  A lane holds a whole scale group of its weight row (16
// bytes); the lanes' words are exchanged (v_permlane16_swap, v_permlane32_swap) so that one MFMA holds one scale group (FEW: four MFMAs
// take the four words of a lane in turn; one MFMA adds its lane groups' eight products in that order too, so both forms have the same bits,
// and both keep a sum per scale group modulo 4 and add those at the end of an item);
// nibbles become the bf16 value u / 2^9 (unpack8_fp8), another MFMA of the same activations with the constant -8 / 2^9 takes
// the 8 off beforehand for both of the item's row blocks, one fp32 FMA per value applies the scale and the finished sum is
// multiplied by 2^9: weights are exact.  32 x 15 < 2^9, so every group's sum is finite for all finite activations, and it
// errs by 8 / 2^24 of its largest activation at most where the weight there is 0.  (With 128 + u, the magic number of the
// GEMVs, sums overflowed to NaN from activations of 1e35 on and the error was 17 times this: 512 x 512, one activation 1e5
// or 1e6 times the others and all weights there 0, 8.9e-3 or 0.21 off, now 2.4e-3 or 4.4e-3, of which 2.3e-3 is the
// rounding of h and y.  Signed operands, v_cvt_off_f32_i4 and no second MFMA, would leave no error and take 4 % more time;
// this form takes 0.3 % more than 128 + u.)  An infinite activation gives NaN, as in the GEMVs.
// Blocks past the end and rows without a token are requested beyond the buffer's range and arrive as zeros.
#include <type_traits>

#include "chadq_common.h"

namespace chadq {

constexpr int FEW_ROWS = 16;     // activation rows of an expert
constexpr int FEW_ENTRIES = 16;  // experts (one entry of the tile list each, as every expert has at most FEW_ROWS rows)
constexpr int RB = 2;            // blocks of 16 weight rows per item
constexpr int kOwnLds = FEW_ENTRIES * (56 + 4 * FEW_ROWS) + 2 * 4 * RB * 64 * 16;  // s_ent, s_xoff, s_red of the kernel
// Activations in LDS: what leaves three workgroups on a compute unit (its LDS is dealt out in pieces of 1280 bytes).
constexpr int kXlBytes = 163840 / 3 / 1280 * 1280 - kOwnLds;
constexpr uint32_t kBeyond = 0x80000000u;
constexpr int kRange = 0x7FFFFFFF;

// 8 nibbles u -> 8 bf16 u / 2^9, exact: a nibble in a byte of its own is the e4m3 number u / 2^9 (its low eight values are
// the subnormals, the others the next binade, with the same spacing).  Order: (u0, u2) (u4, u6) (u1, u3) (u5, u7).
__device__ __forceinline__ void unpack8_fp8(uint32_t w, uint32_t p[4]) {
    const uint32_t lo = w & 0x0F0F0F0Fu, hi = (w >> 4) & 0x0F0F0F0Fu;
    p[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, false));
    p[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.f, true));
    p[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, false));
    p[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.f, true));
}
// 8 bf16 activations in the same order
__device__ __forceinline__ void order_x8(const uint32_t a[4], uint32_t o[4]) {
    o[0] = __builtin_amdgcn_perm(a[1], a[0], 0x05040100u);
    o[1] = __builtin_amdgcn_perm(a[3], a[2], 0x05040100u);
    o[2] = __builtin_amdgcn_perm(a[1], a[0], 0x07060302u);
    o[3] = __builtin_amdgcn_perm(a[3], a[2], 0x07060302u);
}

// XL: activations through LDS (at most kXlBytes of them); with FEW two blocks of weights on their way beside the one being summed, else one.  FEW: no expert
// has more than four rows.  stream: weights are requested non-temporal (in tile order they always are).
template <int MODE, bool TILED, bool XL, bool FEW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void moe_few_i4g32_kernel(
    const GemmGroup *__restrict__ groups, const int32_t *__restrict__ tiles, const int32_t *__restrict__ tok, int ntiles, int E, int N,
    int K, int nsplit, int stream, size_t split_stride) {
    struct Entry {
        const void *w[2], *s[2], *x;
        void *y;
        int rows, pad;
    };
    __shared__ Entry s_ent[FEW_ENTRIES];
    __shared__ uint32_t s_xoff[FEW_ENTRIES][FEW_ROWS];
    __shared__ __attribute__((aligned(16))) f32x4 s_red[2][4][RB][64];
    static_assert(sizeof(s_ent) + sizeof(s_xoff) + sizeof(s_red) == kOwnLds, "the LDS that kXlBytes leaves out");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, j = lane >> 4;

    {   // thread (entry, row)
        const int n = tid >> 4, m = tid & 15;
        const int tile = n < ntiles ? tiles[n] : -1;
        int rows = 0;
        if (tile >= 0) {
            const int e = tile & 0xFFFF;
            const GemmGroup a = groups[MODE == 1 ? e : 2 * E + e];
            rows = a.M < FEW_ROWS ? a.M : FEW_ROWS;
            uint32_t row = m;
            if (MODE == 1) row = m < rows ? (uint32_t)tok[a.pad + m] : 0u;
            s_xoff[n][m] = m < rows ? row * (uint32_t)K * 2u : kBeyond;
            if (m == 0) {
                const GemmGroup b = groups[MODE == 1 ? E + e : 2 * E + e], d = groups[2 * E + e];
                s_ent[n] = Entry{{a.w, b.w}, {a.sc, b.sc}, a.x, MODE == 1 ? const_cast<uint16_t *>(d.x) : a.y, rows, 0};
            }
        } else if (m == 0) {
            s_ent[n].rows = 0;
        }
    }
    __syncthreads();
    int entries = 0;  // the list holds them in front
    while (entries < ntiles && s_ent[entries].rows > 0) ++entries;
    entries = __builtin_amdgcn_readfirstlane(entries);
    const int ntn = MODE == 1 ? N / 16 : N / 32, per = MODE == 1 ? ntn : ntn * nsplit;
    const int all = entries * per, nb = K >> 8;
    // items of a workgroup: every grid-th, or (XL: the activations change with the expert) a run of neighbours
    const int stride = XL ? 1 : gridDim.x, begin = XL ? (int)((int64_t)blockIdx.x * all / gridDim.x) : blockIdx.x;
    const int total = XL ? (int)((int64_t)(blockIdx.x + 1) * all / gridDim.x) : all;
    auto first_block = [&](int split) { return MODE == 1 ? split * nb : split * nb / nsplit; };
    auto blocks_of = [&](int item) {  // of each wave
        const int split = MODE == 1 ? 0 : item % per / ntn;
        return (first_block(split + 1) - first_block(split) + 3) >> 2;
    };

    struct Block {  // 256 k = eight scale groups
        u32x4 w[RB][2], s[RB];
    };
    // The activations of the block being summed (FEW), or of half of it; a place is refilled as soon as it has been used.
    u32x4 xq[XL ? 1 : FEW ? 8 : 4];
    // ---- the request side
    int l_item = begin, l_i = 0, l_n = 0, l_kb = 0, l_end = 0;
    __amdgpu_buffer_rsrc_t wr[RB], sr[RB], xr, x_rsrc, x_rsrc0;
    uint32_t x_voff = kBeyond, x_kb = 0, x_voff0 = kBeyond, x_kb0 = 0;  // where the activations of the last block requested and of the one before it are
    uint32_t woff = 0, soff = 0, xoff = 0;  // of the lane, in the first row block
    // the second row block: the same rows of the up matrix, or the next 16 rows
    const uint32_t wblk = MODE == 1 ? 0u : TILED ? 256u : 8u * K, sblk = MODE == 1 ? 0u : TILED ? 128u : (uint32_t)K;
    auto uniform = [](const void *p) {
        const uint64_t v = reinterpret_cast<uint64_t>(p);
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
        return reinterpret_cast<void *>(((uint64_t)hi << 32) | lo);
    };
    auto open = [&]() {
        const int en = l_item / per, rem = l_item % per, nt = rem % ntn, split = rem / ntn;
        l_kb = first_block(split) + wave;
        l_end = first_block(split + 1);
        l_n = blocks_of(l_item);
        l_i = 0;
        xr = __builtin_amdgcn_make_buffer_rsrc(uniform(s_ent[en].x), 0, kRange, 0x00020000);
        xoff = FEW ? (r >> 2) == j ? s_xoff[en][r & 3] + 64u * j : kBeyond : s_xoff[en][r] + 16u * j;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            wr[b] = __builtin_amdgcn_make_buffer_rsrc(uniform(s_ent[en].w[b]), 0, kRange, 0x00020000);
            sr[b] = __builtin_amdgcn_make_buffer_rsrc(uniform(s_ent[en].s[b]), 0, kRange, 0x00020000);
        }
        const uint32_t n = (MODE == 1 ? nt * 16 : nt * 32) + r;
        if (TILED) {  // units of 32 rows x 256 k: [8 groups][32 rows][16 B]; scales [even, odd groups][32 rows][4]
            woff = (n >> 5) * (uint32_t)nb * 4096u + j * 512u + (n & 31u) * 16u;
            soff = (n >> 5) * (uint32_t)nb * 512u + (n & 31u) * 8u;
        } else {  // a load takes 8 rows x 128 bytes, whole lines: the lanes of rows 8..15 take groups 4..7 of rows 0..7
            woff = (n & ~8u) * (uint32_t)(K >> 1) + j * 16u + (r >> 3) * 64u;
            soff = n * (uint32_t)(K >> 4);
        }
    };
    auto request = [&](Block &q) {
        x_rsrc0 = x_rsrc;
        x_voff0 = x_voff;
        x_kb0 = x_kb;
        if (l_item >= total) {
            x_voff = kBeyond;
            return;
        }
        const uint32_t kb = l_kb, beyond = l_kb < l_end ? 0u : kBeyond, wv = woff | beyond, sv = soff | beyond, xv = xoff | beyond;
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            if (TILED) {
                const uint32_t sk = kb * 512u + b * sblk;
                const u32x2 ev = __builtin_amdgcn_raw_buffer_load_b64(sr[b], sv, sk, 0), od = __builtin_amdgcn_raw_buffer_load_b64(sr[b], sv, sk + 256u, 0);
                q.s[b] = u32x4{ev.x, ev.y, od.x, od.y};
            } else {
                q.s[b] = __builtin_amdgcn_raw_buffer_load_b128(sr[b], sv, kb * 16u + b * sblk, 0);
            }
        }
        auto weights = [&](auto policy) {
#pragma unroll
            for (int b = 0; b < RB; ++b)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    q.w[b][h] = __builtin_amdgcn_raw_buffer_load_b128(wr[b], wv, kb * (TILED ? 4096u : 128u) + b * wblk + h * (TILED ? 2048u : 4u * K),
                                                                      decltype(policy)::value);
        };
        // (one branch, not one per load: 1 % of the calls of five to 16 tokens)
        if (TILED || stream) weights(std::integral_constant<int, 2>{});
        else weights(std::integral_constant<int, 0>{});
        if constexpr (!XL) {
            x_rsrc = xr;
            x_voff = xv;
            x_kb = kb;
        }
        l_kb += 4;
        if (++l_i == l_n) {
            l_item += stride;
            if (l_item < total) open();
        }
    };

    auto request_x = [&](int g, bool last) {  // piece g of the last block requested, or of the one before it
        const uint32_t at = FEW ? 256u * (g >> 2) + 16u * (g & 3) : 64u * g;
        xq[FEW ? g : g & 3] = last ? __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, x_voff, x_kb * 512u + at, 0)
                                   : __builtin_amdgcn_raw_buffer_load_b128(x_rsrc0, x_voff0, x_kb0 * 512u + at, 0);
    };

    bf16x8 bias;
    {
        const u32x4 v = {0xBC80BC80u, 0xBC80BC80u, 0xBC80BC80u, 0xBC80BC80u};  // -8 / 2^9
        __builtin_memcpy(&bias, &v, 16);
    }
    // ---- the summing side
    int c_item = begin, c_i = 0, c_n = 0, par = 0;
    constexpr int NC = FEW ? 1 : 4;
    f32x4 acc[RB][NC];  // [row block][scale group modulo 4]; at most four rows: [row block][0], the lane's groups
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int t = 0; t < NC; ++t) acc[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto finish = [&]() {
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            f32x4 v;
            if constexpr (FEW) {  // the four lane groups' sums meet, (0 + 1) + (2 + 3) as below
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t a = __float_as_uint(acc[b][0][e]);
                    const u32x2 h = __builtin_amdgcn_permlane16_swap(a, a, false, false);
                    const uint32_t c = __float_as_uint(__uint_as_float(h.x) + __uint_as_float(h.y));
                    const u32x2 q = __builtin_amdgcn_permlane32_swap(c, c, false, false);
                    v[e] = __uint_as_float(q.x) + __uint_as_float(q.y);
                }
            } else {
                v = (acc[b][0] + acc[b][1 % NC]) + (acc[b][2 % NC] + acc[b][3 % NC]);
            }
            s_red[par][wave][b][lane] = v;
#pragma unroll
            for (int t = 0; t < NC; ++t) acc[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        // the bare barrier instruction: __syncthreads() would also wait for every load in flight.  Two buffers: the next
        // item's sums go to the other one, and nobody writes to this one again before the barrier of that item.
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int en = c_item / per, rem = c_item % per, nt = rem % ntn, split = rem / ntn;
        const int m = tid >> 4, n = tid & 15, src = 16 * (m >> 2) + n;
        float v[RB];
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            v[b] = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) v[b] += reinterpret_cast<const float *>(&s_red[par][w][b][src])[m & 3];
            v[b] *= 512.f;  // 2^9
        }
        if (m < s_ent[en].rows) {
            if (MODE == 1) {
                uint16_t *const y = reinterpret_cast<uint16_t *>(s_ent[en].y) + (size_t)m * N + nt * 16 + n;
                *y = (uint16_t)f32_to_bf16_bits(v[0] / (1.f + __expf(-v[0])) * v[1]);
            } else {
                float *const y = reinterpret_cast<float *>(s_ent[en].y) + split * split_stride + (size_t)m * N + nt * 32 + n;
#pragma unroll
                for (int b = 0; b < RB; ++b) y[16 * b] = v[b];
            }
        }
        par ^= 1;
    };
    // XL: the rows of an item's expert, the item's k, in operand order; rows without a token read a block of zeros
    extern __shared__ __attribute__((aligned(16))) uint8_t s_x[];
    int x_en = -1, x_split = -1, x_first = 0, x_last = 0;
    uint32_t x_base = 0, x_mask = 0;
    auto stage = [&]() {
        const int en = c_item / per, split = c_item % per / ntn;
        if (en == x_en && split == x_split) return;
        x_en = en;
        x_split = split;
        x_first = first_block(split);
        const int span = first_block(split + 1) - x_first, rows = s_ent[en].rows, pitch = span * 512 + 16;
        x_last = span - 1;
        const uint8_t *const src = reinterpret_cast<const uint8_t *>(s_ent[en].x) + (size_t)x_first * 512;
        for (int p = tid; p < rows * span * 32; p += 256) {
            const int m = p / (span * 32), c = p % (span * 32);
            const u32x4 v = *reinterpret_cast<const u32x4 *>(src + s_xoff[en][m] + c * 16);
            const uint32_t a[4] = {v.x, v.y, v.z, v.w};
            uint32_t o[4];
            order_x8(a, o);
            *reinterpret_cast<u32x4 *>(s_x + 512 + m * pitch + c * 16) = u32x4{o[0], o[1], o[2], o[3]};
        }
        if (tid < 32) *reinterpret_cast<u32x4 *>(s_x + tid * 16) = u32x4{0, 0, 0, 0};
        const bool mine = FEW ? (r >> 2) == j && (r & 3) < rows : r < rows;
        x_base = FEW ? (mine ? 512u + (r & 3) * pitch + 64u * j : 0u) : (mine ? 512u + r * pitch : 0u) + 16u * j;
        x_mask = mine ? ~0u : 0u;
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto consume = [&](Block &q) {  // false after the workgroup's last item
        uint32_t xa = 0;
        if constexpr (XL) {
            if (c_i == 0) stage();
            const int kb = c_i * 4 + wave;  // (a block past the end: its weights and scales are zeros)
            xa = x_base + ((uint32_t)(kb < x_last ? kb : x_last) * 512u & x_mask);
        }
        if (!TILED) {  // the two loads trade halves: [h] then holds groups 4h .. 4h+3 of rows 0..15
#pragma unroll
            for (int b = 0; b < RB; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int lo = (int)q.w[b][0][e], hi = (int)q.w[b][1][e];
                    q.w[b][0][e] = (uint32_t)__builtin_amdgcn_update_dpp(lo, hi, 0x128, 0xF, 0xC, false);  // row_ror 8 into lanes 8..15
                    q.w[b][1][e] = (uint32_t)__builtin_amdgcn_update_dpp(hi, lo, 0x128, 0xF, 0x3, false);  // ... into lanes 0..7
                }
        }
        auto operand = [&](int g, int at) {  // piece g of the block's activations (`at`: its place in LDS)
            bf16x8 av;
            if constexpr (XL) {
                av = *reinterpret_cast<const bf16x8 *>(s_x + xa + at);
            } else {
                const u32x4 v = xq[FEW ? g : g & 3];
                const uint32_t a[4] = {v.x, v.y, v.z, v.w};
                uint32_t o[4];
                order_x8(a, o);
                __builtin_memcpy(&av, o, 16);
            }
            return av;
        };
        if constexpr (FEW) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                bf16x8 av[4];
                f32x4 d[RB] = {};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    av[e] = operand(4 * h + e, 256 * h + 16 * e);
                    d[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[e], bias, d[0], 0, 0, 0);
                }
#pragma unroll
                for (int b = 1; b < RB; ++b) d[b] = d[0];
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int b = 0; b < RB; ++b) {
                        uint32_t p[4];
                        unpack8_fp8(q.w[b][h][e], p);
                        bf16x8 bv;
                        __builtin_memcpy(&bv, p, 16);
                        d[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[e], bv, d[b], 0, 0, 0);
                    }
#pragma unroll
                for (int b = 0; b < RB; ++b) {  // the lane's group: 4h + j
                    const u32x4 s = q.s[b];
                    const uint32_t sw = TILED ? (j & 1 ? s[2 + h] : s[h]) : (j & 2 ? s[2 * h + 1] : s[2 * h]);
                    acc[b][0] += d[b] * f16_bits_to_f32((uint16_t)(sw >> ((TILED ? j >> 1 : j & 1) * 16)));
                }
                if constexpr (!XL)
#pragma unroll
                    for (int e = 0; e < 4; ++e) request_x(4 * h + e, true);
            }
        } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t word[RB][4];  // [row block][group]
#pragma unroll
            for (int b = 0; b < RB; ++b) {
                const u32x4 w = q.w[b][h];
                const u32x2 lo = __builtin_amdgcn_permlane16_swap(w.x, w.y, false, false);
                const u32x2 hi = __builtin_amdgcn_permlane16_swap(w.z, w.w, false, false);
                const u32x2 g02 = __builtin_amdgcn_permlane32_swap(lo.x, hi.x, false, false);
                const u32x2 g13 = __builtin_amdgcn_permlane32_swap(lo.y, hi.y, false, false);
                word[b][0] = g02.x;
                word[b][1] = g13.x;
                word[b][2] = g02.y;
                word[b][3] = g13.y;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bf16x8 av = operand(4 * h + t, 64 * (4 * h + t));
                if constexpr (!XL) request_x(4 * (h ^ 1) + t, h == 1);
                const f32x4 d0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bias, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    uint32_t p[4];
                    unpack8_fp8(word[b][t], p);
                    bf16x8 bv;
                    __builtin_memcpy(&bv, p, 16);
                    const f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, d0, 0, 0, 0);
                    const uint32_t sw = q.s[b][TILED ? 2 * (t & 1) + h : 2 * h + (t >> 1)];  // group 4h + t
                    acc[b][t] += d * f16_bits_to_f32((uint16_t)((TILED ? t >> 1 : t & 1) ? sw >> 16 : sw & 0xFFFFu));
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // (else the halves' words are all in registers at once, more than there are)
        }
        }
        if (++c_i == c_n) {
            finish();
            c_i = 0;
            c_item += stride;
            if (c_item >= total) return false;
            c_n = blocks_of(c_item);
        }
        return true;
    };
    if (l_item >= total) return;
    open();
    c_n = l_n;
    if constexpr (XL && FEW) {
        Block q0, q1, q2;
        request(q0);
        request(q1);
        for (;;) {
            request(q2);
            if (!consume(q0)) break;
            request(q0);
            if (!consume(q1)) break;
            request(q1);
            if (!consume(q2)) break;
        }
    } else {
        Block q0, q1;
        request(q0);
        if constexpr (!XL) {
#pragma unroll
            for (int g = 0; g < (FEW ? 8 : 4); ++g) request_x(g, true);
        }
        for (;;) {
            request(q1);
            if (!consume(q0)) break;
            request(q0);
            if (!consume(q1)) break;
        }
    }
}

// T <= 16: no expert gets more than one tile of rows.  32-bit byte offsets into a matrix.  Row order: always (whole calls
// of 1 to 16 tokens on thirteen expert layers, 7 to 1500 MB: 1.01 to 2.6 times as fast as on the many-row kernel).
// In tile order the many-row kernel streams large experts better but has a launch more and coarser tiles, which is what few
// bytes take.  Whole calls there, many-row / this kernel in us, by the experts' bytes hit (at most) and the tokens:
//     7 MB  1 token  29.3 / 17.5    27 MB  1  40.8 / 24.2    27 MB 16  31.4 / 23.5    54 MB  1  49.8 / 31.1    54 MB  4  38.2 / 30.6
//   108 MB  1 token  60.7 / 42.2   108 MB  2  50.7 / 36.5   108 MB  4  42.0 / 37.7   108 MB 16  43.5 / 44.3
//   189 MB  1 token  76.2 / 63.1   216 MB  4  56.3 / 60.4   216 MB 16  65.2 / 75.6   378 MB 16  86.2 / 75.4   378 MB  1 103.8 / 107.7
//   756 MB  4 tokens 116.7 / 120.3  756 MB 16 153.0 / 185.5  1512 MB 16 280 / 352
// Up to 64 MB this kernel is ahead at every number of tokens; beyond 100 MB it depends on the tokens and the shape.
bool moe_few_ok(int T, int H, int F, int E, int top_k, bool tiled) {
    if (T > FEW_ROWS || E > FEW_ENTRIES || H % 256 != 0 || F % 256 != 0 || (int64_t)H * F / 2 >= (int64_t)kRange) return false;
    const int64_t hit = T * top_k < E ? T * top_k : E;
    return !tiled || hit * H * F * 27 / 16 <= (int64_t)64 << 20;  // three matrices of 9/16 byte per weight
}

int moe_few_tile_rows() { return FEW_ROWS; }

// K splits of the down product: items of at least four blocks of 256 k
int moe_few_down_splits(int F) { return F >= 4096 ? 4 : F >= 2048 ? 2 : 1; }

static int few_x_bytes(int T, int span) { return 512 + T * (span * 512 + 16); }

// `per` items per expert, `span` blocks of 256 k each.
// Activations through LDS from six items per workgroup on, or 32 blocks of 256 k (`items`: of all experts that T tokens hit on
// average, dealt to 768 workgroups).  Below, what a workgroup does first - wait for its rows, which it asks for behind its first weights,
// order them, meet at a barrier - costs more than the reads of each item that it saves, and its neighbouring items can be one more than
// another workgroup's.  Whole calls, us, that way / the other: rows, 2 tokens, 8 experts of 2304 x 1536, top 1 28.1 / 21.2; tiles, 14 tokens, 4 of
// 1280 x 4352 39.8 / 32.5; rows, 5 tokens, 8 of 3328 x 10496 (5 items of 13 blocks | 3 of 10) 113 / 127; tiles, 6 tokens, 8 of 256 x 12288 (7
// items of one block) 40 / 43.  Of 5300 calls of random sizes 164
// take it, 4 % faster on average and none more than 4 % slower than the other way.
bool moe_few_through_lds(int T, int E, int top_k, int per, int span) {
    float miss = 1.f;
    for (int t = 0; t < T; ++t) miss *= 1.f - (float)top_k / (float)E;
    const float items = (float)E * (1.f - miss) * (float)per / 768.f;
    return few_x_bytes(T, span) <= kXlBytes && (items >= 6.f || items * (float)span >= 32.f);
}

template <int MODE, bool TILED>
static int few_launch(const GemmGroup *groups, const int32_t *tiles, const int32_t *tok, int ntiles, int T, int E, int top_k, int N, int K,
                      int nsplit, size_t split_stride, hipStream_t st) {
    const int per = MODE == 1 ? N / 16 : N / 32 * nsplit;
    const int64_t most = (int64_t)ntiles * per;
    const int span = (K / 256 + nsplit - 1) / nsplit, x_bytes = few_x_bytes(T, span);
    const dim3 grid(most < 768 ? (int)most : 768);
    const int stream = (int64_t)E * N * K * 27 / 16 > (int64_t)400 << 20;  // all experts' bytes
    const bool lds = moe_few_through_lds(T, E, top_k, per, span);
#define CHADQ_FEW(XL, FEW)                                                                                                                        \
    hipLaunchKernelGGL((moe_few_i4g32_kernel<MODE, TILED, XL, FEW>), grid, dim3(256), XL ? x_bytes : 0, st, groups, tiles, tok, ntiles, E, N, K, \
                       nsplit, stream, split_stride)
    if (T <= 4) {
        if (lds) CHADQ_FEW(true, true);
        else CHADQ_FEW(false, true);
    } else {
        if (lds) CHADQ_FEW(true, false);
        else CHADQ_FEW(false, false);
    }
#undef CHADQ_FEW
    return hip_check(hipGetLastError(), "moe_few launch");
}

// gate/up with the SiLU gate: h bf16 [P,F] through the down descriptors' x pointers
int moe_few_gateup(const GemmGroup *groups, const int32_t *tiles, const int32_t *tok, int ntiles, int T, int E, int top_k, int F, int H, bool tiled,
                   hipStream_t st) {
    return tiled ? few_launch<1, true>(groups, tiles, tok, ntiles, T, E, top_k, F, H, 1, 0, st) : few_launch<1, false>(groups, tiles, tok, ntiles, T, E, top_k, F, H, 1, 0, st);
}

// down: fp32 parts [nsplit][P,H]
int moe_few_down(const GemmGroup *groups, const int32_t *tiles, int ntiles, int T, int E, int top_k, int H, int F, int nsplit, size_t split_stride, bool tiled,
                 hipStream_t st) {
    return tiled ? few_launch<0, true>(groups, tiles, nullptr, ntiles, T, E, top_k, H, F, nsplit, split_stride, st)
                 : few_launch<0, false>(groups, tiles, nullptr, ntiles, T, E, top_k, H, F, nsplit, split_stride, st);
}

}  // namespace chadq
