// A prompt through the Gemma-2B-shaped decoder: T tokens at once through every layer, filling the KV caches.  One token
// at a time, as the decode step runs it, every token streams all of the weights (1.2 GB over 18 layers, 0.5 ms); here a
// layer's weights are read once per chunk of tokens and the products run on the matrix cores.
//
// Nothing is rounded that the decode step does not round: activations become bf16 in the same four places (the two norms,
// the attention vector, the gated activation), weights are taken exactly (gemm_tile_q.hip, EXACT), sums, residual stream,
// rotation and softmax are fp32, K and V rows bf16.
//
// Per layer: residual add + RMSNorm | qkv product | rotation and cache rows, by a launch of their own where the
// product is split over K, else in its epilogue | attention | output product | residual add +
// RMSNorm | gate/up product with the GeGLU in its epilogue | down product.  Products with few tiles are split over K; the
// kernel that consumes them adds the parts, in order.  In the last layer everything behind the cache rows runs for the last
// token only: nothing else of it is ever read.
#include "chadq_common.h"
#include "gemm_tile_q.h"

namespace chadq {

// x[t] = row tokens[t] of the int4 table [V, d] (clamped into it); eight weights per thread and round, d % 32 == 0
__global__ __launch_bounds__(256) void prompt_embed_kernel(const int32_t *__restrict__ tokens, const uint8_t *__restrict__ wp,
                                                           const uint16_t *__restrict__ sc, float *__restrict__ x, int d, int V) {
    const int t = min(max(tokens[blockIdx.x], 0), V - 1);
    const uint8_t *row = wp + (size_t)t * (d / 2);
    const uint16_t *srow = sc + (size_t)t * (d / 32);
    float *const xo = x + (size_t)blockIdx.x * d;
    for (int k8 = threadIdx.x; k8 < (d >> 3); k8 += 256) {
        const uint32_t w = *reinterpret_cast<const uint32_t *>(row + 4 * k8);
        const float s = f16_bits_to_f32(srow[k8 >> 2]);
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (float)((int)((w >> (4 * e)) & 15u) - 8) * s;
        *reinterpret_cast<f32x4 *>(xo + 8 * k8) = f32x4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4 *>(xo + 8 * k8 + 4) = f32x4{v[4], v[5], v[6], v[7]};
    }
}

// One row per workgroup: r = res + the np parts (part p of row t at parts + (p * rows + t) * d, added in order), kept in
// res_out if there were any (may be res), then, if y, y = bf16(r / sqrt(mean(r^2) + eps) * w * kExactX).  d % 4 == 0, d <= 2048.
// NP: the number of parts, so that every load is in flight before the first sum (one memory round trip, not np of them).
template <int NP>
__global__ __launch_bounds__(256) void prompt_add_norm_kernel(const float *res, float *res_out, const float *__restrict__ parts,
                                                              const float *__restrict__ w, uint16_t *__restrict__ y, int d, float eps) {
    __shared__ float s_ss[4];
    const int tid = threadIdx.x, nv = d >> 2, rows = gridDim.x;
    const f32x4 *const r4 = reinterpret_cast<const f32x4 *>(res + (size_t)blockIdx.x * d);
    f32x4 *const o4 = reinterpret_cast<f32x4 *>(res_out + (size_t)blockIdx.x * d);
    f32x4 r[2], wv[2], pv[2][NP > 0 ? NP : 1];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int i = tid + 256 * j, ii = i < nv ? i : 0;
        r[j] = r4[ii];
        wv[j] = y ? reinterpret_cast<const f32x4 *>(w)[ii] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < NP; ++p) pv[j][p] = reinterpret_cast<const f32x4 *>(parts + ((size_t)p * rows + blockIdx.x) * d)[ii];
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int i = tid + 256 * j;
#pragma unroll
        for (int p = 0; p < NP; ++p) r[j] += pv[j][p];
        if (i < nv) {
            if (NP > 0) o4[i] = r[j];
            ss += r[j].x * r[j].x + r[j].y * r[j].y + r[j].z * r[j].z + r[j].w * r[j].w;
        }
    }
    if (!y) return;
    ss = wave_sum_to_lane63(ss);
    if ((tid & 63) == 63) s_ss[tid >> 6] = ss;
    __syncthreads();
    const float rinv = rsqrtf((s_ss[0] + s_ss[1] + s_ss[2] + s_ss[3]) / (float)d + eps);
    auto bits = [](float v) { return f32_to_bf16_bits(v * kExactX); };
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int i = tid + 256 * j;
        if (i < nv) {
            const uint32_t lo = bits(r[j].x * rinv * wv[j].x) | (bits(r[j].y * rinv * wv[j].y) << 16);
            const uint32_t hi = bits(r[j].z * rinv * wv[j].z) | (bits(r[j].w * rinv * wv[j].w) << 16);
            reinterpret_cast<u32x2 *>(y + (size_t)blockIdx.x * d)[i] = u32x2{lo, hi};
        }
    }
}

static void add_norm_launch(int rows, const float *res, float *res_out, const float *parts, int np, const float *w, uint16_t *y, int d,
                            float eps, hipStream_t st) {
#define CHADQ_ADD_NORM(NP) hipLaunchKernelGGL(prompt_add_norm_kernel<NP>, dim3(rows), dim3(256), 0, st, res, res_out, parts, w, y, d, eps)
    switch (np) {  // at most kExactMaxSplits
        case 0: CHADQ_ADD_NORM(0); break;
        case 1: CHADQ_ADD_NORM(1); break;
        case 2: CHADQ_ADD_NORM(2); break;
        case 3: CHADQ_ADD_NORM(3); break;
        case 4: CHADQ_ADD_NORM(4); break;
        case 5: CHADQ_ADD_NORM(5); break;
        case 6: CHADQ_ADD_NORM(6); break;
        case 7: CHADQ_ADD_NORM(7); break;
        default: CHADQ_ADD_NORM(8); break;
    }
#undef CHADQ_ADD_NORM
}
static_assert(kExactMaxSplits == 8, "add_norm_launch and the rotation know up to eight parts");

// Workgroup (t, head): the np parts of a head of row t of qkv ([hq*dh | dh | dh]) summed; q and k (head hq) rotated at
// position pos + t (rope table as chadq_rope_table writes it), q to q_out fp32 [T][hq*dh], k and v (head hq + 1) to row
// pos + t of the caches.  One thread per rotation pair, all of its loads in flight together: 128 >= dh / 2 threads.
__global__ __launch_bounds__(128) void prompt_rope_kernel(const float *__restrict__ qkv, int np, const float *__restrict__ table,
                                                          float *__restrict__ q_out, uint16_t *__restrict__ kc,
                                                          uint16_t *__restrict__ vc, int hq, int dh, int pos) {
    const int t = blockIdx.x, head = blockIdx.y, T = gridDim.x, half = dh >> 1, j = threadIdx.x;
    if (j >= half) return;
    const size_t p = (size_t)(pos + t), stride = (size_t)T * (hq + 2) * dh;
    const float *const src = qkv + (size_t)t * (hq + 2) * dh + (size_t)head * dh + j;
    float av[kExactMaxSplits], bv[kExactMaxSplits];
#pragma unroll
    for (int s = 0; s < kExactMaxSplits; ++s)
        if (s < np) {
            av[s] = src[s * stride];
            bv[s] = src[s * stride + half];
        }
    const float cs = table[(p * half + j) * 2], sn = table[(p * half + j) * 2 + 1];
    float a = av[0], b = bv[0];
#pragma unroll
    for (int s = 1; s < kExactMaxSplits; ++s)
        if (s < np) {
            a += av[s];
            b += bv[s];
        }
    const float ra = a * cs - b * sn, rb = b * cs + a * sn;
    if (head < hq) {
        float *const o = q_out + ((size_t)t * hq + head) * dh + j;
        o[0] = ra;
        o[half] = rb;
    } else if (head == hq) {
        kc[p * dh + j] = (uint16_t)f32_to_bf16_bits(ra);
        kc[p * dh + j + half] = (uint16_t)f32_to_bf16_bits(rb);
    } else {
        vc[p * dh + j] = (uint16_t)f32_to_bf16_bits(a);
        vc[p * dh + j + half] = (uint16_t)f32_to_bf16_bits(b);
    }
}

// Causal multi-query attention of T new tokens at positions pos .. pos+T-1 over the cache rows 0 .. pos+T-1.
// Rows of work: r = t * hq + h (one K/V head serves every row).  A workgroup takes 16 rows, its four waves the blocks of
// 32 positions in turn, each with a running maximum, sum and output of its own (no barrier in the loop); they meet once
// at the end.  128 workgroups at 256 tokens of 8 heads, and a wave's blocks at a context of 256 are two: launch and
// memory latency bound it, which is why a workgroup takes no more rows.
// Both products on v_mfma_f32_16x16x32_bf16 with the fp32 side (q, then the probabilities) as two bf16 operands:
//   scores  A = q, B = K rows as they lie in the cache (16 bytes per lane).  D: lane (position = lane % 16, g) holds rows
//           4g .. 4g+3.
//   output  A = the probabilities, through a small LDS tile into row order; B = V[8g .. 8g+7][column]: a lane loads 8
//           positions x 8 columns, transposes them with 32 byte permutes and leaves 16-byte operands in LDS
//           ([g][column]; the place of a column inside its group of eight is XORed with the group, so that neither the
//           stores, one column of many groups, nor the loads, 16 columns, meet in the same banks).
// The rows of a workgroup belong to one to sixteen tokens and share the V operands: a position that the later ones see and
// the earlier ones must not goes in like any other while its V row is finite (its probability is 0 for those), and apart,
// row by row, if it is not.
template <int DH>
__global__ __launch_bounds__(256) void prompt_attn_kernel(const float *__restrict__ q, const uint16_t *__restrict__ kc,
                                                          const uint16_t *__restrict__ vc, uint16_t *__restrict__ out, int T,
                                                          int pos, int hq) {
    constexpr int ST = DH / 32, CB = DH / 16, CG = DH / 8, PP = 36;
    __shared__ __attribute__((aligned(16))) uint8_t s_v[4][DH * 64];    // V operands of a wave's block; at the end its output
    __shared__ __attribute__((aligned(16))) float s_p[4][16 * PP];
    __shared__ float s_m[4][16], s_l[4][16];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, g = lane >> 4;
    const int r0 = blockIdx.x * 16, total = T * hq;
    const int t_last = min(r0 + 15, total - 1) / hq;
    const int nctx = pos + t_last + 1, nblk = (nctx + 31) >> 5;
    const int seen = pos + r0 / hq + 1;  // every row of the workgroup sees the positions below, only some those from here on

    int lim[4];  // first position row 4g+e may not see
#pragma unroll
    for (int e = 0; e < 4; ++e) lim[e] = pos + min(r0 + 4 * g + e, total - 1) / hq + 1;
    const float scale = rsqrtf((float)DH);
    float m[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY}, l[4] = {0.f, 0.f, 0.f, 0.f};
    f32x4 o[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint8_t *const sv = s_v[wave];
    float *const sp = s_p[wave];

    // A wave's next K and V rows are requested as soon as the registers that hold the current ones are free.
    u32x4 kv[2][ST];
    auto load_k = [&](int b) {
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            const uint16_t *kr = kc + (size_t)min(b * 32 + 16 * blk + li, nctx - 1) * DH + 8 * g;
#pragma unroll
            for (int s = 0; s < ST; ++s) kv[blk][s] = *reinterpret_cast<const u32x4 *>(kr + 32 * s);
        }
    };
    constexpr int NT = (4 * CG + 63) / 64;  // V: task (gq, cg) = positions 8gq..+7, columns 8cg..+7
    const bool vlive = 4 * CG % 64 == 0 || lane < 4 * CG;
    u32x4 vr[NT][8];
    auto load_v = [&](int b) {
#pragma unroll
        for (int it = 0; it < NT; ++it) {
            const int task = vlive ? it * 64 + lane : 0, gq = task / CG, cg = task % CG;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                vr[it][e] = *reinterpret_cast<const u32x4 *>(vc + (size_t)min(b * 32 + 8 * gq + e, nctx - 1) * DH + 8 * cg);
        }
    };
    if (wave < nblk) {
        load_v(wave);
        load_k(wave);
    }
    bf16x8 qh[ST], ql[ST];
    {
        const float *qr = q + (size_t)min(r0 + li, total - 1) * DH + 8 * g;
#pragma unroll
        for (int s = 0; s < ST; ++s)
            split_bf16x8(*reinterpret_cast<const f32x4 *>(qr + 32 * s), *reinterpret_cast<const f32x4 *>(qr + 32 * s + 4), qh[s], ql[s]);
    }
    for (int b = wave; b < nblk; b += 4) {
        const int p0 = b * 32;
        // Positions only some of the rows see in a block, one of them with a V row that is not finite: the others' probability 0
        // times it would be NaN.  (Packed maxima of the magnitudes, two instructions per word, of the words e that can hold
        // such a position: with 8 heads there is one position, an eighth of the block.  It does not show in the time of a call:
        // 256 tokens through 18 layers, 2881 us with and 2882 without.)
        bool apart = false;
        if (p0 + 32 > seen) {
            const int lo = max(seen - p0, 0), hi = min(nctx - p0, 32);
            u16x2 top[4] = {};
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (lo + ((e - lo) & 7) < hi)  // the first position from lo on that is e modulo 8
#pragma unroll
                    for (int it = 0; it < NT; ++it)
#pragma unroll
                        for (int k = 0; k < 4; ++k) top[k] = __builtin_elementwise_max(top[k], __builtin_bit_cast(u16x2, vr[it][e][k] & 0x7FFF7FFFu));
            top[0] = __builtin_elementwise_max(__builtin_elementwise_max(top[0], top[1]), __builtin_elementwise_max(top[2], top[3]));
            apart = __any(top[0].x >= 0x7F80 || top[0].y >= 0x7F80);
        }
        const int pz = apart ? seen : nctx;  // rows from here on (past the context, or to be added apart) become zeros
#pragma unroll
        for (int it = 0; it < NT; ++it) {
            const int task = it * 64 + lane, gq = task / CG, cg = task % CG;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (p0 + 8 * gq + e >= pz) vr[it][e] = u32x4{0, 0, 0, 0};
            if (vlive) {
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    u32x4 w;
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        w[k] = __builtin_amdgcn_perm(vr[it][2 * k + 1][c >> 1], vr[it][2 * k][c >> 1], (c & 1) ? 0x07060302u : 0x05040100u);
                    *reinterpret_cast<u32x4 *>(sv + (gq * DH + 8 * cg + (c ^ (cg & 7))) * 16) = w;
                }
            }
        }
        if (b + 4 < nblk) load_v(b + 4);
        f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int st = 0; st < ST; ++st)
#pragma unroll
            for (int blk = 0; blk < 2; ++blk) {
                bf16x8 kb;
                __builtin_memcpy(&kb, &kv[blk][st], 16);
                s[blk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qh[st], kb, s[blk], 0, 0, 0);
                s[blk] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ql[st], kb, s[blk], 0, 0, 0);
            }
        if (b + 4 < nblk) load_k(b + 4);
        float alpha[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float s0 = p0 + li < lim[e] ? s[0][e] * scale : -INFINITY, s1 = p0 + 16 + li < lim[e] ? s[1][e] * scale : -INFINITY;
            float mx = fmaxf(s0, s1);
            mx = fmaxf(mx, dpp_f32<0x128, 0xF>(mx));  // row_ror 8, 4, 2, 1: over the 16 lanes that hold the row
            mx = fmaxf(mx, dpp_f32<0x124, 0xF>(mx));
            mx = fmaxf(mx, dpp_f32<0x122, 0xF>(mx));
            mx = fmaxf(mx, dpp_f32<0x121, 0xF>(mx));
            const float mn = fmaxf(m[e], mx), ms = mn == -INFINITY ? 0.f : mn;  // a block none of which the row may see
            const float e0 = __expf(s0 - ms), e1 = __expf(s1 - ms);
            float sum = e0 + e1;
            sum += dpp_f32<0x128, 0xF>(sum);
            sum += dpp_f32<0x124, 0xF>(sum);
            sum += dpp_f32<0x122, 0xF>(sum);
            sum += dpp_f32<0x121, 0xF>(sum);
            alpha[e] = __expf(m[e] - ms);
            l[e] = l[e] * alpha[e] + sum;
            m[e] = mn;
            sp[(4 * g + e) * PP + li] = e0;
            sp[(4 * g + e) * PP + 16 + li] = e1;
        }
        // (one wave's own LDS: the compiler waits for the writes it depends on; no other wave is involved)
        __builtin_amdgcn_wave_barrier();
        bf16x8 ph, pl;
        split_bf16x8(*reinterpret_cast<const f32x4 *>(sp + li * PP + 8 * g), *reinterpret_cast<const f32x4 *>(sp + li * PP + 8 * g + 4), ph, pl);
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const int cg = 2 * c + (li >> 3);
            const bf16x8 vb = *reinterpret_cast<const bf16x8 *>(sv + (g * DH + 8 * cg + ((li & 7) ^ (cg & 7))) * 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[c][e] *= alpha[e];
            o[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph, vb, o[c], 0, 0, 0);
            o[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl, vb, o[c], 0, 0, 0);
        }
        if (__builtin_expect(apart, false)) {  // to the rows that see them, one position after the other
            for (int p = max(seen, p0); p < min(nctx, p0 + 32); ++p) {
                float pr[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) pr[e] = sp[(4 * g + e) * PP + p - p0];
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    const float v = bf16_bits_to_f32(vc[(size_t)p * DH + 16 * c + li]);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (p < lim[e]) o[c][e] = __builtin_fmaf(pr[e], v, o[c][e]);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    // the four waves' shares of every row meet
    if (li == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s_m[wave][4 * g + e] = m[e];
            s_l[wave][4 * g + e] = l[e];
        }
    }
    __syncthreads();
    float f[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int r = 4 * g + e;
        const float M = fmaxf(fmaxf(s_m[0][r], s_m[1][r]), fmaxf(s_m[2][r], s_m[3][r]));  // finite: position 0 is seen by every row
        f[e] = __expf(m[e] - M);
    }
    float *const so = reinterpret_cast<float *>(sv);  // [16 rows][DH]
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) so[(4 * g + e) * DH + 16 * c + li] = o[c][e] * f[e];
    __syncthreads();
    for (int i = tid; i < 16 * DH / 4; i += 256) {
        const int r = i / (DH / 4);
        if (r0 + r >= total) break;
        const float M = fmaxf(fmaxf(s_m[0][r], s_m[1][r]), fmaxf(s_m[2][r], s_m[3][r]));
        float den = 0.f;
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            den += __expf(s_m[w][r] - M) * s_l[w][r];
            v += reinterpret_cast<const f32x4 *>(s_v[w])[i];
        }
        auto bits = [&](float o) { return f32_to_bf16_bits(o / den * kExactX); };  // (for the exact product that reads them)
        const u32x2 ob = {bits(v.x) | (bits(v.y) << 16), bits(v.z) | (bits(v.w) << 16)};
        *reinterpret_cast<u32x2 *>(out + (size_t)r0 * DH + 4 * i) = ob;
    }
}

static int prompt_attn_launch(const float *q, const uint16_t *kc, const uint16_t *vc, uint16_t *out, int T, int pos, int hq, int dh,
                              hipStream_t st) {
    const dim3 grid((T * hq + 15) / 16);
    if (dh == 256) hipLaunchKernelGGL(prompt_attn_kernel<256>, grid, dim3(256), 0, st, q, kc, vc, out, T, pos, hq);
    else if (dh == 128) hipLaunchKernelGGL(prompt_attn_kernel<128>, grid, dim3(256), 0, st, q, kc, vc, out, T, pos, hq);
    else hipLaunchKernelGGL(prompt_attn_kernel<64>, grid, dim3(256), 0, st, q, kc, vc, out, T, pos, hq);
    return hip_check(hipGetLastError(), "prompt attention launch");
}

// ---- workspace: everything between the launches of one call
struct PromptWs {
    float *x, *parts, *q;  // residual stream [T,d]; the parts of whichever product came last; rotated q [T][hq*dh]
    uint16_t *xn, *h;      // normalised rows / attention vectors [T][max(d, hq*dh)]; gated activation [T][ffn]
};

static size_t prompt_layout(uint8_t *base, int T, int d, int hq, int dh, int ffn, PromptWs *ws) {
    size_t o = 0;
    auto take = [&](size_t bytes) {
        uint8_t *p = base ? base + o : nullptr;
        o += (bytes + 255) & ~(size_t)255;
        return p;
    };
    const size_t wq = (size_t)(hq + 2) * dh, t = (size_t)T;
    size_t parts = 0;  // floats
    auto need = [&](int M, int N, int K) {
        const size_t n = (size_t)gemm_exact_splits(M, N, K) * M * N;
        parts = n > parts ? n : parts;
    };
    // (every number of row tiles up to T: a shorter chunk may come with the same workspace, and fewer rows can take more splits)
    for (int M = 32; M < T + 64; M += M < 64 ? M : 64) {
        const int m = M < T ? M : T;
        need(m, (int)wq, d);
        need(m, d, hq * dh);
        need(m, d, ffn);
    }
    PromptWs w;
    w.x = (float *)take(t * d * 4);
    w.parts = (float *)take(parts * 4);
    w.q = (float *)take(t * hq * dh * 4);
    w.xn = (uint16_t *)take(t * (d > hq * dh ? d : hq * dh) * 2);
    w.h = (uint16_t *)take(t * ffn * 2);
    if (ws) *ws = w;
    return o;
}

bool prompt_i4g32_ok(int d, int hq, int dh, int ffn) {
    return d >= 256 && d <= 2048 && d % 256 == 0 && hq >= 1 && hq <= 64 && (dh == 64 || dh == 128 || dh == 256) && (hq * dh) % 256 == 0 &&
           ffn >= 256 && ffn % 256 == 0 && gemm_tile_q_ok(ffn) && gemm_tile_q_ok(hq * dh);
}

size_t prompt_i4g32_workspace_bytes(int T, int d, int hq, int dh, int ffn) { return prompt_layout(nullptr, T, d, hq, dh, ffn, nullptr); }

int prompt_i4g32_launch(const chadq_prompt_layer_i4g32 *layers, int n_layers, const int32_t *tokens, const uint8_t *emb,
                        const uint16_t *semb, int V, const float *rope_table, int T, int pos, int d, int hq, int dh, int ffn, float eps,
                        float *x_last, void *workspace, hipStream_t st) {
    PromptWs ws;
    prompt_layout(reinterpret_cast<uint8_t *>(workspace), T, d, hq, dh, ffn, &ws);
    const int wq = (hq + 2) * dh;
    const bool rotated = gemm_exact_qkv_pays(T, wq, d);  // q and k are, by the product's epilogue
    hipLaunchKernelGGL(prompt_embed_kernel, dim3(T), dim3(256), 0, st, tokens, emb, semb, ws.x, d, V);
    int np = 0, rc;  // parts pending for the residual stream
    int rows = T;
    float *x = ws.x;
#define CHADQ_STEP(call)          \
    do {                          \
        rc = (call);              \
        if (rc != 0) return rc;   \
    } while (0)
    for (int li = 0; li < n_layers; ++li) {
        const chadq_prompt_layer_i4g32 &L = layers[li];
        add_norm_launch(T, x, x, ws.parts, np, L.ln1, ws.xn, d, eps, st);
        if (rotated) {
            CHADQ_STEP(gemm_exact_qkv_launch(ws.xn, L.wqkv, L.sqkv, QkvOut{rope_table, ws.q, L.kcache, L.vcache, hq, dh, pos}, T, d, st));
        } else {
            np = gemm_exact_splits(T, wq, d);
            CHADQ_STEP(gemm_exact_scaled_f32_launch(ws.xn, L.wqkv, L.sqkv, ws.parts, T, wq, d, np, st));
            hipLaunchKernelGGL(prompt_rope_kernel, dim3(T, hq + 2), dim3(128), 0, st, ws.parts, np, rope_table, ws.q, L.kcache, L.vcache, hq, dh, pos);
        }
        const float *q = ws.q;
        if (li == n_layers - 1) {  // of the last layer only the last token goes on
            rows = 1;
            x = ws.x + (size_t)(T - 1) * d;
            q = ws.q + (size_t)(T - 1) * hq * dh;
        }
        CHADQ_STEP(prompt_attn_launch(q, L.kcache, L.vcache, ws.xn, rows, pos + T - rows, hq, dh, st));
        np = gemm_exact_splits(rows, d, hq * dh);
        CHADQ_STEP(gemm_exact_scaled_f32_launch(ws.xn, L.wo, L.so, ws.parts, rows, d, hq * dh, np, st));
        add_norm_launch(rows, x, x, ws.parts, np, L.ln2, ws.xn, d, eps, st);
        CHADQ_STEP(gemm_exact_scaled_geglu_launch(ws.xn, L.wgu, L.sgu, ws.h, rows, 2 * ffn, d, st));
        np = gemm_exact_splits(rows, d, ffn);
        CHADQ_STEP(gemm_exact_scaled_f32_launch(ws.h, L.wd, L.sd, ws.parts, rows, d, ffn, np, st));
    }
#undef CHADQ_STEP
    add_norm_launch(1, x, x_last, ws.parts, np, (const float *)nullptr, (uint16_t *)nullptr, d, eps, st);
    return hip_check(hipGetLastError(), "prompt launches");
}

}  // namespace chadq
