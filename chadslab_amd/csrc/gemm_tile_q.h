// The dequant-GEMM of gemm_tile_q.hip: launch functions and the tile choice.
#pragma once
#include "chadq_common.h"

namespace chadq {
namespace tileq {
enum { EPI_BF16 = 0, EPI_F32 = 1, EPI_GEGLU = 2, EPI_QKV = 3 };
}

bool gemm_tile_q_ok(int K);
enum GemmTile { TILE_32x64, TILE_64x64, TILE_96x64, TILE_128x64, TILE_96x128, TILE_128x128, TILE_192x128, TILE_256x128, TILE_256x256,
                SHORT_32x64, SHORT_64x64, SHORT_128x128, SHORT_256x256 };
// the tile (activation rows x weight rows) that takes the product in the shortest time; guard: K no multiple of the tiles' steps, or int4
// scales that are not 16-byte aligned
GemmTile gemm_tile_pick(int M, int N, int K, bool int4, bool guard);
// y bf16 [M,N]; gemm_tile_q_ok(K)
int gemm_tile_i4g32_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, uint16_t *y, int M, int N, int K, GemmTile tile, hipStream_t st);
int gemm_tile_i8row_launch(const uint16_t *x, const int8_t *w8, const float *sc, uint16_t *y, int M, int N, int K, GemmTile tile, hipStream_t st);
// K parts (1: none) in which a product of few tiles and a long K is the quicker one, their k (np * span >= K, none is empty) and tile; the parts
// (fp32 [np][M,N], at `parts`) added to y
int gemm_split_parts(int M, int N, int K, bool int4, GemmTile *tile, int *span);
int gemm_tile_parts_launch(const uint16_t *x, const uint8_t *w, const void *sc, uint16_t *y, int M, int N, int K, bool int4, bool guard, GemmTile tile, int np,
                           int span, float *parts, hipStream_t st);
// int4 weights taken exactly (nothing rounded before the fp32 sums); K % 256 == 0, x, wp and sc 16-byte aligned unless it says otherwise
// The activations of a prompt's products (not those of gemm_exact_few_rows_launch) carry this factor, and the gated one's result carries it too: the
// operands are (u - 8) / 2^4, and with it no group's sum overflows while the activations are finite.  The factor is exact for bf16 activations of
// 2^-121 and more; smaller ones lose up to five bits.
constexpr float kExactX = 0x1p-5f;
constexpr int kExactMaxSplits = 8;
int gemm_exact_splits(int M, int N, int K);  // K splits to use for gemm_exact_scaled_f32_launch
// rows (and *columns) of the tile that the f32 and geglu launches below take for `parts` K splits of `per` 256-k blocks; *us: what the launch takes
int gemm_exact_tile(int M, int N, int per, int parts, bool geglu, float *us, int *columns);
// y_parts fp32 [ksplit][M,N]
int gemm_exact_scaled_f32_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, float *y_parts, int M, int N, int K, int ksplit,
                                 hipStream_t st);
// weight rows in (gate, up) pairs: h[m,i] = bf16(gelu_tanh(y[m,2i]) * y[m,2i+1] * kExactX), [M, N/2]
int gemm_exact_scaled_geglu_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, uint16_t *h, int M, int N, int K, hipStream_t st);
// The product of a prompt's M tokens with [q heads | k | v] (hq + 2 heads of dh, in whole K): q and k rotated at positions pos + m (table as
// chadq_rope_table writes it), q fp32 [M][hq*dh], k and v as bf16 rows pos + m of the caches.
struct QkvOut {
    const float *table;
    float *q;
    uint16_t *kc, *vc;
    int hq, dh, pos;
};
bool gemm_exact_qkv_pays(int M, int N, int K);  // against the plain product and a launch for the rest
int gemm_exact_qkv_tile(int M, int N, int K);   // rows of its tile (64 columns)
int gemm_exact_qkv_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, const QkvOut &out, int M, int K, hipStream_t st);
// y [M,N] fp32 or bf16, at most 32 rows, any K % 32 == 0 with gemm_tile_q_ok(K), any alignment of the scales, plain activations
int gemm_exact_few_rows_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, float *y, int M, int N, int K, bool bf16_out,
                               hipStream_t st);

}  // namespace chadq
