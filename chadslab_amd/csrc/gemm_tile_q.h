// The dequant-GEMM of gemm_tile_q.hip: launch functions and the tile choice.
#pragma once
#include "chadq_common.h"

namespace chadq {
namespace tileq {
enum { EPI_BF16 = 0, EPI_F32 = 1, EPI_GEGLU = 2 };
}

bool gemm_tile_q_ok(int K);
// y bf16 [M,N]; big: 256 x 256 tiles, else 128 x 128
int gemm_tile_i4g32_launch(const uint16_t *x, const uint8_t *wp, const uint16_t *sc, uint16_t *y, int M, int N, int K, bool big, hipStream_t st);
int gemm_tile_i8row_launch(const uint16_t *x, const int8_t *w8, const float *sc, uint16_t *y, int M, int N, int K, bool big, hipStream_t st);

}  // namespace chadq
