// Many-row products of quantized weights that are unpacked into scratch memory first (e2h_unpacked_gemm.hip).
#pragma once

#include "e2h_common.h"

namespace e2h {

int64_t int8_unpacked_bytes(int64_t M, int64_t N, int64_t K);  // scratch; 0: the shape is not for this form
int int8_unpacked_gemm(const uint16_t *x, const int8_t *q, const uint16_t *scales, uint16_t *y, int M, int N, int K, uint16_t *w, hipStream_t stream);

}  // namespace e2h
