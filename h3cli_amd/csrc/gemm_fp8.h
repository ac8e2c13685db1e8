// The FP8 projection GEMM (gemm_fp8.hip) as quant.hip launches it.
#pragma once
#include "gemm.h"

struct Fp8GemmArgs {
    uint16_t *y;
    const uint8_t *x, *w;     // E4M3 codes [m, k], [n, k]
    const float *sx, *sw;     // device scalars: activation and weight scales
    unsigned m, n, k;
    TileSplit tile;           // set by h3_gemm_fp8
};
int h3_gemm_fp8(h3_gpu *g, Fp8GemmArgs a);
