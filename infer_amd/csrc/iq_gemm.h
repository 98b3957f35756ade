// iq_gemm.h -- the wide-tile prefill GEMM (iq_gemmw.hip) as launch_gemm
// (iq_gemm.hip) calls it.
#pragma once

#include "iq_internal.h"
#include "iq_plan.h"

namespace iq {

struct GemmwParams {
    const uint16_t* a;   // [T][K] bf16, or the prepared fp16 hi part
    const uint16_t* al;  // [T][K] prepared fp16 lo part, or null (bf16)
    const float* rs;     // [T] row factors of the prepared operands, or null
    const uint8_t* q;
    const uint16_t* scales;
    const uint8_t* zeros;
    const uint16_t* bias;
    float* y;
    float* part;         // [splits][split tiles][bm][256] fp32 range sums
    int64_t T, N, K, G;
    int tiles_m, tiles_n;
    int full;            // tiles done whole
    int splits, gch;     // K ranges of the others, groups per range
};

// The wide-tile GEMM with the tiles and K ranges of pl (gemmw_choose).
hipError_t launch_gemmw(GemmwParams p, int kind, const GemmwPlan& pl, hipStream_t stream);

}  // namespace iq
