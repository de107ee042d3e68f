// gemm_f32.h -- the f32-accurate prompt GEMM (gemm_f32.hip) behind the
// quantized GEMM entry points of q4k_gemm.hip.
#pragma once

#include "common.h"

namespace doe {

struct GemmF32Args {
    const float *a;       // f32 [m][k]
    const float *norm_w;  // RMSNorm of a's rows first, or NULL
    float norm_eps;
    int norm_offset;
    const void *b;  // row-wise Q4_K (fmt 0) or Q8_0 (fmt 1) weights
    int fmt;
    float *c;               // f32 [m][n]; pairs: [m][n / 2]
    const float *residual;  // c = the product + residual (may be c), or NULL; splits == 1 only
    bool pairs;             // GeGLU over columns (2j, 2j + 1); splits == 1 only
    float *part;            // splits > 1: the K splits' partial products [splits][m][n]
    int64_t m, n, k;
};

// How a product of this shape runs: its K splits and the bytes of workspace
// its f16 copy of A takes (16-byte aligned, in front of the partials).
struct GemmF32Plan {
    int tile_rows;  // 64 or 128 (x 128 columns)
    int64_t splits, chunks_per_split, a_bytes;
};
GemmF32Plan gemm_f32_plan(int64_t m, int64_t n, int64_t k, int fmt, int num_cus);
int gemm_f32_launch(const GemmF32Args &g, const GemmF32Plan &plan, void *workspace, hipStream_t st);

}  // namespace doe
