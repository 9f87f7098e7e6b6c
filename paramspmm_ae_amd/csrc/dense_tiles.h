// Operand layouts that the tall-skinny dense products share (dense_atb.hip, dense_xw.hip, dense_grad.hip).
#pragma once
#include "spmm_kernel.h"

// LDS row stride of a staged weight matrix with K2 columns: the four k-rows a contraction step reads fall into different
// bank halves
#define XWW_STRIDE(K2) (((K2) + 63) / 64 * 64 + 4)

typedef float psp_mfma_acc __attribute__((ext_vector_type(4)));

template <int V> __device__ __forceinline__ void psp_atb_load(const float *p, float *out)
{
    if (V == 4) {
        const psp_f32x4 x = *(const psp_f32x4 *)p;
        out[0] = x[0], out[1] = x[1], out[2] = x[2], out[3] = x[3];
    } else if (V == 3) {
        typedef float f32x3 __attribute__((ext_vector_type(3), aligned(4)));
        const f32x3 x = *(const f32x3 *)p;
        out[0] = x[0], out[1] = x[1], out[2] = x[2];
    } else if (V == 2) {
        const psp_f32x2 x = *(const psp_f32x2 *)p;
        out[0] = x[0], out[1] = x[1];
    } else {
        out[0] = *p;
    }
}
// R tiles are loaded in pieces of four (16 bytes per lane) and a last one of R % 4: column that index i of tile m stands for
template <int R> __device__ __forceinline__ int psp_atb_col(int m, int i)
{
    constexpr int N4 = R / 4 * 4, REM = R % 4;
    return m < N4 ? (m / 4) * 64 + 4 * i + m % 4 : N4 * 16 + REM * i + (m - N4);
}
template <int R> __device__ __forceinline__ void psp_atb_load_row(const float *row, int c, float (&out)[R])
{
    constexpr int N4 = R / 4 * 4, REM = R % 4;
#pragma unroll
    for (int m = 0; m < N4; m += 4) psp_atb_load<4>(row + m * 16 + 4 * c, out + m);
    if constexpr (REM > 0) psp_atb_load<REM>(row + N4 * 16 + REM * c, out + N4);
}
