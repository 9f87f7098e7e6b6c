// Attention layer of gnn_conv.py:128-180 on the PCSR formats (CSR, 2x1 blocks, plain or row-split), one launch per direction:
// the SDDMM and the SpMM of a direction gather the same rows of the same matrix, so the SpMM walk forms the scores from the
// rows it gathers (psp_attention in spmm_kernel.h).  On the windowed layout attn_window.hip does the same.
//
// Bound by the gathers, of which there is one per stored entry and direction instead of two.  Lane groups cover the whole
// width: 4 / 8 / 16 lanes of one piece, from 68 columns on 16 lanes of two pieces.  Random-order block model of 1 M rows,
// 21 M entries, K = 32: SDDMM 427 + scaling 29 + SpMM 417 us forward, SpMM 416 + SDDMM 423 + dot product 42 us backward
// as separate operators.
#include "spmm_launch_impl.h"

// *out = the sum of v[0 .. n): the wavefronts' shares of the weight gradient, in a fixed order.  One workgroup: n is some
// 10^5 at most.
__global__ void __launch_bounds__(1024) psp_attn_wsum_kernel(const float *__restrict__ v, int n, float *__restrict__ out)
{
    __shared__ double part[16];
    double s = 0.0;
    const int n4 = n & ~3;
    for (int i = threadIdx.x * 4; i < n4; i += 4096) {
        const psp_f32x4 t = *(const psp_f32x4_a4 *)(v + i);
        s += ((double)t[0] + (double)t[1]) + ((double)t[2] + (double)t[3]);
    }
    if (n4 + (int)threadIdx.x < n) s += (double)v[n4 + threadIdx.x];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < 16; i++) s += part[i];
        *out = (float)s;
    }
}

// lanes per row and pieces per lane
static psp_spmm_plan attn_plan(int K, int blkWarpNum)
{
    const int nvec = psp_ceil_div(K, 4);
    psp_spmm_plan p;
    p.vec = 4;
    p.coarsen = nvec > 16 ? 2 : 1;
    p.lanes_per_row = nvec <= 4 ? 4 : nvec <= 8 ? 8 : 16;
    p.rows_per_wave = PSP_WAVE / p.lanes_per_row;
    p.unroll = p.coarsen == 1 ? 4 : 2;
    p.col_tiles = 1;
    p.waves_per_block = blkWarpNum & ~PSP_BW_STRIPE_MASK;
    p.log_segs_per_wave = -1;
    p.even_split = 0;
    p.xcd_stripe_rows = ((blkWarpNum & PSP_BW_STRIPE_MASK) >> PSP_BW_STRIPE_SHIFT) * 256;
    return p;
}

template <int NR, bool SPLIT, bool BWD, bool SLOT>
static int attn_enqueue(const psp_spmm_plan &p, const int *rowPtr, const int *colIdx, const float *val, const int *target_row,
                        const float *X, float *Y, int nrows, int K, int rows_out, const float *alpha, float *score, float *wsum,
                        const float *slot, hipStream_t st)
{
#define PSP_ATTN(LOGL_, C_, U_)                                                                                                   \
    {                                                                                                                             \
        typedef psp_attention<LOGL_, BWD, SLOT> xt_t;                                                                             \
        return psp_spmm_enqueue<NR, SPLIT>(psp_spmm_kernel<C_, 4, U_, NR, SPLIT, false, false, true, float, xt_t>, p, rowPtr, colIdx, \
                                           val, target_row, X, Y, nrows, K, rows_out, st, (const float *)nullptr, (float *)nullptr, 0, \
                                           xt_t{alpha, score, wsum, slot});                                                       \
    }
    if (p.lanes_per_row == 4) PSP_ATTN(2, 1, 4)
    if (p.lanes_per_row == 8) PSP_ATTN(3, 1, 4)
    if (p.coarsen == 1) PSP_ATTN(4, 1, 4)
    PSP_ATTN(4, 2, 2)
#undef PSP_ATTN
}

static int attn_launch(bool bwd, int fmt, const int *rowPtr, const int *colIdx, const float *val, const int *target_row, const float *X,
                       float *Y, int nrows, int K, int rows_out, int blkWarpNum, const float *alpha, float *score, float *wsum,
                       const float *slot, hipStream_t st)
{
    PSP_REQUIRE(fmt >= 0 && fmt <= 3, "attn: format code must be 0..3 (got %d)", fmt);
    PSP_REQUIRE(K >= 4 && K <= PSP_ATTN_MAX_K, "attn: K must be 4 .. %d (got %d)", PSP_ATTN_MAX_K, K);
    const int bw = blkWarpNum & ~PSP_BW_STRIPE_MASK;
    PSP_REQUIRE(bw == 4 || bw == 8, "attn: blkWarpNum must be 4 or 8 (got %d)", bw);
    PSP_REQUIRE(nrows >= 0 && rows_out >= 0, "attn: negative size (rows %d, rows_out %d)", nrows, rows_out);
    PSP_REQUIRE(Y != nullptr || rows_out == 0, "attn: Y is null");
    const bool split = fmt == 1 || fmt == 3;
    const int nr = fmt >= 2 ? 2 : 1;
    if (!split) PSP_REQUIRE((long long)nrows * nr <= rows_out, "attn: Y has %d rows, the matrix needs %lld", rows_out, (long long)nrows * nr);
    if (nrows > 0) PSP_REQUIRE(rowPtr && X && (!split || target_row), "attn: null pointer");
    const psp_spmm_plan p = attn_plan(K, blkWarpNum);
#define PSP_GO(NR_, SPLIT_)                                                                                                  \
    return !bwd ? attn_enqueue<NR_, SPLIT_, false, false>(p, rowPtr, colIdx, val, target_row, X, Y, nrows, K, rows_out, alpha, score, wsum, slot, st) \
         : NR_ > 1 || slot ? attn_enqueue<NR_, SPLIT_, true, true>(p, rowPtr, colIdx, val, target_row, X, Y, nrows, K, rows_out, alpha, score, wsum, slot, st) \
                           : attn_enqueue<NR_, SPLIT_, true, (NR_ > 1)>(p, rowPtr, colIdx, val, target_row, X, Y, nrows, K, rows_out, alpha, score, wsum, slot, st)
    if (fmt == 0) PSP_GO(1, false);
    if (fmt == 1) PSP_GO(1, true);
    if (fmt == 2) PSP_GO(2, false);
    PSP_GO(2, true);
#undef PSP_GO
}

PSP_EXPORT int psp_attn_forward_f32(int fmt, const int *rowPtr, const int *colIdx, const float *val_b, const int *target_row,
                                    const float *X, const float *alpha, float *att, float *Y, int nrows, int K, int rows_out,
                                    int blkWarpNum, psp_stream_t stream)
{
    PSP_REQUIRE((colIdx != nullptr) == (att != nullptr), "attn: colIdx and att must both be given (or both be null for a matrix without entries)");
    PSP_REQUIRE(fmt < 2 || val_b || !colIdx, "attn: block values are null");
    return attn_launch(false, fmt, rowPtr, colIdx, val_b, target_row, X, Y, nrows, K, rows_out, blkWarpNum, alpha, att, nullptr,
                       nullptr, (hipStream_t)stream);
}

// one float per wavefront of the backward launch; a wavefront takes at least half its lane groups' number of segments
PSP_EXPORT int psp_attn_workspace_floats(int nrows, int K)
{
    PSP_REQUIRE(nrows >= 0 && K >= 4 && K <= PSP_ATTN_MAX_K, "attn: bad size (rows %d, K %d)", nrows, K);
    return psp_ceil_div(nrows, attn_plan(K, 4).rows_per_wave / 2);
}

PSP_EXPORT int psp_attn_backward_f32(int fmt, const int *rowPtr, const int *colIdx, const float *att, const int *target_row,
                                     const float *slot, const float *dY, float *G, float *wsum, float *workspace, int nrows, int K, int rows_out,
                                     int blkWarpNum, psp_stream_t stream)
{
    PSP_REQUIRE(wsum, "attn: null pointer for the weight gradient");
    PSP_REQUIRE((colIdx != nullptr) == (att != nullptr), "attn: colIdx and att must both be given (or both be null for a matrix without entries)");
    PSP_REQUIRE(fmt < 2 || slot || !colIdx, "attn: the slots' columns are null");
    PSP_REQUIRE(workspace || nrows == 0, "attn: workspace is null");
    int rc = attn_launch(true, fmt, rowPtr, colIdx, att, target_row, dY, G, nrows, K, rows_out, blkWarpNum, nullptr, nullptr, workspace,
                         slot, (hipStream_t)stream);
    if (rc != PSP_OK) return rc;
    const int waves = nrows > 0 ? psp_ceil_div(nrows, 1 << psp_spmm_log_segs(attn_plan(K, blkWarpNum), nrows, fmt == 1 || fmt == 3)) : 0;
    hipLaunchKernelGGL(psp_attn_wsum_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, workspace, waves, wsum);
    return psp_check_launch("attention weight gradient");
}
