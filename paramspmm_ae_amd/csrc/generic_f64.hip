// Double-precision SpMM and SDDMM for all six layouts (CSR / 2x1 / 3x1 blocks, plain or row-split).  The reference
// dispatches its kernels for double as well as float (AT_DISPATCH_FLOATING_TYPES, SpMM_kernel.cu:149, sddmm_kernel.cu
// :161).  Both run the float path's walks (spmm_kernel.h, sddmm_kernel.h) on pieces of two doubles, one 16-byte load.
#include "psp_common.h"
#include "spmm_launch_impl.h"
#include "sddmm_kernel.h"

// SDDMM of rows wider than the lane groups' registers hold (K > PSP_SDDMM_F64_MAX_K): one wavefront per segment, groups of
// W lanes (W covers min(K, 64) columns) take its entries in turn.  out[nblk, NR] (out[nnz] for NR = 1); entries whose block
// value is zero are written as zero.
template <int NR, bool SPLIT>
__global__ void __launch_bounds__(256)
sddmm_f64_kernel(const int *__restrict__ rowPtr, const int *__restrict__ colIdx, const double *__restrict__ val_b,
                 const int *__restrict__ target_row, const double *__restrict__ A, const double *__restrict__ B,
                 double *__restrict__ out, int nseg, int K, int logW)
{
    const int lane = threadIdx.x & 63;
    const int s = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (s >= nseg) return;
    const int lb = rowPtr[s], hb = rowPtr[s + 1];
    const int key = SPLIT ? target_row[s] : s;
    const int W = 1 << logW, G = 64 >> logW;
    const int sub = lane & (W - 1), grp = lane >> logW;
    for (int p0 = lb; p0 < hb; p0 += G) {  // wave-uniform trip count: the exchange below needs every lane
        const int p = p0 + grp;
        const bool have = p < hb;
        const double *b = B + (size_t)(have ? colIdx[p] : 0) * K;
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const bool live = have && (NR == 1 || val_b[(size_t)p * NR + r] != 0.0);  // uniform within a group
            double part = 0.0;
            if (live) {
                const double *a = A + (size_t)(key * NR + r) * K;
                for (int k = sub; k < K; k += W) part = fma(a[k], b[k], part);
            }
#pragma unroll
            for (int i = 0; i < 6; i++) {
                const double other = __shfl_xor(part, 1 << i);
                if ((1 << i) < W) part += other;  // wave-uniform
            }
            if (sub == 0 && have) out[(size_t)p * NR + r] = live ? part : 0.0;
        }
    }
}

// lanes per group of that kernel: the power of two that covers min(width, 64)
static int f64_log_group(int width)
{
    int logW = 0;
    while ((1 << logW) < width && logW < 6) logW++;
    return logW;
}

typedef void (*spmm_f64_kernel_t)(const int *, const int *, const double *, const int *, const double *, double *,
                                  int, int, int, int, int, int, int, const float *, float *, int, int, psp_plain);

// Mapping: two pieces of two doubles per lane, two entries in flight, lane groups of up to 8 lanes for rows of up to 32
// doubles (one column tile of 256 bytes) and up to 16 beyond.  Bound by the memory traffic; of thirteen mappings (1 / 2 / 4
// pieces x 4 ... 32 lanes x 1 ... 4 entries) measured on a mesh, an R-MAT and a block-model graph at N = 16 / 32 / 47 / 100
// this one is within 12 % of the best nearly everywhere.  Mesh of 2.1 M rows, 2x1 blocks, N = 32: 806 us before (one
// wavefront per block-row, 8-byte loads, Y cleared by a pass of its own) -> 272 us, 4.5 TB/s of the bytes it cannot do
// without; CSR 299 us.  Rows of up to 8 doubles: one piece per lane, four entries in flight and groups of four lanes even
// where fewer would cover the row -- with one lane per row a wavefront's 64 rows were 64 serial chains (N = 3 on the block
// model: 349 us).
template <int NR, bool SPLIT>
static int spmm_f64_launch(const int *rowPtr, const int *colIdx, const double *val, const int *target_row, const double *X,
                           double *Y, int nseg, int N, int rows_out, hipStream_t st)
{
    const int V = N >= 2 ? 2 : 1, nvec = psp_ceil_div(N, V);
    const int C = nvec <= 4 ? 1 : 2, U = C == 1 ? 4 : 2, widest = nvec <= 16 ? 8 : 16;
    int L = 4;
    while (L < widest && L * C < nvec) L <<= 1;
    spmm_f64_kernel_t k = V == 1 ? psp_spmm_kernel<1, 1, 4, NR, SPLIT, false, false, true, double>
                        : C == 1 ? psp_spmm_kernel<1, 2, 4, NR, SPLIT, false, false, true, double>
                                 : psp_spmm_kernel<2, 2, 2, NR, SPLIT, false, false, true, double>;
    psp_spmm_plan plan;
    plan.vec = V;
    plan.coarsen = C;
    plan.lanes_per_row = L;
    plan.rows_per_wave = PSP_WAVE / L;
    plan.unroll = U;
    plan.col_tiles = psp_ceil_div(nvec, L * C);
    plan.waves_per_block = 4;
    plan.log_segs_per_wave = -1;
    plan.even_split = 0;
    plan.xcd_stripe_rows = 0;
    return psp_spmm_enqueue<NR, SPLIT>(k, plan, rowPtr, colIdx, val, target_row, X, Y, nseg, N, rows_out, st, (const float *)nullptr,
                                       (float *)nullptr, 0);
}

PSP_EXPORT int psp_spmm_f64(const int *rowPtr, const int *colIdx, const double *val, const int *target_row,
                            const double *X, double *Y, int nseg, int N, int rows_out, int vec_size, psp_stream_t stream)
{
    PSP_REQUIRE(nseg >= 0 && N >= 0 && rows_out >= 0, "spmm_f64: negative size");
    PSP_REQUIRE(vec_size >= 1 && vec_size <= 3, "spmm_f64: vec_size must be 1, 2 or 3 (got %d)", vec_size);
    PSP_REQUIRE(Y || rows_out == 0 || N == 0, "spmm_f64: Y is null");
    if (!target_row) PSP_REQUIRE((long long)nseg * vec_size <= rows_out, "spmm_f64: Y has %d rows, the matrix needs %lld",
                                 rows_out, (long long)nseg * vec_size);
    hipStream_t st = (hipStream_t)stream;
    if (N == 0) return PSP_OK;
    if (nseg > 0) PSP_REQUIRE(rowPtr && X, "spmm_f64: rowPtr / X is null");
#define PSP_F64(NR_, SPLIT_) spmm_f64_launch<NR_, SPLIT_>(rowPtr, colIdx, val, target_row, X, Y, nseg, N, rows_out, st)
    if (vec_size == 1) return target_row ? PSP_F64(1, true) : PSP_F64(1, false);
    if (vec_size == 2) return target_row ? PSP_F64(2, true) : PSP_F64(2, false);
    return target_row ? PSP_F64(3, true) : PSP_F64(3, false);
#undef PSP_F64
}

typedef void (*sddmm_f64_kernel_t)(const int *, const int *, const double *, const int *, const double *, const double *, double *,
                                   int, int, int, int, int, float *);
#define PSP_SDDMM_F64_MAX_K 512  // 64 lanes x 4 pieces of two doubles

template <int NR, bool SPLIT>
static int sddmm_f64_launch(const int *rowPtr, const int *colIdx, const double *val_b, const int *target_row,
                            const double *A, const double *B, double *out, int nseg, int K, hipStream_t st)
{
    if (K > PSP_SDDMM_F64_MAX_K) {
        hipLaunchKernelGGL((sddmm_f64_kernel<NR, SPLIT>), dim3(psp_ceil_div(nseg, 4)), dim3(256), 0, st, rowPtr, colIdx, val_b,
                           target_row, A, B, out, nseg, K, f64_log_group(K));
        return psp_check_launch("sddmm f64 kernel");
    }
    // vectors per lane and lanes per row: as for float (psp_sddmm_launch)
    const int V = K >= 2 ? 2 : 1, nvec = psp_ceil_div(K, V);
    // at least four lanes, as above
    int C = std::min(psp_ceil_div(nvec, 16), 4), logL = 2;
    while ((C << logL) < nvec) logL++;
    if (logL < 4) C = 1;
    sddmm_f64_kernel_t k = nullptr;
#define PSP_CASE(L_, C_, U_) \
    if constexpr (L_ >= 2) { \
        if (V == 2 && logL == L_ && C == C_) k = psp_sddmm_kernel<L_, C_, 2, U_, NR, SPLIT, false, false, false, double>; \
    }
    PSP_SDDMM_FOR_EACH_LCU(PSP_CASE)
#undef PSP_CASE
    if (V == 1) k = psp_sddmm_kernel<2, 1, 1, 4, NR, SPLIT, false, false, false, double>;
    PSP_REQUIRE(k, "sddmm_f64: no kernel for K = %d", K);
    const int logR = 6 - logL;
    int logW = SPLIT ? (logR > 4 ? logR : 4) : logR;
    while (logW > 0 && (nseg >> logW) < 4096) logW--;
    if (logW < logR - 1) logW = logR - 1;
    const int segs_per_block = 4 << logW;
    const psp_grid1d g = psp_xcd_grid(psp_ceil_div(nseg, segs_per_block), psp_stripe_rows() / segs_per_block);
    hipLaunchKernelGGL(k, dim3(g.launch), dim3(256), 0, st, rowPtr, colIdx, val_b, target_row, A, B, out, nseg, K, logW, g.real,
                       g.stripe, (float *)nullptr);
    return psp_check_launch("sddmm f64 kernel");
}

PSP_EXPORT int psp_sddmm_f64(const int *rowPtr, const int *colIdx, const double *val_b, const int *target_row,
                             const double *A, const double *B, double *out, int nseg, int K, int vec_size,
                             psp_stream_t stream)
{
    PSP_REQUIRE(nseg >= 0 && K >= 1, "sddmm_f64: bad size (segments %d, K %d)", nseg, K);
    PSP_REQUIRE(vec_size >= 1 && vec_size <= 3, "sddmm_f64: vec_size must be 1, 2 or 3 (got %d)", vec_size);
    if (nseg == 0) return PSP_OK;
    // colIdx, out and the block values may be null for a matrix without stored entries (only rowPtr, on the device, tells)
    PSP_REQUIRE(rowPtr && A && B, "sddmm_f64: null pointer");
    PSP_REQUIRE((colIdx != nullptr) == (out != nullptr), "sddmm_f64: colIdx and out must both be given (or both be null for a matrix without entries)");
    PSP_REQUIRE(vec_size == 1 || val_b || !colIdx, "sddmm_f64: block values are null");
    hipStream_t st = (hipStream_t)stream;
#define PSP_F64(NR_, SPLIT_) sddmm_f64_launch<NR_, SPLIT_>(rowPtr, colIdx, val_b, target_row, A, B, out, nseg, K, st)
    if (vec_size == 1) return target_row ? PSP_F64(1, true) : PSP_F64(1, false);
    if (vec_size == 2) return target_row ? PSP_F64(2, true) : PSP_F64(2, false);
    return target_row ? PSP_F64(3, true) : PSP_F64(3, false);
#undef PSP_F64
}
