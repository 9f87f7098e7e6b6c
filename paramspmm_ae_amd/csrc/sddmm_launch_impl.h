// Host launcher shared by the four SDDMM translation units.
#pragma once
#include "sddmm_kernel.h"
#include <map>
#include <mutex>
#include <utility>

// Workgroups of `waves` wavefronts that fit a CU (asked once per kernel and size; races write the same value)
static inline int psp_sddmm_per_cu(psp_sddmm_kernel_t k, int waves)
{
    static std::mutex lock;
    static std::map<std::pair<psp_sddmm_kernel_t, int>, int> known;
    std::lock_guard<std::mutex> hold(lock);
    int &n = known[{k, waves}];
    if (n == 0 && (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void *)k, waves * PSP_WAVE, 0) != hipSuccess || n < 1)) n = 1;
    return n;
}

template <int NR, bool SPLIT>
int psp_sddmm_launch(const int *rowPtr, const int *colIdx, const float *val, const int *target_row,
                     const float *A, const float *B, const float *scale, float *out, int nrows, int K,
                     int blkWarpNum, hipStream_t stream, float *row_max)
{
    constexpr bool BCSR = NR > 1;
    const bool balanced = !SPLIT && (blkWarpNum & PSP_BW_BALANCED) != 0;  // plain layouts only; row-split input is balanced
    blkWarpNum &= ~PSP_BW_BALANCED;
    const int stripe_flag = ((blkWarpNum & PSP_BW_STRIPE_MASK) >> PSP_BW_STRIPE_SHIFT) * 256;  // 0: the library option
    blkWarpNum &= ~PSP_BW_STRIPE_MASK;
    PSP_REQUIRE(blkWarpNum == 4 || blkWarpNum == 8, "blkWarpNum must be 4 or 8");
    PSP_REQUIRE(nrows >= 0 && K >= 1, "sddmm: bad size (rows %d, K %d)", nrows, K);
    if (nrows == 0) return PSP_OK;
    // colIdx, out and the block values may be null for a matrix without stored entries: whether there are any is
    // written in rowPtr, which is on the device, and the kernel touches none of the three then
    PSP_REQUIRE(rowPtr && A && B, "sddmm: null pointer");
    PSP_REQUIRE((colIdx != nullptr) == (out != nullptr), "sddmm: colIdx and out must both be given (or both be null for a matrix without entries)");
    PSP_REQUIRE(!SPLIT || target_row, "sddmm: target_row is null");
    PSP_REQUIRE(!BCSR || val || !colIdx, "sddmm: block values are null");
    PSP_REQUIRE(!(BCSR && scale), "sddmm: scale is only supported for csr formats");
    PSP_REQUIRE(!(BCSR && row_max), "sddmm: row maxima are only supported for csr formats");

    // Widths of 5 to 7: the two pieces of a row would leave lane groups of two.  CSR takes four lanes (two of them idle), blocks a
    // float per lane on eight.  us at K = 6 with two lanes / so, plain and row-split CSR, plain and row-split 2x1 blocks: 300 000 rows
    // of 21 entries 77 / 38, 75 / 39, 142 / 50, 141 / 62; 200 003 skewed rows of 15 33 / 33, 47 / 32, 94 / 105, 87 / 48; a mesh 20 / 31,
    // 21 / 33, 44 / 33, 44 / 31.  8- and 4-byte pieces, in the same order: 45, 46, 76, 77; 35, 37, 103, 54; 38, 39, 25, 26.
    const bool few = K > 4 && K < 8;
    const int V = few && BCSR ? 1 : psp_vec_width(K);
    const int nvec = psp_ceil_div(K, V);
    int C = psp_ceil_div(nvec, 16);
    if (C > 4) C = 4;
    int logL = few ? 2 : 0;
    while ((C << logL) < nvec) logL++;
    if (logL > 6) return psp_fail(PSP_ERR_RANGE, "sddmm: K = %d is too wide (max %d)", K, 1024);
    if (logL < 4 && C > 1) C = 1;

    auto pick = [&](auto bal_) {
        constexpr bool BAL = !SPLIT && decltype(bal_)::value != 0;
        if constexpr (!BCSR) {
            if (row_max)
                return scale ? psp_sddmm_lookup<NR, SPLIT, true, BAL, true>(logL, C, V) : psp_sddmm_lookup<NR, SPLIT, false, BAL, true>(logL, C, V);
        }
        return scale ? psp_sddmm_lookup<NR, SPLIT, !BCSR, BAL>(logL, C, V) : psp_sddmm_lookup<NR, SPLIT, false, BAL>(logL, C, V);
    };
    psp_sddmm_kernel_t k = balanced ? pick(psp_int<1>()) : pick(psp_int<0>());
    if (!k) return psp_fail(PSP_ERR_ARG, "sddmm: no kernel for logL %d coarsen %d vec %d", logL, C, V);
    if (balanced) {
        // A grid that fills the GPU once; its wavefronts divide the stored entries between them in tiles of 256
        // (the entry count is on the device, in rowPtr): each XCD takes one contiguous eighth of the tiles.  "Once" is what the
        // kernel's registers allow: workgroups that start when others have ended would work through their full share alone
        // (10^6 rows of 21 entries, K = 32: 287 us with eight wavefronts per SIMD launched where six fit, 247 with six).
        const int wgs = 256 * psp_sddmm_per_cu(k, blkWarpNum);
        dim3 grid(wgs, 1, 1), block(blkWarpNum * PSP_WAVE, 1, 1);
        hipLaunchKernelGGL(k, grid, block, 0, stream, rowPtr, colIdx, BCSR ? val : scale, target_row, A, B, out, nrows, K,
                           8, wgs, wgs / PSP_XCDS, row_max);
        return psp_check_launch("sddmm kernel (entry-balanced)");
    }

    // segments per wavefront: as for SpMM (one per lane group for plain input, 16 for row-split input, fewer for
    // small matrices); groups of 32 and 64 lanes get two, so that the second row is on its way while the first is worked on
    // (K = 300, five entries per row: 985 -> 685 us)
    const int logR = 6 - logL;
    int logW = SPLIT ? (logR > 4 ? logR : 4) : (logL >= 5 ? logR + 1 : logR);
    while (logW > 0 && (nrows >> logW) < 4096) logW--;
    if (logW < logR - 1) logW = logR - 1;
    const int segs_per_block = blkWarpNum << logW;
    const psp_grid1d g = psp_xcd_grid(psp_ceil_div(nrows, segs_per_block), (stripe_flag ? stripe_flag : psp_stripe_rows()) / segs_per_block);
    dim3 grid(g.launch, 1, 1), block(blkWarpNum * PSP_WAVE, 1, 1);
    hipLaunchKernelGGL(k, grid, block, 0, stream, rowPtr, colIdx, BCSR ? val : scale, target_row, A, B, out, nrows, K,
                       logW, g.real, g.stripe, row_max);
    return psp_check_launch("sddmm kernel");
}
