// Y[n,K2] = X[n,K1] * W  (W [K1,K2] row-major)  or  X * W^T  (W [K2,K1] row-major) for tall-skinny X (n ~ 10^6) and a small
// weight matrix, widths multiples of 16 up to 128: the dense products around the sparse one in the fused GCN layer,
// torch::mm(H, W) and torch::mm(AG, W.t()) in SpCONV/SpCONV.h:43-71, with the ReLU between two layers folded in.  The work is
// reading X and writing Y once; a general GEMM reaches a third of the memory rate at these shapes (98 us for 1M x 16 x 16
// where the traffic needs 30 us).  It runs on the matrix cores (v_mfma_f32_16x16x4_f32, fp32 in, fp32 accumulate): at
// 128 x 128 the product is 32 kflop per row against 1 KB of traffic and matrix-core time and memory time are about equal; at
// 16 and 32 output columns there is little to multiply, but the loads and stores of this form (64 contiguous bytes per row
// and instruction) move more than those of one lane per row with scalar FMAs, which it replaced: 10^6 rows, 16 x 16 32 -> 20
// us, 32 x 16 47 -> 30, 32 x 32 75 -> 47, masked 109 -> 73, 64 x 16 90 -> 53.  Widths off 16, 32, 64 and 128 went to
// PyTorch's GEMM with passes for the activation or the mask: 48 x 48 208 -> 81 us, masked 246 -> 109, 96 x 96 409 -> 185.
//
// RELU_X: X enters the product as max(x, 0) (the activation between two layers, applied as the next layer reads its
// input).  MASK: an output element is kept where the same element of `mask` is positive and zero elsewhere (the
// activation's backward, applied as the gradient with respect to the layer's input is written).
//
// The product is formed transposed, Y^T = W^T X^T, so that a lane ends up with consecutive elements of one output row:
//   * MFMA operand B (4 x 16) is a piece of X^T: lane (r, q) = (lane % 16, lane / 16) supplies X[row r][k]; it loads
//     its row 16 bytes at a time, float4 t covering columns 16t + 4q .. 16t + 4q + 3, so the four q-lanes of a row
//     read 64 contiguous bytes.  Element e of float4 t is used in contraction step (t, e), where the lane's column
//     16t + 4q + e stands for index k = q of the instruction: which four columns a step contracts is free as long as
//     operand A follows the same rule;
//     NATURAL: the lane's float4 is first transposed among the four q-lanes of its row (permlane swaps), so that step (t, e)
//     contracts columns 16t + 4e .. 16t + 4e + 3 and every output is one chain of FMAs in ascending k -- bit for bit the sums of
//     the one-lane-per-row kernel this one replaced.  Up to 32 output columns, where those sums are in use and the four
//     swaps per load vanish in the memory time; the wider outputs never had that order;
//   * operand A (16 x 4) is a piece of W^T read from LDS: lane (r, q) supplies W[16t + 4q + e][16j + r] for column
//     tile j (T = K2 / 16 tiles).  LDS holds the columns of W permuted -- column 16j + r at position
//     ((j / 4) * 16 + r) * 4 + j % 4 -- so a lane fetches four tiles with one 16-byte read and the sixteen r-lanes of
//     such a read cover 256 contiguous bytes (no bank conflicts): two reads per step serve eight MFMAs (sixteen with
//     the two row blocks a wavefront works on).  A tile count that is no multiple of four leaves the last read's tail
//     unused;
//   * result lane (r, q), tile j, element i is Y[row r][16j + 4q + i]: one 16-byte store per tile, the four q-lanes
//     of a row writing 64 contiguous bytes.
// W (K1 rows of K2 + 4 floats: 66 KB at 128 x 128) is staged into LDS once per workgroup, transposed on the way in for
// the X * W^T form.  That is more than the 64 KB a workgroup gets on earlier CDNA parts: the kernel is built for
// gfx950 only, whose CUs have 160 KB, and two workgroups per CU (the launch shape) need 132 KB of it.  The grid is sized
// to the GPU and every wavefront walks blocks of 32 rows with the next block's loads in flight.
#include "psp_common.h"
#include "bf16_split.h"
#include "dense_tiles.h"
#include <cstdlib>

#define XWW_ROWS 32  // rows per wavefront and step: two MFMA row blocks share every operand read from LDS

// 4 x 4 transpose between the four 16-lane rows of a wavefront and the four elements of v: element e of row q <-> element q of
// row e
__device__ __forceinline__ void psp_transpose_rows(psp_f32x4 &v)
{
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    unsigned a = __float_as_uint(v[0]), b = __float_as_uint(v[1]), c = __float_as_uint(v[2]), d = __float_as_uint(v[3]);
    u32x2 t = __builtin_amdgcn_permlane32_swap(a, c, false, false);
    a = t[0], c = t[1];
    t = __builtin_amdgcn_permlane32_swap(b, d, false, false);
    b = t[0], d = t[1];
    t = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = t[0], b = t[1];
    t = __builtin_amdgcn_permlane16_swap(c, d, false, false);
    c = t[0], d = t[1];
    v = psp_f32x4{__uint_as_float(a), __uint_as_float(b), __uint_as_float(c), __uint_as_float(d)};
}

template <int K1, int K2, bool RELU_X, bool MASK, bool NATURAL>
// (the bound of 512 lanes leaves the register allocator 256 registers per lane; launched with 256)
__global__ void __launch_bounds__(512)
psp_xw_kernel(const float *__restrict__ X, const float *__restrict__ W, float *__restrict__ Y, long long n,
                   const float *__restrict__ mask, int transW, long long nblocks)
{
    constexpr int T = K2 / 16;         // column tiles
    constexpr int TQ = (T + 3) / 4;    // 16-byte LDS reads per contraction step
    constexpr int KT = K1 / 16;        // float4 loads per lane and row block
    constexpr int S = XWW_STRIDE(K2);  // LDS row stride: the four k-rows a step reads fall into different bank halves
    static_assert(K2 % 16 == 0 && K1 % 16 == 0, "widths are multiples of 16");
    // two workgroups share a CU's 160 KB of LDS
    static_assert(sizeof(float) * K1 * S <= 80 * 1024, "W does not fit half of a gfx950 CU's LDS");
    __shared__ float Ws[K1 * S];

    for (int idx = threadIdx.x; idx < K1 * K2; idx += blockDim.x) {
        int k, c;
        if (transW) {  // W is [K2, K1]
            c = idx / K1;
            k = idx - c * K1;
        } else {  // W is [K1, K2]
            k = idx / K2;
            c = idx - k * K2;
        }
        Ws[k * S + (((c >> 6) * 16 + (c & 15)) << 2) + ((c >> 4) & 3)] = W[idx];
    }
    __syncthreads();

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int waves = blockDim.x >> 6;
    const long long stride = (long long)gridDim.x * waves;
    long long blk = (long long)blockIdx.x * waves + wave;
    if (blk >= nblocks) return;

    psp_f32x4 xa[2][KT], xb[2][KT];
    auto load_block = [&](long long b, psp_f32x4 (&x)[2][KT]) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            long long row = b * XWW_ROWS + 16 * h + r;
            if (row >= n) row = n - 1;  // loaded and computed, never stored
            const psp_f32x4 *xr = (const psp_f32x4 *)(X + row * K1) + q;
#pragma unroll
            for (int t = 0; t < KT; t++) x[h][t] = xr[4 * t];
        }
    };
    auto compute_block = [&](long long b, psp_f32x4 (&x)[2][KT]) {
        if constexpr (RELU_X) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int t = 0; t < KT; t++)
#pragma unroll
                    for (int e = 0; e < 4; e++) x[h][t][e] = x[h][t][e] < 0.0f ? 0.0f : x[h][t][e];  // NaN stays NaN
        }
        if constexpr (NATURAL) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int t = 0; t < KT; t++) psp_transpose_rows(x[h][t]);
        }
        psp_f32x4 acc[2][T];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int j = 0; j < T; j++) acc[h][j] = psp_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < KT; t++) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const psp_f32x4 *wr = (const psp_f32x4 *)(Ws + (16 * t + (NATURAL ? 4 * e + q : 4 * q + e)) * S) + r;
                psp_f32x4 a4[TQ];
#pragma unroll
                for (int v = 0; v < TQ; v++) a4[v] = wr[16 * v];
#pragma unroll
                for (int j = 0; j < T; j++) {
#pragma unroll
                    for (int h = 0; h < 2; h++)
                        acc[h][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[j / 4][j % 4], x[h][t][e], acc[h][j], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const long long row = b * XWW_ROWS + 16 * h + r;
            if (row >= n) continue;
            psp_f32x4 *yr = (psp_f32x4 *)(Y + row * K2) + q;
            const psp_f32x4 *mr = (const psp_f32x4 *)(mask + row * K2) + q;
#pragma unroll
            for (int j = 0; j < T; j++) {
                psp_f32x4 o = acc[h][j];
                if constexpr (MASK) {
                    const psp_f32x4 m = mr[4 * j];
#pragma unroll
                    for (int c = 0; c < 4; c++) o[c] = psp_relu_grad(o[c], m[c]);
                }
                yr[4 * j] = o;
            }
        }
    };

    // two register sets alternate: the next block's rows are requested before the current block is multiplied
    load_block(blk, xa);
    while (true) {
        long long nxt = blk + stride;
        if (nxt < nblocks) load_block(nxt, xb);
        __builtin_amdgcn_sched_barrier(0);
        compute_block(blk, xa);
        if (nxt >= nblocks) break;
        blk = nxt;
        nxt = blk + stride;
        if (nxt < nblocks) load_block(nxt, xa);
        __builtin_amdgcn_sched_barrier(0);
        compute_block(blk, xb);
        if (nxt >= nblocks) break;
        blk = nxt;
    }
}

// ---- the 128 x 128 product on the bf16 matrix-core path (option dense_split, from PSP_SPLIT_MIN_ROWS rows on) -----------------
// At 128 x 128 the fp32 instruction above needs as long for its 32 kflop per row as the memory system needs for the row's
// 1 KB.  gfx950 multiplies bf16 sixteen times as fast, and an fp32 number is the exact sum of three bf16 numbers
// (x = hi + mid + lo, 8 + 8 + 8 significant bits), so x w = sum of nine bf16 products, of which the six with at least
// 16 significant bits between them (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi) carry the product to 2^-23 of |x||w|
// -- the rounding level of an fp32 product -- and are accumulated in fp32 by v_mfma_f32_16x16x32_bf16.  Six instructions
// of 16 cycles replace eight of 32: the kernel is bound by its 1 KB per row again.  Same transposed form and the same
// lane roles as above; a contraction step covers 32 columns: lane (r, q) supplies the eight values of its float4 pair
// (2s, 2s + 1), i.e. columns 32s + 16 (i / 4) + 4q + i % 4 stand for k = 8q + i, and the W fragments in LDS follow the same
// rule: [s][tile j][hi | mid | lo][lane][8 bf16], one 16-byte read per fragment.  An infinite input turns its products
// into NaN (inf - inf in the split) instead of +-inf; NaN stays NaN.

template <bool RELU_X, bool MASK>
__global__ void __launch_bounds__(512)
psp_xw_split_kernel(const float *__restrict__ X, const float *__restrict__ W, float *__restrict__ Y, long long n,
                         const float *__restrict__ mask, int transW, long long nblocks)
{
    constexpr int K1 = 128, K2 = 128;
    constexpr int T = K2 / 16;   // column tiles
    constexpr int KT = K1 / 16;  // float4 loads per lane and row block
    constexpr int KS = K1 / 32;  // contraction steps
    extern __shared__ __align__(16) unsigned short Wb[];  // [KS][T][3][64][8]

    for (int idx = threadIdx.x; idx < K1 * K2; idx += blockDim.x) {
        const int i = idx & 7, l = (idx >> 3) & 63, sj = idx >> 9;  // sj = s * T + j
        const int j = sj % T, st = sj / T;
        const int r_ = l & 15, q_ = l >> 4;
        const int k = 32 * st + 16 * (i >> 2) + 4 * q_ + (i & 3), c = 16 * j + r_;
        const float w = transW ? W[c * K1 + k] : W[k * K2 + c];
        unsigned hi, mid, lo;
        psp_split3(w, 0.0f, hi, mid, lo);
        unsigned short *at = Wb + ((size_t)(sj * 3) * 64 + l) * 8 + i;
        at[0] = (unsigned short)hi;
        at[64 * 8] = (unsigned short)mid;
        at[2 * 64 * 8] = (unsigned short)lo;
    }
    __syncthreads();

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int waves = blockDim.x >> 6;
    const long long stride = (long long)gridDim.x * waves;
    long long blk = (long long)blockIdx.x * waves + wave;
    if (blk >= nblocks) return;

    psp_f32x4 xa[2][KT], xb[2][KT];
    auto load_block = [&](long long b, psp_f32x4 (&x)[2][KT]) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            long long row = b * XWW_ROWS + 16 * h + r;
            if (row >= n) row = n - 1;  // loaded and computed, never stored
            const psp_f32x4 *xr = (const psp_f32x4 *)(X + row * K1) + q;
#pragma unroll
            for (int t = 0; t < KT; t++) x[h][t] = xr[4 * t];
        }
    };
    auto compute_block = [&](long long b, psp_f32x4 (&x)[2][KT]) {
        psp_f32x4 acc[2][T];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int j = 0; j < T; j++) acc[h][j] = psp_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < KS; st++) {
            psp_u32x4 xh[2], xm[2], xl[2];
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    float a = x[h][2 * st + (g >> 1)][2 * (g & 1)], c = x[h][2 * st + (g >> 1)][2 * (g & 1) + 1];
                    if constexpr (RELU_X) {
                        a = a < 0.0f ? 0.0f : a;  // NaN stays NaN
                        c = c < 0.0f ? 0.0f : c;
                    }
                    unsigned h_, m_, l_;
                    psp_split3(a, c, h_, m_, l_);
                    xh[h][g] = h_, xm[h][g] = m_, xl[h][g] = l_;
                }
            const psp_u32x4 *wf = (const psp_u32x4 *)Wb + (size_t)(st * T * 3) * 64 + lane;
#pragma unroll
            for (int jp = 0; jp < T; jp += 2) {
                psp_u32x4 w[2][3];
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int p = 0; p < 3; p++) w[u][p] = wf[((jp + u) * 3 + p) * 64];
                // small terms first; four independent accumulators between two instructions on the same one
#define XWS_TERM(WP_, XV_)                                                                                          \
    _Pragma("unroll") for (int u = 0; u < 2; u++) _Pragma("unroll") for (int h = 0; h < 2; h++)                       \
        acc[h][jp + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(psp_bf16x8, w[u][WP_]),           \
                                                                 __builtin_bit_cast(psp_bf16x8, XV_[h]), acc[h][jp + u], 0, 0, 0);
                XWS_TERM(2, xh)
                XWS_TERM(0, xl)
                XWS_TERM(1, xm)
                XWS_TERM(1, xh)
                XWS_TERM(0, xm)
                XWS_TERM(0, xh)
#undef XWS_TERM
            }
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const long long row = b * XWW_ROWS + 16 * h + r;
            if (row >= n) continue;
            psp_f32x4 *yr = (psp_f32x4 *)(Y + row * K2) + q;
            const psp_f32x4 *mr = (const psp_f32x4 *)(mask + row * K2) + q;
#pragma unroll
            for (int j = 0; j < T; j++) {
                psp_f32x4 o = acc[h][j];
                if constexpr (MASK) {
                    const psp_f32x4 m = mr[4 * j];
#pragma unroll
                    for (int c = 0; c < 4; c++) o[c] = psp_relu_grad(o[c], m[c]);
                }
                yr[4 * j] = o;
            }
        }
    };

    load_block(blk, xa);
    while (true) {
        long long nxt = blk + stride;
        if (nxt < nblocks) load_block(nxt, xb);
        __builtin_amdgcn_sched_barrier(0);
        compute_block(blk, xa);
        if (nxt >= nblocks) break;
        blk = nxt;
        nxt = blk + stride;
        if (nxt < nblocks) load_block(nxt, xa);
        __builtin_amdgcn_sched_barrier(0);
        compute_block(blk, xb);
        if (nxt >= nblocks) break;
        blk = nxt;
    }
}

typedef void (*psp_xw_kernel_t)(const float *, const float *, float *, long long, const float *, int, long long);

static psp_xw_kernel_t xw_lookup(int K1, int K2, bool relu_x, bool mask)
{
#define XWW_CASE(A_, B_)                                                   \
    if (K1 == A_ && K2 == B_) {                                            \
        constexpr bool nat = B_ <= 32;                                     \
        if (mask) return psp_xw_kernel<A_, B_, false, true, nat>;          \
        return relu_x ? psp_xw_kernel<A_, B_, true, false, nat> : psp_xw_kernel<A_, B_, false, false, nat>; \
    }
#define XWW_ROW(B_) XWW_CASE(16, B_) XWW_CASE(32, B_) XWW_CASE(48, B_) XWW_CASE(64, B_) XWW_CASE(80, B_) XWW_CASE(96, B_) XWW_CASE(112, B_) XWW_CASE(128, B_)
    XWW_ROW(16) XWW_ROW(32) XWW_ROW(48) XWW_ROW(64) XWW_ROW(80) XWW_ROW(96) XWW_ROW(112) XWW_ROW(128)
#undef XWW_ROW
#undef XWW_CASE
    return nullptr;
}

PSP_EXPORT int psp_gemm_xw_supported(int K1, int K2)
{
    if (xw_lookup(K1, K2, false, false) == nullptr) return 0;
    // the staged W must fit what the device grants one workgroup (160 KB per CU on gfx950)
    static int lds_of[64];  // per device, looked up once (0 = not yet; races write the same value)
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int lds = lds_of[dev];
    if (lds == 0) {
        if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) return 0;
        lds_of[dev] = lds;
    }
    return (size_t)lds >= sizeof(float) * (size_t)K1 * (size_t)XWW_STRIDE(K2);
}

PSP_EXPORT int psp_gemm_xw_act_f32(const float *X, const float *W, float *Y, long long n, int K1, int K2, int transW,
                                   int relu_x, const float *mask, psp_stream_t stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    PSP_REQUIRE(n >= 0 && K1 >= 1 && K2 >= 1, "gemm_xw: bad size");
    PSP_REQUIRE(!(transW && relu_x), "gemm_xw: the activation on X exists for the plain product only");
    PSP_REQUIRE(!(!transW && mask), "gemm_xw: the output mask exists for the transposed product only");
    psp_xw_kernel_t k = xw_lookup(K1, K2, relu_x != 0, mask != nullptr);
    PSP_REQUIRE(k != nullptr, "gemm_xw: unsupported widths %d x %d (see psp_gemm_xw_supported)", K1, K2);
    if (n == 0) return PSP_OK;
    PSP_REQUIRE(X && W && Y, "gemm_xw: null pointer");
    PSP_REQUIRE((((size_t)X | (size_t)Y | (size_t)mask) & 15) == 0, "gemm_xw: X, Y and mask must be 16-byte aligned");
    PSP_REQUIRE((n + 255) / 256 <= 0x7fffffffLL, "gemm_xw: too many rows");
    const long long nblocks = (n + XWW_ROWS - 1) / XWW_ROWS;
    if (K1 == 128 && K2 == 128 && n >= PSP_SPLIT_MIN_ROWS && psp_opts().dense_split) {
        psp_xw_kernel_t ks = mask ? psp_xw_split_kernel<false, true>
                                       : (relu_x ? psp_xw_split_kernel<true, false> : psp_xw_split_kernel<false, false>);
        const int lds = (K1 / 32) * (K2 / 16) * 3 * 64 * 16;  // 96 KB: one workgroup of eight wavefronts per CU
        static bool raised[3];
        const int which = mask ? 0 : (relu_x ? 1 : 2);
        if (!raised[which]) {
            const hipError_t e = hipFuncSetAttribute((const void *)ks, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e != hipSuccess) return psp_fail(PSP_ERR_LAUNCH, "gemm_xw: %d bytes of LDS refused: %s", lds, hipGetErrorString(e));
            raised[which] = true;
        }
        // eight wavefronts per workgroup, one workgroup per CU (measured against four and six: 267 / 278 / 283 us at 10^6 rows)
        const int wv = 8;
        const long long want_s = (nblocks + wv - 1) / wv;
        const int grid_s = (int)(want_s < 256 ? want_s : 256);
        hipLaunchKernelGGL(ks, dim3(grid_s), dim3(64 * wv), lds, stream, X, W, Y, n, mask, transW, nblocks);
        return psp_check_launch("gemm_xw split kernel");
    }
    // 4 wavefronts per workgroup, two workgroups per CU (two copies of W in LDS side by side); measured against 6 and 8
    // wavefronts per workgroup and one to four workgroups per CU at 10^6 rows: nothing faster
    const int waves = 4;
    const long long want = (nblocks + waves - 1) / waves;
    const int grid = (int)(want < 512 ? want : 512);
    hipLaunchKernelGGL(k, dim3(grid), dim3(64 * waves), 0, stream, X, W, Y, n, mask, transW, nblocks);
    return psp_check_launch("gemm_xw kernel");
}

PSP_EXPORT int psp_gemm_xw_f32(const float *X, const float *W, float *Y, long long n, int K1, int K2, int transW,
                               psp_stream_t stream)
{
    return psp_gemm_xw_act_f32(X, W, Y, n, K1, K2, transW, 0, nullptr, stream);
}
