// Both gradients of a layer that reads its input Z [n,K1] through a ReLU, from G = A dY [n,K2] and the weights W [K1,K2]:
//   dZ = (G W^T) where Z > 0,    dW = max(Z, 0)^T G
// in one launch.  The two products read the same two matrices; as launches of their own (dense_xw.hip, dense_atb.hip) they
// read them twice, and on a graph of 10^4 rows each costs its 3-4 us of launch and latency whatever it does.
// HBM-bound: 4 n (2 K1 + K2) bytes.  Both products, one after the other -> this kernel, with the sum of the partial products:
// 20 K rows 16 x 16 13.5 -> 8.2 us, 10^6 rows 16 x 16 54 -> 37, 48 x 48 197 -> 150, 64 x 64 302 -> 212
// (memory: 160), 128 x 16 355 -> 249 (227).
#include "psp_common.h"
#include "dense_tiles.h"

// A wavefront takes 16 rows at a time and loads them twice, in the layouts of the two products (both are described in the
// files named above): the second load of a row follows the first at once and finds it in the CU's L1 or the L2.  Everything a
// step needs is requested before its first MFMA; as many workgroups per CU as the registers allow keep the memory busy while
// others multiply.  Steps of 32 rows keep fewer of them: 10^6 rows 48 x 48 155 us against 150, 64 x 64 215 against 212, 200 K rows
// 64 x 64 58 against 52; only at 16 x 16, where the registers do not limit, they are faster (37 against 43).
// The workgroups' parts of dW go to `partial` (K1 x K2 each) and are added afterwards in a fixed order.
// n > 0; rows past n are loaded from row n - 1, enter dW as zeros and are not stored.
constexpr int psp_dense_grad_wgs(int K1, int K2) { return K1 + K2 > 144 ? 2 : K1 + K2 > 80 ? 3 : 4; }  // per CU
constexpr int psp_dense_grad_halves(int K1, int K2) { return K1 + K2 <= 32 ? 2 : 1; }  // 16 rows each, per step
template <int K1, int K2>
__global__ void __launch_bounds__(256, psp_dense_grad_wgs(K1, K2))
psp_dense_grad_kernel(const float *__restrict__ G, const float *__restrict__ Z, const float *__restrict__ W,
                      float *__restrict__ dZ, float *__restrict__ partial, long long n, long long nblocks)
{
    constexpr int RM = K1 / 16, RN = K2 / 16;  // column tiles of Z and of G
    constexpr int H = psp_dense_grad_halves(K1, K2), U = 4 * H;
    constexpr int TQ = (RM + 3) / 4;
    constexpr int S = XWW_STRIDE(K1);
    constexpr int LDS = K2 * S > RM * RN * 256 ? K2 * S : RM * RN * 256;
    __shared__ float lds[LDS];  // W, transposed and permuted as in psp_xw_kernel; at the end the wavefronts' sums

    for (int idx = threadIdx.x; idx < K1 * K2; idx += 256) {
        const int c = idx / K2, k = idx % K2;
        lds[k * S + (((c >> 6) * 16 + (c & 15)) << 2) + ((c >> 4) & 3)] = W[idx];
    }
    __syncthreads();

    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    psp_mfma_acc dw[RM][RN];
#pragma unroll
    for (int m = 0; m < RM; m++)
#pragma unroll
        for (int t = 0; t < RN; t++) dw[m][t] = psp_mfma_acc{0.f, 0.f, 0.f, 0.f};

    for (long long blk = (long long)blockIdx.x * 4 + w; blk < nblocks; blk += (long long)gridDim.x * 4) {
        const long long row0 = blk * (16 * H);
        const bool whole = row0 + 16 * H <= n;
        psp_f32x4 g4[H][RN], z4[H][RM];     // of row 16 h + r: columns 16 t + 4 q ..
        float az[U][RM], bg[U][RN];         // of row 4 u + q: psp_atb_col of r
#pragma unroll
        for (int h = 0; h < H; h++) {
            const long long row = min(row0 + 16 * h + r, n - 1);
#pragma unroll
            for (int t = 0; t < RN; t++) g4[h][t] = ((const psp_f32x4 *)(G + row * K2) + q)[4 * t];
#pragma unroll
            for (int t = 0; t < RM; t++) z4[h][t] = ((const psp_f32x4 *)(Z + row * K1) + q)[4 * t];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const long long row = min(row0 + 4 * u + q, n - 1);
            psp_atb_load_row<RM>(Z + row * K1, r, az[u]);
            psp_atb_load_row<RN>(G + row * K2, r, bg[u]);
        }
        __builtin_amdgcn_sched_barrier(0);  // the loads stay in front of the products

        psp_mfma_acc acc[H][RM];
#pragma unroll
        for (int h = 0; h < H; h++)
#pragma unroll
            for (int j = 0; j < RM; j++) acc[h][j] = psp_mfma_acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < RN; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const psp_f32x4 *wr = (const psp_f32x4 *)(lds + (16 * t + 4 * q + e) * S) + r;
                psp_f32x4 a4[TQ];
#pragma unroll
                for (int v = 0; v < TQ; v++) a4[v] = wr[16 * v];
#pragma unroll
                for (int j = 0; j < RM; j++)
#pragma unroll
                    for (int h = 0; h < H; h++)
                        acc[h][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[j / 4][j % 4], g4[h][t][e], acc[h][j], 0, 0, 0);
            }
#pragma unroll
        for (int h = 0; h < H; h++) {
            const long long row = row0 + 16 * h + r;
            if (row >= n) continue;
            psp_f32x4 *out = (psp_f32x4 *)(dZ + row * K1) + q;
#pragma unroll
            for (int j = 0; j < RM; j++) {
                psp_f32x4 o = acc[h][j];
#pragma unroll
                for (int c = 0; c < 4; c++) o[c] = psp_relu_grad(o[c], z4[h][j][c]);
                out[4 * j] = o;
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool in = whole || row0 + 4 * u + q < n;
#pragma unroll
            for (int m = 0; m < RM; m++) az[u][m] = !in || az[u][m] < 0.0f ? 0.0f : az[u][m];  // NaN stays NaN
#pragma unroll
            for (int t = 0; t < RN; t++) bg[u][t] = in ? bg[u][t] : 0.0f;
#pragma unroll
            for (int m = 0; m < RM; m++)
#pragma unroll
                for (int t = 0; t < RN; t++) dw[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(az[u][m], bg[u][t], dw[m][t], 0, 0, 0);
        }
    }
    __syncthreads();  // W is read no more
    for (int turn = 0; turn < 4; turn++) {
        if (w == turn) {
#pragma unroll
            for (int m = 0; m < RM; m++)
#pragma unroll
                for (int t = 0; t < RN; t++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        float *x = &lds[((m * RN + t) * 4 + v) * 64 + lane];
                        *x = turn == 0 ? dw[m][t][v] : *x + dw[m][t][v];
                    }
        }
        __syncthreads();
    }
    float *dst = partial + (size_t)blockIdx.x * (K1 * K2);
    for (int e = threadIdx.x; e < RM * RN * 256; e += 256) {
        const int l = e & 63, v = (e >> 6) & 3, tile = e >> 8;
        dst[psp_atb_col<RM>(tile / RN, 4 * (l >> 4) + v) * K2 + psp_atb_col<RN>(tile % RN, l & 15)] = lds[e];
    }
}

typedef void (*psp_dense_grad_kernel_t)(const float *, const float *, const float *, float *, float *, long long, long long);

// Up to 25 tiles, K1 K2 <= 80 x 80: the accumulators of 96 x 96 leave one wavefront per SIMD, and the two fp32 products need as
// long on the matrix cores as the memory system for the rows (10^6 rows 478 us as two launches, 416 as one; 200 K rows 114, 120).
static psp_dense_grad_kernel_t dense_grad_lookup(int K1, int K2)
{
#define DG(a, b) \
    if (K1 == a && K2 == b) return psp_dense_grad_kernel<a, b>;
#define DG_ROW(a) DG(a, 16) DG(a, 32) DG(a, 48)
    DG_ROW(16) DG_ROW(32) DG_ROW(48) DG_ROW(64) DG_ROW(80) DG_ROW(96) DG_ROW(112) DG_ROW(128)
#define DG_WIDE(a) DG(a, 64) DG(a, 80)
    DG_WIDE(16) DG_WIDE(32) DG_WIDE(48) DG_WIDE(64) DG_WIDE(80)
    DG(96, 64) DG(16, 96) DG(16, 112) DG(16, 128) DG(32, 96) DG(32, 112) DG(32, 128) DG(48, 96) DG(48, 112) DG(48, 128) DG(64, 96)
#undef DG_WIDE
#undef DG_ROW
#undef DG
    return nullptr;
}
static long long dense_grad_grid(long long n, int K1, int K2)
{
    const long long wgs = (n + 63) / 64, most = 256 * psp_dense_grad_wgs(K1, K2);
    return wgs < most ? wgs : most;
}

PSP_EXPORT int psp_dense_grad_supported(int K1, int K2) { return dense_grad_lookup(K1, K2) != nullptr; }

PSP_EXPORT long long psp_dense_grad_workspace_floats(long long n, int K1, int K2)
{
    return n <= 0 || !dense_grad_lookup(K1, K2) ? 0 : dense_grad_grid(n, K1, K2) * K1 * K2;
}

PSP_EXPORT int psp_dense_grad_f32(const float *G, const float *Z, const float *W, float *dZ, float *dW, long long n, int K1,
                                  int K2, float *workspace, long long workspace_floats, psp_stream_t stream)
{
    psp_dense_grad_kernel_t k = dense_grad_lookup(K1, K2);
    PSP_REQUIRE(k != nullptr, "dense_grad: unsupported widths %d x %d (see psp_dense_grad_supported)", K1, K2);
    PSP_REQUIRE(n > 0 && G && Z && W && dZ && workspace, "dense_grad: null pointer or no rows");
    PSP_REQUIRE((((size_t)G | (size_t)Z | (size_t)dZ) & 15) == 0, "dense_grad: G, Z and dZ must be 16-byte aligned");
    PSP_REQUIRE(n / 128 < 0x7fffffffLL, "dense_grad: too many rows");
    const long long grid = dense_grad_grid(n, K1, K2), rows = 16 * psp_dense_grad_halves(K1, K2);
    PSP_REQUIRE(workspace_floats >= grid * K1 * K2, "dense_grad: the workspace holds %lld floats, %lld needed", workspace_floats, grid * K1 * K2);
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(256), 0, (hipStream_t)stream, G, Z, W, dZ, workspace, n, (n + rows - 1) / rows);
    const int rc = psp_check_launch("dense_grad kernel");
    if (rc != PSP_OK) return rc;
    if (!dW) return (int)grid;
    const psp_partial_sum sum = {workspace, dW, (int)grid, K1 * K2};
    return psp_sum_partials_f32(&sum, 1, stream);
}
