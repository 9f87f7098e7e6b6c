// Parameterised SDDMM kernel for gfx950 (wave64): out[p] = <A[row(p),:], B[col(p),:]> for every stored
// entry p.  Semantics follow SDDMM/sddmm_kernel.cu:917-1287 (the stored values never scale the result; for
// 2x1 blocks they only decide which of the two entries is computed).
//
// A lane group of L = 2^LOGL lanes works on one sparse row at a time; each lane keeps C vectors of V floats of
// the A row in registers and loads the matching part of the B row, so a group reads L*V*4 contiguous bytes per load.
// The per-lane partial dot products are summed across the group with DPP / ds_swizzle butterflies.  The L
// results of one chunk of L non-zeros are parked one per lane and written with a single coalesced store
// (the reference stores one float per warp per non-zero).
#pragma once
#include "psp_common.h"
#include "spmm_kernel.h"  // psp_vec, psp_group_sum

template <int I> struct psp_int { static constexpr int value = I; };

// psp_group_sum (spmm_kernel.h) for double: both halves of a value cross the lanes, then they are added as one number
template <int LOGL> __device__ __forceinline__ double psp_group_sum(double v)
{
#define PSP_DPP_ADD64(CTRL)                                                                            \
    v += __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true),     \
                          __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true))
    if constexpr (LOGL >= 1) PSP_DPP_ADD64(0xB1);
    if constexpr (LOGL >= 2) PSP_DPP_ADD64(0x4E);
    if constexpr (LOGL >= 3) PSP_DPP_ADD64(0x141);
    if constexpr (LOGL >= 4) PSP_DPP_ADD64(0x140);
#undef PSP_DPP_ADD64
    if constexpr (LOGL >= 5) v += psp_bperm_f((int)((threadIdx.x ^ 16) & 63), v);
    if constexpr (LOGL >= 6) v += psp_bperm_f((int)((threadIdx.x ^ 32) & 63), v);
    return v;
}

// Maximum over aligned groups of 2^LOGL lanes (all lanes of the group active); every lane receives it.
template <int LOGL> __device__ __forceinline__ float psp_group_max(float v)
{
#define PSP_DPP_MAX(CTRL) v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xF, 0xF, false)))
    if constexpr (LOGL >= 1) PSP_DPP_MAX(0xB1);
    if constexpr (LOGL >= 2) PSP_DPP_MAX(0x4E);
    if constexpr (LOGL >= 3) PSP_DPP_MAX(0x141);
    if constexpr (LOGL >= 4) PSP_DPP_MAX(0x140);
#undef PSP_DPP_MAX
    if constexpr (LOGL >= 5) v = fmaxf(v, __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401F)));
    if constexpr (LOGL >= 6) v = fmaxf(v, __int_as_float(__builtin_amdgcn_ds_bpermute((int)((threadIdx.x ^ 32) & 63) << 2, __float_as_int(v))));
    return v;
}

// val: bcsr -> [nblk,2] block values (gate); csr -> optional per-entry scale (may be null when !SCALE)
//
// The gathers bind it: the rows of B come from wherever the columns point, and what counts is how many of them are under
// way.  So a group walks its entries U at a time whatever rows they belong to, with the next U requested before the
// current U are multiplied (two register sets), and changes its A row between two entries where one ends.  The walk by
// rows before this one stopped at every row's end, which on short rows left half of each step empty and nothing under way
// across it.  U = 2 up to 128 columns: 4 cost 10-16 registers and one to two wavefronts per SIMD (10^6 rows of 21 entries, plain, K = 32 /
// 64 / 128: by rows 236 / 428 / 784 us, U = 4 224 / 395 / 733, U = 2 198 / 357 / 667); U = 1 with four vectors per lane.
//
// The walk is the one of the SpMM kernel: a wavefront owns W = 2^logW consecutive segments, their stored entries
// are divided evenly between the 64/L lane groups, and a group reloads its A row (prefetched one segment ahead)
// whenever it crosses into another row.  Every stored entry is written exactly once, so `out` needs no clearing.
//
// MAX (CSR layouts): the largest result of every row is also raised into row_max[row] (atomic
// max, once per row and window; the caller has filled the array with the lowest float).  The attention
// pipeline's softmax-weighted SpMM takes its reference maxima from there instead of sweeping the entries again.
//
// BAL (plain layouts): the launch is a fixed grid of wavefronts that divide the *stored entries* between them -- each
// takes consecutive tiles of 2^logW entries, finds the rows that hold them with a 64-ary search in rowPtr and walks
// them window by window (up to 64 rows at a time, cut at the tile's ends).  Every entry's result is independent, so a
// row may be cut anywhere, and a hub row of 10^5 entries spreads over a hundred wavefronts instead of pinning one.
// T: float, or double in pieces of V = 2 (generic_f64.hip).
template <int LOGL, int C, int V, int U, int NR, bool SPLIT, bool SCALE, bool BAL = false, bool MAX = false, typename T = float>
__global__ void __launch_bounds__(512)
psp_sddmm_kernel(const int *__restrict__ rowPtr, const int *__restrict__ colIdx, const T *__restrict__ val,
                 const int *__restrict__ target_row, const T *__restrict__ A, const T *__restrict__ B,
                 T *__restrict__ out, int nseg, int K, int logW, int tiles, int stripe, float *__restrict__ row_max)
{
    typedef typename psp_vec<V, T>::type vec_t;
    typedef T pair_t __attribute__((ext_vector_type(2)));
    constexpr bool BCSR = NR > 1;  // NR rows per stored entry: 1 = CSR, 2 = 2x1 blocks, 3 = 3x1 blocks
    constexpr int L = 1 << LOGL;
    constexpr int R = PSP_WAVE >> LOGL;
    static_assert(U <= L, "unroll must not exceed the group width");
    static_assert(!BAL || !SPLIT, "the entry-balanced walk is for the plain layouts (row-split input is balanced already)");
    __shared__ int2 s_seg[PSP_MAX_WAVES][PSP_WAVE];  // (end offset, A row) of the wavefront's filled segments
    // CSR results of narrow groups wait here until the group has a 128-byte line of `out` together and then leave
    // in one burst of stores: a group stores only L floats at a time, and lines written piecemeal are evicted from the
    // L2 half-written by the gather stream (measured: 3x the result's bytes in HBM writes at L = 4).
    // 2x1 blocks hold pairs (16 blocks to a line); 3x1 blocks are stored directly.
    constexpr int LINE = 128 / sizeof(T);
    constexpr int HOLD = (NR <= 2 && LOGL >= 2 && ((LINE / NR) >> LOGL) >= 2) ? ((LINE / NR) >> LOGL) : 1;  // chunks held back per group
    __shared__ __align__(16) T s_hold[HOLD > 1 ? PSP_MAX_WAVES : 1][HOLD > 1 ? HOLD * PSP_WAVE * NR : 1];

    static_assert(!MAX || (sizeof(T) == 4 && !BCSR), "row maxima exist for the CSR layouts in single precision");
    __shared__ float s_max[MAX ? PSP_MAX_WAVES : 1][MAX ? PSP_WAVE : 1];  // largest result so far of each filled segment

    const int lane = threadIdx.x & (PSP_WAVE - 1);
    const int wave = threadIdx.x >> 6;
    const int sub = lane & (L - 1);
    const int grp = lane >> LOGL;
    const int grp_base = lane - sub;

    int off[C], dup[C];  // dup: leading columns of a piece that was moved back to end with the row (psp_vec_col)
    bool live[C];
#pragma unroll
    for (int i = 0; i < C; i++) {
        const int col = ((i << LOGL) + sub) * V;
        live[i] = col < K;
        off[i] = psp_vec_col<V>(col, K);
        dup[i] = col - off[i];
    }

    // One window: the segments s0 .. s0+nvalid-1 (at most 64), of which only the entries inside [pbeg, pend) count
    // (the plain walk passes the whole range of the segments).  tabW: power of two >= nvalid.
    auto run_window = [&](const int s0, const int nvalid, const int pbeg, const int pend, const int tabW) {
    const int W = tabW;
    const int P0 = pbeg;
    const int P1 = min(rowPtr[s0 + nvalid], pend);
    {
        const bool in = lane < nvalid;
        const int e = in ? min(rowPtr[s0 + lane + 1], pend) : P1;
        const int e_up = __shfl_up(e, 1);  // cross-lane reads stay outside any lane-dependent branch
        const int b_ = (lane == 0) ? P0 : e_up;
        const bool filled = in && e > b_;
        const unsigned long long fmask = __ballot(filled);
        const int slot = __popcll(fmask & ((1ull << lane) - 1ull));
        s_seg[wave][lane] = make_int2(P1, -1);
        if constexpr (MAX) s_max[wave][lane] = PSP_F32_LOWEST;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (filled) s_seg[wave][slot] = make_int2(e, SPLIT ? target_row[s0 + lane] : s0 + lane);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int2 *w_seg = s_seg[wave];
    if (P0 >= P1) return;

    const int q = (P1 - P0 + R - 1) >> (6 - LOGL);
    int a0 = P0 + grp * q;
    if (a0 > P1) a0 = P1;
    const int b0 = min(P1, a0 + q);
    if (a0 >= b0) return;  // the whole group leaves together; nothing below reads other groups' lanes

    // A row(s) of a segment; dead tail vectors and repeated columns are zero so they add nothing to the dot product
    auto load_a = [&](int key, T (&dst)[NR][C][V]) {
#pragma unroll
        for (int r = 0; r < NR; r++)
#pragma unroll
            for (int i = 0; i < C; i++) {
                vec_t t;
                if constexpr (V == 1) t = (T)0;
                else {
#pragma unroll
                    for (int e = 0; e < V; e++) t[e] = (T)0;
                }
                if (live[i]) t = psp_load_vec<V, T>(A + (size_t)(key * NR + r) * (size_t)K + off[i]);
#pragma unroll
                for (int e = 0; e < V; e++) dst[r][i][e] = e >= dup[i] ? psp_elem<V, T>(t, e) : (T)0;
            }
    };

    int cur = 0;
    for (int step = W >> 1; step >= 1; step >>= 1)
        if (w_seg[cur + step - 1].x <= a0) cur += step;
    int row_end = w_seg[cur].x;
    int mykey = w_seg[cur].y;
    T a[NR][C][V], a_nxt[NR][C][V];
    load_a(mykey, a);
    {
        const int nk = cur + 1 < PSP_WAVE ? w_seg[cur + 1].y : -1;
        load_a(nk >= 0 ? nk : mykey, a_nxt);
    }

    float lmax = PSP_F32_LOWEST;  // largest result among this lane's entries of the current row
    auto emit_row_max = [&](int slot) {
        const float m = psp_group_max<LOGL>(lmax);
        if constexpr (MAX) {
            if (sub == 0) __hip_atomic_fetch_max(&s_max[wave][slot], m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        lmax = PSP_F32_LOWEST;
    };

    // lane `sub` of the group picks up entry base+sub (column index and, where the format has one, its value); the
    // next chunk's are requested before the current chunk is worked on
    auto fetch = [&](int base, int &c_out, T (&g_out)[NR]) {
        const int q = base + sub;
        const int qq = q < b0 ? q : b0 - 1;
        c_out = colIdx[qq];
        if constexpr (NR == 2) {
            const pair_t t = ((const pair_t *)val)[qq];
            g_out[0] = t[0];
            g_out[1] = t[1];
        } else if constexpr (NR > 2) {
#pragma unroll
            for (int r = 0; r < NR; r++) g_out[r] = val[(size_t)qq * NR + r];
        } else {
            g_out[0] = SCALE ? val[qq] : (T)1;
        }
    };
    int c_cur;
    T gate[NR];
    fetch(a0, c_cur, gate);
    int held = 0;         // chunks waiting in s_hold (group-uniform)
    int hold_base = a0;   // entry of the first of them
    // every lane reads back what it wrote itself, so the wavefront's program order is all the ordering needed
    auto release = [&]() {
#pragma unroll
        for (int j = 0; j < HOLD; j++) {
            const int pp = hold_base + (j << LOGL) + sub;
            if (j < held && pp < b0) {
                if constexpr (NR == 2) ((pair_t *)out)[pp] = ((const pair_t *)s_hold[wave])[j * PSP_WAVE + lane];
                else out[pp] = s_hold[wave][j * PSP_WAVE + lane];
            }
        }
        hold_base += held << LOGL;
        held = 0;
    };

    constexpr int STEPS = L / U;
    static_assert(STEPS == 1 || STEPS % 2 == 0, "the two register sets alternate through a chunk");
    vec_t bv[2][U][C];
    auto gather = [&](int k, int cols, vec_t (&dst)[U][C]) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const T *br = B + (size_t)psp_bperm_i(grp_base + k + u, cols) * (size_t)K;
#pragma unroll
            for (int i = 0; i < C; i++) dst[u][i] = psp_load_vec<V, T>(br + off[i]);
        }
    };
    // the current row is finished: go to the next filled segment, whose A row was requested one segment ago
    auto next_row = [&]() {
        const int2 nx = w_seg[++cur];
        row_end = nx.x;
        if (nx.y != mykey) {
            if constexpr (MAX) emit_row_max(cur - 1);  // the group is converged here: the condition is group-uniform
            mykey = nx.y;
#pragma unroll
            for (int r = 0; r < NR; r++)
#pragma unroll
                for (int i = 0; i < C; i++)
#pragma unroll
                    for (int e = 0; e < V; e++) a[r][i][e] = a_nxt[r][i][e];
        }
        const int nk = cur + 1 < PSP_WAVE ? w_seg[cur + 1].y : -1;
        if (nk >= 0 && nk != mykey) load_a(nk, a_nxt);
    };
    gather(0, c_cur, bv[0]);

    for (int base = a0; base < b0; base += L) {
        const int p = base + sub;
        const bool ok = p < b0;
        int c_nxt = c_cur;
        T gate_nxt[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) gate_nxt[r] = (T)0;
        if (base + L < b0) fetch(base + L, c_nxt, gate_nxt);
        T res[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) res[r] = (T)0;

        // U entries at a time, the next U entries' rows of B on the way meanwhile (from the next chunk's columns at the end)
        auto step = [&](const int st, auto set_) {
            constexpr int SET = decltype(set_)::value;
            if (base + st * U >= b0) return;
            if (base + (st + 1) * U < b0) {
                if (st + 1 < STEPS) gather((st + 1) * U, c_cur, bv[1 - SET]);
                else gather(0, c_nxt, bv[1 - SET]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int e_ = base + st * U + u;
                if (e_ == row_end && e_ < b0) next_row();
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    T part = (T)0;
#pragma unroll
                    for (int i = 0; i < C; i++)
#pragma unroll
                        for (int e = 0; e < V; e++) part = psp_fma(a[r][i][e], psp_elem<V, T>(bv[SET][u][i], e), part);
                    part = psp_group_sum<LOGL>(part);
                    if (sub == st * U + u && e_ < b0) {
                        res[r] = part;
                        if constexpr (MAX) lmax = fmaxf(lmax, SCALE ? part * gate[0] : part);
                    }
                }
            }
            if constexpr (STEPS == 1) {
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int i = 0; i < C; i++) bv[0][u][i] = bv[1][u][i];
            }
        };
        if constexpr (STEPS == 1) step(0, psp_int<0>());
        else {
#pragma unroll(LOGL >= 5 ? 1 : STEPS)  // (wide groups: 2 x 16 or 2 x 32 copies of the body would not fit the instruction cache)
            for (int st = 0; st < STEPS; st += 2) {
                step(st, psp_int<0>());
                step(st + 1, psp_int<1>());
            }
        }
        if (ok) {
            if constexpr (NR == 2 && HOLD == 1) {
                // entries of a block whose value is zero are padding: written as zero (sddmm_kernel.cu:1103,1115)
                pair_t o;
                o[0] = gate[0] != (T)0 ? res[0] : (T)0;
                o[1] = gate[1] != (T)0 ? res[1] : (T)0;
                ((pair_t *)out)[p] = o;
            } else if constexpr (NR > 2) {
#pragma unroll
                for (int r = 0; r < NR; r++) out[(size_t)p * NR + r] = gate[r] != (T)0 ? res[r] : (T)0;
            } else if constexpr (HOLD == 1) {
                out[p] = SCALE ? res[0] * gate[0] : res[0];
            }
        }
        if constexpr (HOLD > 1) {
            if constexpr (NR == 2) {
                pair_t o;  // padding entries of a block (value zero) are written as zero (sddmm_kernel.cu:1103,1115)
                o[0] = gate[0] != (T)0 ? res[0] : (T)0;
                o[1] = gate[1] != (T)0 ? res[1] : (T)0;
                ((pair_t *)s_hold[wave])[held * PSP_WAVE + lane] = o;
            } else {
                s_hold[wave][held * PSP_WAVE + lane] = SCALE ? res[0] * gate[0] : res[0];
            }
            if (++held == HOLD) release();
        }
        c_cur = c_nxt;
#pragma unroll
        for (int r = 0; r < NR; r++) gate[r] = gate_nxt[r];
    }
    if constexpr (HOLD > 1) release();
    if constexpr (MAX) emit_row_max(cur);
    };  // run_window

    // The window's row maxima leave together, one per lane (a row's segments are neighbours in the table: their first takes the
    // maximum of all), because neighbouring rows' atomics then share a request: one atomic per row and lane group, sent
    // as each row closed, took up to a third of the kernel (10^6 rows of 21 entries, K = 32: 309 us, like this 281, without maxima
    // 247).  Stores for the rows that no other wavefront touches made it slower, not faster (atomics act behind the L2, and
    // lines that see both kinds go back and forth).
    auto flush_max = [&](const int tabW) {
        if constexpr (MAX) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int key = s_seg[wave][lane].y;
            float m = s_max[wave][lane];
            bool first = true;
            if constexpr (SPLIT) {
                first = lane == 0 || s_seg[wave][lane > 0 ? lane - 1 : 0].y != key;
                for (int d = 1; d < tabW; d <<= 1) {
                    const int k_ = psp_bperm_i((lane + d) & (PSP_WAVE - 1), key);
                    const float m_ = psp_bperm_f((lane + d) & (PSP_WAVE - 1), m);
                    if (lane + d < PSP_WAVE && k_ == key) m = fmaxf(m, m_);
                }
            }
            if (first && key >= 0 && m > PSP_F32_LOWEST) psp_atomic_max_f32(row_max + key, m);
        }
    };
    if constexpr (!BAL) {
        const int tile = psp_xcd_tile(stripe);
        if (tile >= tiles) return;
        const int s0 = (tile * (int)(blockDim.x >> 6) + wave) << logW;
        if (s0 >= nseg) return;  // wave-uniform
        const int nvalid = min(1 << logW, nseg - s0);
        run_window(s0, nvalid, rowPtr[s0], 0x7fffffff, 1 << logW);
        flush_max(1 << logW);
    } else {
        // Tiles of 2^logW stored entries.  Each XCD (workgroups are dealt to them round-robin) owns one contiguous
        // eighth of the tiles and its wavefronts take them in turn, so at any time an XCD works on a run of
        // neighbouring tiles -- neighbouring rows, whose B rows share its L2 -- and all XCDs carry the same load.
        const int nnz = rowPtr[nseg];
        const int ntiles = (int)(((long long)nnz + (1 << logW) - 1) >> logW);
        const int wpb = blockDim.x >> 6;
        const int xcd = blockIdx.x % PSP_XCDS;
        const int waves_per_xcd = (gridDim.x / PSP_XCDS) * wpb;
        const int tiles_per_xcd = (ntiles + PSP_XCDS - 1) / PSP_XCDS;
        const int band_end = min(ntiles, (xcd + 1) * tiles_per_xcd);
        for (int t = xcd * tiles_per_xcd + (blockIdx.x / PSP_XCDS) * wpb + wave; t < band_end; t += waves_per_xcd) {
        const int e0 = t << logW;
        const int e1 = min(nnz, e0 + (1 << logW));
        // first row whose end lies past e0: 64-ary search, one independent load per lane and round
        int lo = 0, hi = nseg;  // rowPtr[i + 1] <= e0 for i < lo, > e0 for i >= hi
        while (lo < hi) {
            const int step = (hi - lo + 63) >> 6;
            const int i = lo + lane * step;
            const bool gt = i >= hi || rowPtr[i + 1] > e0;  // ascending probes: false up to some lane, true from there on
            const unsigned long long m = __ballot(gt);
            const int f = m ? __ffsll((long long)m) - 1 : 64;
            int nlo = f == 0 ? lo : lo + (f - 1) * step + 1;
            int nhi = f == 64 ? hi : lo + f * step;
            lo = nlo < hi ? nlo : hi;
            hi = nhi < hi ? nhi : hi;
        }
        int s0 = lo, pbeg = e0;
        while (pbeg < e1 && s0 < nseg) {  // wave-uniform
            const int nvalid = min(PSP_WAVE, nseg - s0);
            run_window(s0, nvalid, pbeg, e1, PSP_WAVE);
            flush_max(PSP_WAVE);
            // the next window's table overwrites this one's: every group has finished reading it here
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            pbeg = min(rowPtr[s0 + nvalid], e1);
            s0 += nvalid;
        }
        }  // tiles of this wavefront
    }
}

typedef void (*psp_sddmm_kernel_t)(const int *, const int *, const float *, const int *, const float *,
                                   const float *, float *, int, int, int, int, int, float *);

// (LOGL, C, U) triples that exist.  C grows only once the group is 16 lanes wide (DPP-only reduction);
// beyond 64 vectors the group widens to 32 and 64 lanes.
#define PSP_SDDMM_FOR_EACH_LCU(M_) \
    M_(0, 1, 1) M_(1, 1, 1) M_(2, 1, 2) M_(3, 1, 2) M_(4, 1, 2) \
    M_(4, 2, 2) M_(4, 3, 2) M_(4, 4, 1) M_(5, 4, 1) M_(6, 4, 2)

template <int NR, bool SPLIT, bool SCALE, bool BAL = false, bool MAX = false>
static psp_sddmm_kernel_t psp_sddmm_lookup(int logL, int C, int V)
{
#define PSP_CASE(L_, C_, U_)                                                               \
    if (logL == L_ && C == C_) {                                                           \
        if (V == 4) return psp_sddmm_kernel<L_, C_, 4, U_, NR, SPLIT, SCALE, BAL, MAX>;       \
        return psp_sddmm_kernel<L_, C_, 1, U_, NR, SPLIT, SCALE, BAL, MAX>;                   \
    }
    PSP_SDDMM_FOR_EACH_LCU(PSP_CASE)
#undef PSP_CASE
    return nullptr;
}

template <int NR, bool SPLIT>
int psp_sddmm_launch(const int *rowPtr, const int *colIdx, const float *val, const int *target_row,
                     const float *A, const float *B, const float *scale, float *out, int nrows, int K,
                     int blkWarpNum, hipStream_t stream, float *row_max);
