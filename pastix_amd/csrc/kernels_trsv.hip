// Supernodal forward / backward solve kernels for CDNA4 (gfx950)
// (reference kernels/solve_ztrsmsp.c:67-557, sopalin/sequential_ztrsm.c:34-103).
//
// The sweeps read b from x and leave the solution in x; the forward result
// z = inv(L) b lives in a separate buffer so that every workgroup of a cblk
// can read the cblk's input while others write their rows of the output.
// The sweeps go over solve nodes: a node is one cblk, or a run of cblks
// whose diagonal blocks and coupling blocks form one dense lower-triangular
// block, solved with that block's whole inverse.
// Forward sweep, level by level:
//   k_fwd_diag : workgroup (nd, ib) gathers, for rows [0, 64*ib+64) of node
//                nd, b minus the update-buffer entries of these rows (stored
//                contiguously per row, sources in increasing order), then
//                writes rows [64*ib, 64*ib+64) of z_nd = inv(L_nd) y;
//   k_fwd_prod : the products of the members' panel rows outside their node
//                on 64-row tiles, each product row stored at its entry of
//                the update buffer.
// Backward sweep, levels from the root down:
//   k_bwd_prod : partial[j] = sum over a strip of L[r, j] x[row(r)] (panel
//                rows outside the node);
//   k_bwd_diag : workgroup (nd, ib) forms y = z_nd - the strips' partials for
//                columns [64*ib, K) and writes rows [64*ib, 64*ib+64) of
//                x_nd = inv(L_nd)^T y.
// The diagonal inverses are stored whole (zeros in the other triangle), so
// the triangular products run over full 64-column blocks.  Every output
// element is produced in a fixed order by one workgroup: no atomics,
// bitwise-reproducible solves.  NW: waves of a workgroup.  Several
// right-hand sides take the kernels on the matrix cores (k_*_m,
// k_diag_gemm16), one takes the vector kernels.
#include <algorithm>

#include "dev_common.h"
#include "dev_types.h"
#include "kernels.h"

namespace pxa {

static inline int grid8(int n) { return ((n + 7) / 8) * 8; }
// levels whose widest cblk has at most this many columns run the solve
// kernels on 4-wave workgroups,
constexpr int SOLVE_NARROW = 64;
// and one-wave workgroups at most this many (the leaf levels)
constexpr int SOLVE_TINY = 16;
// levels whose widest node has more columns gather once per 64-row block
// before the diagonal kernels (k_fwd_gather, k_bwd_reduce)
constexpr int SOLVE_SPLIT = 512;

// red holds NW x 64 partial sums; the sum over waves is taken in wave order
// by the threads of wave 0.
template <typename T, int NW>
__device__ __forceinline__ void wave_sum_store(T acc, T *red, int r, int q, bool ok, T *out) {
    red[q * 64 + r] = acc;
    __syncthreads();
    if (q == 0 && ok) {
        T v = red[r];
#pragma unroll
        for (int w = 1; w < NW; w++) v += red[w * 64 + r];
        *out = v;
    }
}

// The same for partial sums held as E consecutive rows per lane: lane l of
// wave q holds rows E*(l % (64/E)) + i of columns l / (64/E); the E lanes of a
// row group combine with lane shuffles, then the waves as above (row r =
// the calling lane).
template <typename T, int NW, int E>
__device__ __forceinline__ void wave_sum_store_rows(T (&acc)[E], T *red, int r, int q, bool ok, T *out) {
    constexpr int G = 64 / E;
#pragma unroll
    for (int off = G; off < 64; off *= 2)
#pragma unroll
        for (int i = 0; i < E; i++) acc[i] += __shfl_xor(acc[i], off);
    if (r < G) {
#pragma unroll
        for (int i = 0; i < E; i++) red[q * 64 + E * r + i] = acc[i];
    }
    __syncthreads();
    if (q == 0 && ok) {
        T v = red[r];
#pragma unroll
        for (int w = 1; w < NW; w++) v += red[w * 64 + r];
        *out = v;
    }
}

// ------------------- one right-hand side: level kernels ---------------------
template <typename T, int NW>
__global__ __launch_bounds__(NW * 64) void k_fwd_diag(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                      const YSlices ys, const T *__restrict__ ybuf,
                                                      const T *__restrict__ b, T *__restrict__ z,
                                                      const T *__restrict__ w1, const T *__restrict__ w1t) {
    extern __shared__ char smem_raw[];
    T *y = reinterpret_cast<T *>(smem_raw);
    __shared__ T red[NW * 64];
    // the blocks with the most rows to gather and columns to read (the last
    // ones of a node) take the lowest workgroup ids, so that they start first
    const int id = (int)gridDim.x - 1 - xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const DiagItem it = items[id];
    const int tid = threadIdx.x, r = tid & 63, q = tid >> 6;
    const int nd = it.nd, r0 = it.ib * 64;
    const int fc = S.cblk_fcol[S.node_cblk[nd]];
    const int Kc = S.cblk_fcol[S.node_cblk[nd + 1]] - fc;
    const int nrow = min(Kc, r0 + 64);
    // y = b minus the pending products of rows [0, nrow): gl consecutive
    // lanes per row, as many as fill the workgroup in one pass (at most 64,
    // at most the node's first row's entry count), lane j summing the
    // entries j, j + gl, ... of its row, UL loads issued together, in order;
    // the lanes' sums combined by xor shuffles in a fixed order.  With one
    // lane per row, consecutive lanes read consecutive rows' entries, which
    // the sliced update buffer keeps side by side.
    const int ne = ys.cnt[fc];
    int gl = 1;
    while (gl < 64 && gl * 2 <= ne && nrow * gl * 2 <= NW * 64) gl *= 2;
    // rows of the inverse: E consecutive per lane (16-byte loads); the first
    // PF column groups are fetched before the gather, so that their latency
    // overlaps it
    constexpr int E = Vec<T>::E, G = 64 / E, PF = 4;
    const int rr = E * (r % G), kc = r / G;
    const bool mrow = r0 + rr < Kc;
    const T *M = w1 + S.node_winv[nd] + r0 + rr;
    // with W^T at hand (LL^t): row i of W is read as column i of W^T
    // (contiguous), NW lanes per row (row r0 + jt, lane lt)
    const bool tw = w1t != nullptr;
    const int jt = tid / NW, lt = tid % NW, it_row = r0 + jt;
    const T *MT = tw ? w1t + S.node_winv[nd] + (int64_t)it_row * Kc : nullptr;
    T mpre[PF][E];
#pragma unroll
    for (int f = 0; f < PF; f++) {
        if (tw) {
            const int k = E * lt + f * NW * E;
            if (it_row < Kc && k <= it_row) ld_rows(MT + k, k, it_row + 1, mpre[f]);
        } else {
            const int k = q * E + kc + f * NW * E;
            if (mrow && k < nrow) ld_rows(M + (int64_t)k * Kc, rr, Kc - r0, mpre[f]);
        }
    }
    constexpr int UL = 16;
    for (int base = 0; base < nrow * gl; base += NW * 64) {
        const int t = base + tid, i = t / gl, j = t % gl;
        T v = 0;
        if (i < nrow) {
            const int g = fc + i, ne_i = ys.cnt[g];
            const T *yb = ybuf + ys.base[g >> 6] + (g & 63);
            for (int e = j; e < ne_i; e += UL * gl) {
                T a[UL];
#pragma unroll
                for (int k = 0; k < UL; k++) a[k] = (e + k * gl < ne_i) ? yb[(int64_t)(e + k * gl) * 64] : (T)0;
#pragma unroll
                for (int k = 0; k < UL; k++) v += a[k];
            }
        }
        for (int o = gl >> 1; o >= 1; o >>= 1) v += __shfl_xor(v, o);
        if (i < nrow && j == 0) y[i] = b[fc + i] - v;
    }
    __syncthreads();
    if (tw) {
        // W[i, k] = W^T[k, i] is nonzero for k <= i; y holds rows [0, nrow)
        T a2[E];
#pragma unroll
        for (int e = 0; e < E; e++) a2[e] = 0;
        if (it_row < Kc) {
#pragma unroll
            for (int f = 0; f < PF; f++) {
                const int k = E * lt + f * NW * E;
                if (k <= it_row) {
#pragma unroll
                    for (int e = 0; e < E; e++) a2[e] += mpre[f][e] * y[min(k + e, it_row)];
                }
            }
#pragma unroll 4
            for (int k = E * lt + PF * NW * E; k <= it_row; k += NW * E) {
                T m[E];
                ld_rows(MT + k, k, it_row + 1, m);
#pragma unroll
                for (int e = 0; e < E; e++) a2[e] += m[e] * y[min(k + e, it_row)];
            }
        }
        T v = 0;
#pragma unroll
        for (int e = 0; e < E; e++) v += a2[e];
#pragma unroll
        for (int o = NW / 2; o >= 1; o >>= 1) v += __shfl_xor(v, o, NW);
        if (lt == 0 && it_row < Kc) z[fc + it_row] = v;
        return;  // uniform: tw is the same for the whole workgroup
    }
    const int i = r0 + r;
    T acc[E];
#pragma unroll
    for (int e = 0; e < E; e++) acc[e] = 0;
    if (mrow) {
#pragma unroll
        for (int f = 0; f < PF; f++) {
            const int k = q * E + kc + f * NW * E;
            if (k < nrow) {
#pragma unroll
                for (int e = 0; e < E; e++) acc[e] += mpre[f][e] * y[k];
            }
        }
#pragma unroll 4
        for (int k = q * E + kc + PF * NW * E; k < nrow; k += NW * E) {
            T m[E];
            ld_rows(M + (int64_t)k * Kc, rr, Kc - r0, m);
#pragma unroll
            for (int e = 0; e < E; e++) acc[e] += m[e] * y[k];
        }
    }
    wave_sum_store_rows<T, NW, E>(acc, red, r, q, i < Kc, z + fc + i);
}

template <typename T, int NW>
__global__ __launch_bounds__(NW * 64) void k_fwd_prod(DevSymbol S, const FwdItem *__restrict__ items, int nitems,
                                                      const T *__restrict__ coef, const T *__restrict__ z,
                                                      const int32_t *__restrict__ ydst, T *__restrict__ ybuf) {
    extern __shared__ char smem_raw[];
    T *xs = reinterpret_cast<T *>(smem_raw);
    __shared__ T red[NW * 64];
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const FwdItem it = items[id];
    const int tid = threadIdx.x, r = tid & 63, q = tid >> 6;
    const int c = it.c;
    const int fc = S.cblk_fcol[c];
    const int Kc = S.cblk_fcol[c + 1] - fc;
    const int64_t ld = S.cblk_stride[c];
    for (int t = tid; t < Kc; t += NW * 64) xs[t] = z[fc + t];
    __syncthreads();
    const int nr = it.r1 - it.r0;
    // E consecutive rows per lane (one 16-byte load), E columns per wave
    // instruction
    constexpr int E = Vec<T>::E, G = 64 / E;
    const int rr = E * (r % G), kc = r / G;
    T acc[E];
#pragma unroll
    for (int i = 0; i < E; i++) acc[i] = 0;
    if (rr < nr) {
        const T *rows = coef + S.cblk_coef[c] + it.r0 + rr;
#pragma unroll 2
        for (int k = q * E + kc; k < Kc; k += NW * E) {
            T a[E];
            ld_rows(rows + (int64_t)k * ld, rr, nr, a);
#pragma unroll
            for (int i = 0; i < E; i++) acc[i] += a[i] * xs[k];
        }
    }
    const int dst = (r < nr) ? ydst[it.slot + r] : 0;
    wave_sum_store_rows<T, NW, E>(acc, red, r, q, r < nr, ybuf + dst);
}

// one strip (panel rows [r0, r1), any multiple of 64 of them, column block
// blockIdx.y) of the backward products, 4 waves: partial[j] = sum over the
// strip's rows of L[r, k0+j] x[row(r)], 64 rows at a time, the next chunk's
// loads in flight while the current one is summed
template <typename T>
__global__ __launch_bounds__(256) void k_bwd_prod(DevSymbol S, const BwdItem *__restrict__ items, int nitems,
                                                  const T *__restrict__ coef, const T *__restrict__ x,
                                                  T *__restrict__ part) {
    __shared__ T tile[64][65];
    __shared__ T xr[64];
    __shared__ T red[256];
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const BwdItem it = items[id];
    const int k0 = blockIdx.y * 64;
    const int c = it.c;
    const int Kc = S.cblk_fcol[c + 1] - S.cblk_fcol[c];
    if (k0 >= Kc) return;
    const int tid = threadIdx.x, lane = tid & 63, q = tid >> 6;
    const int64_t ld = S.cblk_stride[c];
    const int64_t rb = S.cblk_rowbase[c];
    // E consecutive rows per lane (one 16-byte load), 4E columns per pass
    constexpr int E = Vec<T>::E, G = 64 / E, NP = 64 / (4 * E);
    const int rr = E * (lane % G), kc = lane / G;
    const T *P = coef + S.cblk_coef[c];
    T a[NP][E], xv = 0;
    auto gload = [&](int r0) {
        const int nr = min(64, it.r1 - r0);
#pragma unroll
        for (int u = 0; u < NP; u++) {
            const int cc = q * E + kc + 4 * E * u;
            ld_rows(P + r0 + rr + (int64_t)(k0 + cc) * ld, rr, (k0 + cc < Kc) ? nr : 0, a[u]);
        }
        if (tid < 64) xv = (tid < nr) ? x[S.panel_grow[rb + r0 + tid]] : (T)0;
    };
    T acc = 0;
    gload(it.r0);
    for (int r0 = it.r0; r0 < it.r1; r0 += 64) {
        // the chunk in registers goes to LDS, the next one is fetched
#pragma unroll
        for (int u = 0; u < NP; u++) {
            const int cc = q * E + kc + 4 * E * u;
#pragma unroll
            for (int i = 0; i < E; i++) tile[rr + i][cc] = a[u][i];
        }
        if (tid < 64) xr[tid] = xv;
        __syncthreads();
        if (r0 + 64 < it.r1) gload(r0 + 64);
#pragma unroll 4
        for (int row = q * 16; row < q * 16 + 16; row++) acc += tile[row][lane] * xr[row];
        __syncthreads();
    }
    wave_sum_store<T, 4>(acc, red, lane, q, k0 + lane < Kc, part + (int64_t)it.slot + k0 + lane);
}

template <typename T, int NW>
__global__ __launch_bounds__(NW * 64) void k_bwd_diag(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                      const BwdItem *__restrict__ bitems, const T *__restrict__ z,
                                                      T *__restrict__ x, const T *__restrict__ part,
                                                      const T *__restrict__ wb) {
    extern __shared__ char smem_raw[];
    T *y = reinterpret_cast<T *>(smem_raw);
    __shared__ T red[NW * 64];
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const DiagItem it = items[id];
    const int tid = threadIdx.x, r = tid & 63, q = tid >> 6;
    const int nd = it.nd, r0 = it.ib * 64;
    const int cb0 = S.node_cblk[nd], cb1 = S.node_cblk[nd + 1];
    const int fc = S.cblk_fcol[cb0];
    const int Kc = S.cblk_fcol[cb1] - fc;
    // y = z_c - the strips' partials for columns [r0, Kc): all columns at
    // once (cpp per pass), each summed over every L-th strip by L threads,
    // whose sums are then added in thread order; one barrier pair per pass.
    // Column k of the node belongs to member cblk m (column k - o of it, o
    // = fcol[m] - fc); m's strips [tb, te) own consecutive partial slots, w
    // apart, the first at bitems[tb].slot.
    const int ncol = Kc - r0;
    const int cpp = max(1, min(ncol, NW * 64)), L = (NW * 64) / cpp;
    for (int c0 = 0; c0 < ncol; c0 += cpp) {
        const int cc = tid % cpp, h = tid / cpp;
        const int k = r0 + c0 + cc;
        T acc = 0;
        if (h < L && c0 + cc < ncol) {
            int lo = cb0, hi = cb1 - 1;  // the last member whose first column is <= k
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (S.cblk_fcol[mid] - fc <= k) lo = mid;
                else hi = mid - 1;
            }
            const int o = S.cblk_fcol[lo] - fc, w = S.cblk_fcol[lo + 1] - S.cblk_fcol[lo];
            const int tb = S.cblk_btile[2 * lo], te = S.cblk_btile[2 * lo + 1];
            const T *p0 = part + ((te > tb) ? (int64_t)bitems[tb].slot : 0) + (k - o);
#pragma unroll 4
            for (int j = tb + h; j < te; j += L) acc += p0[(int64_t)(j - tb) * w];
        }
        if (h < L) red[h * cpp + cc] = acc;
        __syncthreads();
        if (h == 0 && c0 + cc < ncol) {
            T v = red[cc];
            for (int w = 1; w < L; w++) v += red[w * cpp + cc];
            y[k] = z[fc + k] - v;
        }
        __syncthreads();
    }
    const int i = r0 + r;
    // rows of the inverse: E consecutive per lane (16-byte loads)
    constexpr int E = Vec<T>::E, G = 64 / E;
    const int rr = E * (r % G), kc = r / G;
    T acc2[E];
#pragma unroll
    for (int e = 0; e < E; e++) acc2[e] = 0;
    if (r0 + rr < Kc) {
        // wb holds inv(L_cc)^T (or inv(U_cc)) column-major: upper triangular
        const T *M = wb + S.node_winv[nd] + r0 + rr;
#pragma unroll 4
        for (int k = r0 + q * E + kc; k < Kc; k += NW * E) {
            T m[E];
            ld_rows(M + (int64_t)k * Kc, rr, Kc - r0, m);
#pragma unroll
            for (int e = 0; e < E; e++) acc2[e] += m[e] * y[k];
        }
    }
    wave_sum_store_rows<T, NW, E>(acc2, red, r, q, i < Kc, x + fc + i);
}

// Backward strips of narrow cblks (at most C columns), one right-hand side:
// four strips per wave, 16 lanes each; lane l sums rows l, l + 16, ... of
// every column in registers, the 16 lanes combine by xor shuffles, lane j
// stores column j.
template <typename T, int C>
__global__ __launch_bounds__(64) void k_bwd_prod_narrow(DevSymbol S, const BwdItem *__restrict__ items, int nitems,
                                                        const T *__restrict__ coef, const T *__restrict__ x,
                                                        T *__restrict__ part) {
    const int lane = threadIdx.x, grp = lane >> 4, l = lane & 15;
    const int id = xcd_remap(blockIdx.x, gridDim.x) * 4 + grp;
    BwdItem it{0, 0, 0, 0};
    int Kc = 0;
    int64_t ld = 0, rb = 0;
    const T *P = coef;
    if (id < nitems) {
        it = items[id];
        Kc = S.cblk_fcol[it.c + 1] - S.cblk_fcol[it.c];
        ld = S.cblk_stride[it.c];
        rb = S.cblk_rowbase[it.c];
        P = coef + S.cblk_coef[it.c];
    }
    T acc[C];
#pragma unroll
    for (int k = 0; k < C; k++) acc[k] = 0;
    for (int r = it.r0 + l; r < it.r1; r += 16) {
        const T xr = x[S.panel_grow[rb + r]];
#pragma unroll
        for (int k = 0; k < C; k++)
            if (k < Kc) acc[k] += P[r + (int64_t)k * ld] * xr;
    }
#pragma unroll
    for (int off = 1; off < 16; off *= 2)
#pragma unroll
        for (int k = 0; k < C; k++) acc[k] += __shfl_xor(acc[k], off);
    // lane j of the group stores columns j, j + 16, ...
#pragma unroll
    for (int k = 0; k < C; k++)
        if ((k & 15) == l && k < Kc) part[(int64_t)it.slot + k] = acc[k];
}

// Levels of wide nodes (more than SOLVE_SPLIT columns): the gathers run once
// per 64-row block in a launch of their own instead of in every diagonal
// workgroup that needs the rows (workgroup ib needs rows [0, 64 ib + 64)).
// Forward: b minus the rows' update-buffer entries, in place in b; wave q
// sums the entries q, q + 4, ... of the block's rows (lane = row, so the
// sliced buffer's loads are contiguous), the waves combined in order.  One
// right-hand side per grid row.
template <typename T>
__global__ __launch_bounds__(256) void k_fwd_gather(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                    const YSlices ys, const T *__restrict__ ybuf, int64_t ldy,
                                                    T *__restrict__ b, int64_t ldb) {
    __shared__ T red[4][64];
    const int tid = threadIdx.x, lane = tid & 63, q = tid >> 6;
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const int u = blockIdx.y;
    const DiagItem it = items[id];
    const int fc = S.cblk_fcol[S.node_cblk[it.nd]];
    const int K = S.cblk_fcol[S.node_cblk[it.nd + 1]] - fc;
    const int i = it.ib * 64 + lane;
    constexpr int UL = 8;
    T v = 0;
    if (i < K) {
        const int g = fc + i, ne = ys.cnt[g];
        const T *yb = ybuf + u * ldy + ys.base[g >> 6] + (g & 63);
        for (int e = q; e < ne; e += 4 * UL) {
            T a[UL];
#pragma unroll
            for (int k = 0; k < UL; k++) a[k] = (e + 4 * k < ne) ? yb[(int64_t)(e + 4 * k) * 64] : (T)0;
#pragma unroll
            for (int k = 0; k < UL; k++) v += a[k];
        }
    }
    red[q][lane] = v;
    __syncthreads();
    if (q == 0 && i < K) b[fc + i + u * ldb] -= ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

// Backward: z minus the strips' partials of the block's columns, in place in
// z; wave q sums the strips q, q + 4, ... of each column's member (lane =
// column), the waves combined in order.
template <typename T>
__global__ __launch_bounds__(256) void k_bwd_reduce(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                    const BwdItem *__restrict__ bitems, T *__restrict__ z,
                                                    int64_t ldz, const T *__restrict__ part, int nrhs_tot) {
    __shared__ T red[4][64];
    const int tid = threadIdx.x, lane = tid & 63, q = tid >> 6;
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const int u = blockIdx.y;
    const DiagItem it = items[id];
    const int cb0 = S.node_cblk[it.nd], cb1 = S.node_cblk[it.nd + 1];
    const int fc = S.cblk_fcol[cb0];
    const int K = S.cblk_fcol[cb1] - fc;
    const int k = it.ib * 64 + lane;
    T v = 0;
    if (k < K) {
        int lo = cb0, hi = cb1 - 1;  // the last member whose first column is <= k
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (S.cblk_fcol[mid] - fc <= k) lo = mid;
            else hi = mid - 1;
        }
        const int o = S.cblk_fcol[lo] - fc, w = S.cblk_fcol[lo + 1] - S.cblk_fcol[lo];
        const int tb = S.cblk_btile[2 * lo], te = S.cblk_btile[2 * lo + 1];
        if (te > tb) {
            const int64_t stride = (int64_t)w * nrhs_tot;
            const T *p0 = part + (int64_t)bitems[tb].slot * nrhs_tot + (int64_t)u * w + (k - o);
            for (int j = q; j < te - tb; j += 4) v += p0[(int64_t)j * stride];
        }
    }
    red[q][lane] = v;
    __syncthreads();
    if (q == 0 && k < K) z[fc + k + u * ldz] -= ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

// Wide levels, one right-hand side, after the gathers: the diagonal GEMV on
// 16-row blocks (four workgroups per 64-row item), so that a node's inverse
// is read by four times as many compute units.  Forward (UPPER false): rows
// [r, r+16) of z = W y, y = b's node rows (already gathered), columns [0,
// r+16); backward (UPPER true): rows of x = WB y, y = z's node rows,
// columns [r, K).  Thread t keeps E consecutive rows (16-byte loads) and the
// columns c, c + 64/... of its column phase; the phases combine through LDS
// in a fixed order.
template <typename T, bool UPPER>
__global__ __launch_bounds__(256) void k_diag_gemv16(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                     const T *__restrict__ src, T *__restrict__ dst,
                                                     const T *__restrict__ w) {
    constexpr int E = Vec<T>::E, RL = 16 / E, NC = 256 / RL;  // lanes per column, column phases
    extern __shared__ char smem_raw[];
    T *y = reinterpret_cast<T *>(smem_raw);
    __shared__ T red[NC][17];
    const int tid = threadIdx.x;
    // forward: the blocks with the most columns (the last rows of a node)
    // take the lowest workgroup ids, so that they start first
    const int g0 = xcd_remap(blockIdx.x, gridDim.x);
    const int gid = UPPER ? g0 : (int)gridDim.x - 1 - g0;
    const int id = gid >> 2, sub = gid & 3;
    if (id >= nitems) return;
    const DiagItem it = items[id];
    const int fc = S.cblk_fcol[S.node_cblk[it.nd]];
    const int K = S.cblk_fcol[S.node_cblk[it.nd + 1]] - fc;
    const int r = it.ib * 64 + sub * 16;
    if (r >= K) return;  // uniform: the whole workgroup leaves
    const int nr = min(16, K - r);
    const int k0 = UPPER ? r : 0, k1 = UPPER ? K : min(K, r + 16);
    for (int k = k0 + tid; k < k1; k += 256) y[k - k0] = src[fc + k];
    __syncthreads();
    const int rr = E * (tid % RL), c = tid / RL;
    const T *M = w + S.node_winv[it.nd] + r + rr;
    T acc[E];
#pragma unroll
    for (int e = 0; e < E; e++) acc[e] = 0;
#pragma unroll 4
    for (int k = k0 + c; k < k1; k += NC) {
        T m[E];
        ld_rows(M + (int64_t)k * K, rr, nr, m);
        const T yv = y[k - k0];
#pragma unroll
        for (int e = 0; e < E; e++) acc[e] += m[e] * yv;
    }
#pragma unroll
    for (int e = 0; e < E; e++) red[c][rr + e] = acc[e];
    __syncthreads();
    if (tid < nr) {
        T v = red[0][tid];
        for (int q = 1; q < NC; q++) v += red[q][tid];
        dst[fc + r + tid] = v;
    }
}

// Forward, LL^t, one right-hand side, after the gathers: rows [r, r+16) of
// z = W y as dot products down columns r..r+15 of WT = W^T (the backward
// inverse): row i of W is column i of WT, one contiguous run, so a block
// reads 16 adjacent columns instead of 16 rows strided across the whole
// inverse (FP64 80^3: 305 -> 175 us per solve).  Sixteen lanes per output
// row, E consecutive k per lane (16-byte loads); the lanes' sums combine by
// xor shuffles in a fixed order.  (The same form for the backward GEMV,
// down the columns of the forward inverse, was slower: 178 against 150 us.)
template <typename T>
__global__ __launch_bounds__(256) void k_fwd_gemv16t(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                     const T *__restrict__ src, T *__restrict__ dst,
                                                     const T *__restrict__ wt) {
    constexpr int E = Vec<T>::E;
    extern __shared__ char smem_raw[];
    T *y = reinterpret_cast<T *>(smem_raw);
    const int tid = threadIdx.x;
    // the blocks with the most columns (the last rows of a node) take the
    // lowest workgroup ids, so that they start first
    const int gid = (int)gridDim.x - 1 - xcd_remap(blockIdx.x, gridDim.x);
    const int id = gid >> 2, sub = gid & 3;
    if (id >= nitems) return;
    const DiagItem it = items[id];
    const int fc = S.cblk_fcol[S.node_cblk[it.nd]];
    const int K = S.cblk_fcol[S.node_cblk[it.nd + 1]] - fc;
    const int r = it.ib * 64 + sub * 16;
    if (r >= K) return;  // uniform: the whole workgroup leaves
    const int k1 = min(K, r + 16);
    for (int k = tid; k < k1; k += 256) y[k] = src[fc + k];
    __syncthreads();
    const int j = tid >> 4, l = tid & 15;
    const int i = r + j;  // output row; W[i, k] = WT[k, i] is nonzero for k <= i
    T acc = 0;
    if (i < K) {
        const T *col = wt + S.node_winv[it.nd] + (int64_t)i * K;
        T a2[E];
#pragma unroll
        for (int e = 0; e < E; e++) a2[e] = 0;
#pragma unroll 4
        for (int k = E * l; k <= i; k += 16 * E) {
            T m[E];
            ld_rows(col + k, k, i + 1, m);
#pragma unroll
            for (int e = 0; e < E; e++) a2[e] += m[e] * y[min(k + e, i)];
        }
#pragma unroll
        for (int e = 0; e < E; e++) acc += a2[e];
    }
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 16);
    if (l == 0 && i < K) dst[fc + i] = acc;
}

// Levels of narrow nodes (at most SOLVE_TINY columns), one right-hand side:
// four nodes per wave, 16 lanes each, lane i owning row (forward) or column
// (backward) i of its node; the node's inverse is read into registers
// before the gathers, the product takes y by lane shuffles.
template <typename T>
__global__ __launch_bounds__(64) void k_fwd_diag_tiny(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                      const YSlices ys, const T *__restrict__ ybuf,
                                                      const T *__restrict__ b, T *__restrict__ z,
                                                      const T *__restrict__ w1) {
    const int lane = threadIdx.x, grp = lane >> 4, i = lane & 15;
    const int id = xcd_remap(blockIdx.x, gridDim.x) * 4 + grp;
    int fc = 0, K = 0;
    int64_t wo = 0;
    if (id < nitems) {
        const int nd = items[id].nd;
        fc = S.cblk_fcol[S.node_cblk[nd]];
        K = S.cblk_fcol[S.node_cblk[nd + 1]] - fc;
        wo = S.node_winv[nd];
    }
    const bool row = i < K;
    T wv[16];
#pragma unroll
    for (int k = 0; k < 16; k++) wv[k] = (row && k < K) ? w1[wo + i + (int64_t)k * K] : (T)0;
    T y = 0;
    if (row) {
        const int g = fc + i, ne = ys.cnt[g];
        const T *yb = ybuf + ys.base[g >> 6] + (g & 63);
        T v = 0;
        for (int e = 0; e < ne; e += 8) {
            T a[8];
#pragma unroll
            for (int k = 0; k < 8; k++) a[k] = (e + k < ne) ? yb[(int64_t)(e + k) * 64] : (T)0;
#pragma unroll
            for (int k = 0; k < 8; k++) v += a[k];
        }
        y = b[g] - v;
    }
    T acc = 0;
#pragma unroll
    for (int k = 0; k < 16; k++) acc += wv[k] * __shfl(y, (grp << 4) + k);
    if (row) z[fc + i] = acc;
}

template <typename T>
__global__ __launch_bounds__(64) void k_bwd_diag_tiny(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                      const BwdItem *__restrict__ bitems, const T *__restrict__ z,
                                                      T *__restrict__ x, const T *__restrict__ part,
                                                      const T *__restrict__ wb) {
    const int lane = threadIdx.x, grp = lane >> 4, k = lane & 15;
    const int id = xcd_remap(blockIdx.x, gridDim.x) * 4 + grp;
    int fc = 0, K = 0, cb0 = 0, cb1 = 0;
    int64_t wo = 0;
    if (id < nitems) {
        const int nd = items[id].nd;
        cb0 = S.node_cblk[nd];
        cb1 = S.node_cblk[nd + 1];
        fc = S.cblk_fcol[cb0];
        K = S.cblk_fcol[cb1] - fc;
        wo = S.node_winv[nd];
    }
    const bool col = k < K;
    // row k of inv(L_nd)^T: WB[k + j*K], j >= k
    T wv[16];
#pragma unroll
    for (int j = 0; j < 16; j++) wv[j] = (col && j < K) ? wb[wo + k + (int64_t)j * K] : (T)0;
    T y = 0;
    if (col) {
        // member m of column k, its strips' partials (consecutive slots, w apart)
        int m = cb0;
        while (m + 1 < cb1 && S.cblk_fcol[m + 1] - fc <= k) m++;
        const int o = S.cblk_fcol[m] - fc, w = S.cblk_fcol[m + 1] - S.cblk_fcol[m];
        const int tb = S.cblk_btile[2 * m], te = S.cblk_btile[2 * m + 1];
        T v = 0;
        if (te > tb) {
            const T *pp = part + (int64_t)bitems[tb].slot + (k - o);
            for (int j = 0; j < te - tb; j++) v += pp[(int64_t)j * w];
        }
        y = z[fc + k] - v;
    }
    T acc = 0;
#pragma unroll
    for (int j = 0; j < 16; j++) acc += wv[j] * __shfl(y, (grp << 4) + j);
    if (col) x[fc + k] = acc;
}

// ---------------------------------------------------------------------------
// Several right-hand sides: the same sweeps as products on the matrix cores,
// sixteen right-hand sides to an MFMA block and NB blocks to a workgroup, so
// that a panel crosses once for up to 16 NB of them (a node's inverse once for
// up to 16).  Bound by the levels' memory latency (a 53x47x50 factor is 0.46
// GB).  The vector kernels these replace took two (diagonal steps) or eight
// columns at a time and read the factor again for the next ones: 53x47x50
// FP64, 2 columns 1165 -> 847 us, 8 1484 -> 917, 32 3212 -> 1267; FP32 867 ->
// 601, 1154 -> 655, 2477 -> 904.
//
// The vector kernels' sums were spread over up to 64 lanes and waves.  To
// round as little, an accumulator takes no chain of MFMAs longer than sixteen
// inner indices (four in the diagonal steps of narrow nodes): each is summed
// from zero and then added.  Residuals of 2 to 64 right-hand sides over the
// vector kernels' (LL^t, LDL^t and LU of 2D and 3D grids), mean and largest:
// with 64 rows, 32 or 64 indices of a wide inverse and all of a narrow one to
// a chain 1.06 and 1.11 in FP64, 1.08 and 1.15 in FP32; so 0.985 and 0.993,
// 0.988 and 0.996, for 0.7 % of the time of 32 columns.
//
// Products are formed transposed, D(u, row) = sum_k Y(k, u) M(row, k): a lane's results of one
// MFMA register belong to one right-hand side, so sixteen lanes store
// consecutive rows.  Rows and right-hand sides that do not exist repeat an
// existing one (their results are not stored); inner indices beyond the last
// count as zero on both operands.
// ---------------------------------------------------------------------------

// Forward products: 64 panel rows x K columns of cblk c times z_c.  Lanes
// read E consecutive rows of a column (16 bytes); a wave covers 16 E rows,
// the remaining split of the four waves goes over the columns (KS ways,
// combined through LDS in a fixed order).  z_c is staged KC columns at a time.
// Held to 152 registers, three waves per SIMD (with the sums of all groups
// side by side 204, two): 32 columns, FP64 53x47x50, whole solve 1.41 -> 1.25
// ms.
template <typename T, int NB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_fwd_prod_m(DevSymbol S, const FwdItem *__restrict__ items, int nitems,
                                                    const T *__restrict__ coef, const T *__restrict__ z, int64_t ldz,
                                                    int nrhs, const int32_t *__restrict__ ydst,
                                                    T *__restrict__ ybuf, int64_t ldy) {
    constexpr int E = Vec<T>::E, WR = 4 / E, KS = 4 / WR, KC = 128, NC = 16 * NB, ZP = KC + 2;
    constexpr int ZN = NC * ZP, RN = KS * NC * 64;
    __shared__ T lds[ZN > RN ? ZN : RN];
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const FwdItem it = items[id];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, kq = lane >> 4, wr = wave % WR, ks = wave / WR;
    const int u0 = NC * blockIdx.y, nu = min(NC, nrhs - u0);
    const int fc = S.cblk_fcol[it.c], K = S.cblk_fcol[it.c + 1] - fc;
    const int64_t ld = S.cblk_stride[it.c];
    const int nr = it.r1 - it.r0, row = 16 * E * wr + E * i;
    const T *P = coef + S.cblk_coef[it.c] + it.r0 + (row < nr ? row : 0);
    typename Mfma<T>::v4 acc[E][NB];
#pragma unroll
    for (int e = 0; e < E; e++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[e][b] = {0, 0, 0, 0};
    // thread (k, group) stages right-hand sides group, group + 2, ... of
    // column k of the chunk; the next chunk's are in flight during the MFMAs
    const int zk = tid & (KC - 1), zu = tid / KC;
    T v[NC / 2];
    auto zload = [&](int kc) {
        const T *q = z + fc + min(kc + zk, K - 1) + (int64_t)u0 * ldz;
#pragma unroll
        for (int t = 0; t < NC / 2; t++) v[t] = q[(int64_t)min(zu + 2 * t, nu - 1) * ldz];
    };
    zload(0);
    for (int kc = 0; kc < K; kc += KC) {
        const int kn = min(KC, K - kc);
        if (kc > 0) __syncthreads();
#pragma unroll
        for (int t = 0; t < NC / 2; t++) lds[(zu + 2 * t) * ZP + zk] = (zk < kn) ? v[t] : (T)0;
        __syncthreads();
        if (kc + KC < K) zload(kc + KC);
        // four steps' factor loads together, then their MFMAs, summed from
        // zero: one chain over all columns rounded at the whole sum's size
        // each time (residuals of 32 right-hand sides up to 13 % larger).
        // One group of right-hand sides after the other, so that only its
        // sums are live beside the accumulators
        for (int s0 = 4 * ks; s0 < kn; s0 += 16 * KS) {
            T m[4][E];
#pragma unroll
            for (int j = 0; j < 4; j++) ld_vec(P + (int64_t)(kc + min(s0 + 4 * KS * j + kq, kn - 1)) * ld, m[j]);
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int e = 0; e < E; e++) m[j][e] = (s0 + 4 * KS * j + kq < kn) ? m[j][e] : (T)0;
#pragma unroll
            for (int b = 0; b < NB; b++) {
                typename Mfma<T>::v4 p[E];
#pragma unroll
                for (int e = 0; e < E; e++) p[e] = {0, 0, 0, 0};
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int s = s0 + 4 * KS * j;
                    if (s >= kn) break;  // uniform
                    const T a = lds[(16 * b + i) * ZP + s + kq];
#pragma unroll
                    for (int e = 0; e < E; e++) p[e] = Mfma<T>::mma(a, m[j][e], p[e]);
                }
#pragma unroll
                for (int e = 0; e < E; e++) acc[e][b] += p[e];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; e++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                lds[(ks * NC + 16 * b + Mfma<T>::drow(lane, r)) * 64 + row + e] = acc[e][b][r];
    __syncthreads();
    const int rl = tid & 63;
    if (rl < nr) {
        T *out = ybuf + ydst[it.slot + rl] + (int64_t)u0 * ldy;
        for (int u = tid >> 6; u < nu; u += 4) {
            T v = lds[u * 64 + rl];
#pragma unroll
            for (int q = 1; q < KS; q++) v += lds[(q * NC + u) * 64 + rl];
            out[(int64_t)u * ldy] = v;
        }
    }
}

// Backward products: columns [k0, k0 + 16 WC) of cblk c, panel rows of one
// strip: partial(u, j) = sum_r L(r, j) x(row(r), u).  A lane reads E
// consecutive rows of its column (16 bytes, four lanes to a column); a wave
// takes 16 columns, the waves left over (4 / WC ways, levels of narrow cblks)
// split the rows and combine through LDS in a fixed order.  x is gathered 64
// rows at a time.
template <typename T, int NB, int WC>
__global__ __launch_bounds__(256) void k_bwd_prod_m(DevSymbol S, const BwdItem *__restrict__ items, int nitems,
                                                    const T *__restrict__ coef, const T *__restrict__ x, int64_t ldx,
                                                    int nrhs, T *__restrict__ part) {
    constexpr int E = Vec<T>::E, RS = 4 / WC, NC = 16 * NB, XP = 64 + E, RR = 64 / RS, NG = RR / (4 * E);
    constexpr int XN = NC * XP, RN = RS > 1 ? RS * WC * 16 * NC : 0;
    __shared__ T lds[XN > RN ? XN : RN];
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const BwdItem it = items[id];
    const int fc = S.cblk_fcol[it.c], K = S.cblk_fcol[it.c + 1] - fc;
    const int k0 = blockIdx.y * 16 * WC;
    if (k0 >= K) return;  // uniform: the whole workgroup leaves
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, kq = lane >> 4, wc = wave % WC, rs = wave / WC;
    const int u0 = NC * blockIdx.z, nu = min(NC, nrhs - u0);
    const int64_t ld = S.cblk_stride[it.c];
    const int32_t *grow = S.panel_grow + S.cblk_rowbase[it.c];
    const bool live = k0 + 16 * wc < K;
    const int col = k0 + 16 * wc + i;
    const T *P = coef + S.cblk_coef[it.c] + (int64_t)min(col, K - 1) * ld;
    typename Mfma<T>::v4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) acc[b] = {0, 0, 0, 0};
    // thread (row, group) gathers right-hand sides group, group + 4, ... of
    // its row of the chunk; the next chunk's are in flight during the MFMAs
    const int xr = tid & 63, xu = tid >> 6;
    T v[NC / 4];
    int gr = grow[min(it.r0 + xr, it.r1 - 1)];
    auto xload = [&]() {
        const T *xg = x + gr + (int64_t)u0 * ldx;
#pragma unroll
        for (int t = 0; t < NC / 4; t++) v[t] = xg[(int64_t)min(xu + 4 * t, nu - 1) * ldx];
    };
    xload();
    for (int r0 = it.r0; r0 < it.r1; r0 += 64) {
        const int rn = min(64, it.r1 - r0);
        const bool more = r0 + 64 < it.r1;
        if (more) gr = grow[min(r0 + 64 + xr, it.r1 - 1)];
        T m[NG][E];
        if (live) {
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const int r = RR * rs + 4 * E * g + E * kq;
                ld_vec(P + r0 + (r < rn ? r : 0), m[g]);
            }
        }
        if (r0 > it.r0) __syncthreads();
#pragma unroll
        for (int t = 0; t < NC / 4; t++) lds[(xu + 4 * t) * XP + xr] = (xr < rn) ? v[t] : (T)0;
        __syncthreads();
        if (more) xload();
        if (live) {
            constexpr int GS = 4 / E;  // groups of 16 rows
            typename Mfma<T>::v4 p[NB];
#pragma unroll
            for (int g = 0; g < NG; g++) {
                if (g % GS == 0)
#pragma unroll
                    for (int b = 0; b < NB; b++) p[b] = {0, 0, 0, 0};
#pragma unroll
                for (int e = 0; e < E; e++) m[g][e] = (RR * rs + 4 * E * g + E * kq + e < rn) ? m[g][e] : (T)0;
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    const T *a = &lds[(16 * b + i) * XP + RR * rs + 4 * E * g + E * kq];
#pragma unroll
                    for (int e = 0; e < E; e++) p[b] = Mfma<T>::mma(a[e], m[g][e], p[b]);
                }
                if (g % GS == GS - 1)
#pragma unroll
                    for (int b = 0; b < NB; b++) acc[b] += p[b];
            }
        }
    }
    T *out = part + (int64_t)it.slot * nrhs + (int64_t)u0 * K;
    if constexpr (RS == 1) {
        if (col < K) {
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int u = 16 * b + Mfma<T>::drow(lane, r);
                    if (u < nu) out[(int64_t)u * K + col] = acc[b][r];
                }
        }
    } else {
        __syncthreads();
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                lds[(rs * NC + 16 * b + Mfma<T>::drow(lane, r)) * (16 * WC) + 16 * wc + i] = acc[b][r];
        __syncthreads();
        for (int t = tid; t < 16 * WC * NC; t += 256) {
            const int j = t % (16 * WC), u = t / (16 * WC);
            if (k0 + j < K && u < nu) {
                T w = lds[t];
#pragma unroll
                for (int q = 1; q < RS; q++) w += lds[q * NC * 16 * WC + t];
                out[(int64_t)u * K + k0 + j] = w;
            }
        }
    }
}

// Diagonal steps of nodes of at most 16 W columns: one workgroup of W waves
// per node, 16 rows of the node's inverse to a wave (read into registers
// before the gather), Y staged in LDS.  Forward (UPPER false): Y = b minus the
// rows' update-buffer entries, z = W Y; backward: Y = z minus the strips'
// partials, x = WB Y.
template <typename T, int NB, int W, bool UPPER>
__global__ __launch_bounds__(64 * W) void k_diag_narrow_m(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                          const YSlices ys, const BwdItem *__restrict__ bitems,
                                                          const T *__restrict__ pend, int64_t ldp,
                                                          const T *__restrict__ src, int64_t lds_, T *__restrict__ dst,
                                                          int64_t ldd, int nrhs, const T *__restrict__ inv) {
    constexpr int NC = 16 * NB, KM = 16 * W, YP = KM + 2;
    __shared__ T y[NC][YP];
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, kq = lane >> 4;
    const int u0 = NC * blockIdx.y, nu = min(NC, nrhs - u0);
    const int nd = items[id].nd, cb0 = S.node_cblk[nd], cb1 = S.node_cblk[nd + 1];
    const int fc = S.cblk_fcol[cb0], K = S.cblk_fcol[cb1] - fc;
    // this wave's rows of the inverse, the nonzero side of the diagonal
    const int ro = 16 * wave;
    const int s0 = UPPER ? 4 * wave : 0, s1 = UPPER ? 4 * W : 4 * wave + 4;
    const T *M = inv + S.node_winv[nd] + min(ro + i, K - 1);
    T m[4 * W];
#pragma unroll
    for (int s = 0; s < 4 * W; s++) {
        const int k = 4 * s + kq;
        m[s] = (s >= s0 && s < s1 && k < K) ? M[(int64_t)k * K] : (T)0;
    }
    // Y: thread (row, group) takes right-hand sides group, group + 4, ...
    const int row = tid % KM, ug = tid / KM;
    T v[NC / 4];
#pragma unroll
    for (int t = 0; t < NC / 4; t++) v[t] = 0;
    if (row < K) {
        int ne;
        int64_t step, ldu;
        const T *p;
        if constexpr (!UPPER) {
            const int g = fc + row;
            ne = ys.cnt[g];
            step = 64;
            ldu = ldp;
            p = pend + ys.base[g >> 6] + (g & 63) + (int64_t)u0 * ldp;
        } else {
            // member of the column, its strips' partials
            int c = cb0;
            while (c + 1 < cb1 && S.cblk_fcol[c + 1] - fc <= row) c++;
            const int o = S.cblk_fcol[c] - fc, w = S.cblk_fcol[c + 1] - S.cblk_fcol[c];
            const int tb = S.cblk_btile[2 * c];
            ne = S.cblk_btile[2 * c + 1] - tb;
            step = (int64_t)w * nrhs;
            ldu = w;
            p = pend + (ne > 0 ? (int64_t)bitems[tb].slot * nrhs : 0) + (int64_t)u0 * w + (row - o);
        }
        const T *q = src + fc + row + (int64_t)u0 * lds_;
        T b[NC / 4];
#pragma unroll
        for (int t = 0; t < NC / 4; t++) b[t] = (ug + 4 * t < nu) ? q[(int64_t)(ug + 4 * t) * lds_] : (T)0;
        // two entries' loads together, added in order (a right-hand side
        // beyond the last repeats it: its sum is not used)
        for (int e = 0; e < ne; e += 2) {
            T a0[NC / 4], a1[NC / 4];
            const T *p0 = p + (int64_t)e * step, *p1 = p + (int64_t)min(e + 1, ne - 1) * step;
#pragma unroll
            for (int t = 0; t < NC / 4; t++) {
                const int64_t uo = (int64_t)min(ug + 4 * t, nu - 1) * ldu;
                a0[t] = p0[uo];
                a1[t] = p1[uo];
            }
#pragma unroll
            for (int t = 0; t < NC / 4; t++) {
                v[t] += a0[t];
                v[t] += (e + 1 < ne) ? a1[t] : (T)0;
            }
        }
#pragma unroll
        for (int t = 0; t < NC / 4; t++) v[t] = (ug + 4 * t < nu) ? b[t] - v[t] : (T)0;
    }
#pragma unroll
    for (int t = 0; t < NC / 4; t++) y[ug + 4 * t][row] = v[t];
    __syncthreads();
    if (ro >= K) return;
    typename Mfma<T>::v4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) acc[b] = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4 * W; s += 2) {
        if (s >= s0 && s < s1) {  // uniform in the wave
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const typename Mfma<T>::v4 zero = {0, 0, 0, 0};
                acc[b] += Mfma<T>::mma(y[16 * b + i][4 * s + kq], m[s], zero) +
                          Mfma<T>::mma(y[16 * b + i][4 * s + 4 + kq], m[s + 1], zero);
            }
        }
    }
    if (ro + i < K) {
        T *out = dst + fc + ro + i + (int64_t)u0 * ldd;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int u = 16 * b + Mfma<T>::drow(lane, r);
                if (u < nu) out[(int64_t)u * ldd] = acc[b][r];
            }
    }
}

// Diagonal steps of wider nodes, after the gathers (k_fwd_gather,
// k_bwd_reduce): 16 rows x 16 right-hand sides to a workgroup (four per
// 64-row item), the waves splitting the inner index and combining through
// LDS in wave order.  Forward: z = W y over columns [0, r + 16); backward
// (UPPER): x = WB y over [r, K).  TR: the matrix is given transposed (row i
// at w[i*K ...], one contiguous run), else column-major.
template <typename T, bool UPPER, bool TR>
__global__ __launch_bounds__(256) void k_diag_gemm16(DevSymbol S, const DiagItem *__restrict__ items, int nitems,
                                                     const T *__restrict__ src, int64_t lds_, T *__restrict__ dst,
                                                     int64_t ldd, int nrhs, const T *__restrict__ w) {
    constexpr int E = Vec<T>::E, G = 4 * E;
    __shared__ T red[4][16][17];
    // forward: the blocks with the most columns (the last rows of a node)
    // take the lowest workgroup ids, so that they start first
    const int g0 = xcd_remap(blockIdx.x, gridDim.x);
    const int gid = UPPER ? g0 : (int)gridDim.x - 1 - g0;
    const int id = gid >> 2, sub = gid & 3;
    if (id >= nitems) return;
    const DiagItem it = items[id];
    const int fc = S.cblk_fcol[S.node_cblk[it.nd]];
    const int K = S.cblk_fcol[S.node_cblk[it.nd + 1]] - fc;
    const int r = it.ib * 64 + sub * 16;
    if (r >= K) return;  // uniform: the whole workgroup leaves
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, kq = lane >> 4;
    const int u0 = 16 * blockIdx.y, nu = min(16, nrhs - u0);
    const int k0 = UPPER ? r : 0, k1 = UPPER ? K : min(K, r + 16);
    const T *Y = src + fc + (int64_t)(u0 + min(i, nu - 1)) * lds_;
    const int64_t mi = min(r + i, K - 1);
    const T *M = w + S.node_winv[it.nd] + (TR ? mi * K : mi);
    typename Mfma<T>::v4 acc = {0, 0, 0, 0};
    constexpr int U = 4;  // groups of G inner indices whose loads go out together
    for (int kb0 = k0 + G * wave; kb0 < k1; kb0 += 4 * U * G) {
        T a[U][E], m[U][E];
#pragma unroll
        for (int j = 0; j < U; j++) {
            const int kb = kb0 + 4 * G * j, k = kb + E * kq;
            if (kb >= k1) break;  // uniform
            if (kb + G <= k1) {
                ld_vec(Y + k, a[j]);
                if constexpr (TR) ld_vec(M + k, m[j]);
                else {
#pragma unroll
                    for (int e = 0; e < E; e++) m[j][e] = M[(int64_t)(k + e) * K];
                }
            } else {
#pragma unroll
                for (int e = 0; e < E; e++) {
                    const bool ok = k + e < k1;
                    const int64_t ke = min(k + e, k1 - 1);
                    const T av = Y[ke], mv = M[TR ? ke : ke * K];
                    a[j][e] = ok ? av : (T)0;
                    m[j][e] = ok ? mv : (T)0;
                }
            }
        }
#pragma unroll
        for (int j0 = 0; j0 < U; j0 += 4 / E) {
            typename Mfma<T>::v4 p = {0, 0, 0, 0};
#pragma unroll
            for (int j = j0; j < j0 + 4 / E; j++) {
                if (kb0 + 4 * G * j >= k1) break;  // uniform
#pragma unroll
                for (int e = 0; e < E; e++) p = Mfma<T>::mma(a[j][e], m[j][e], p);
            }
            acc += p;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) red[wave][Mfma<T>::drow(lane, q)][i] = acc[q];
    __syncthreads();
    const int u = tid >> 4, row = tid & 15;
    if (u < nu && r + row < K)
        dst[fc + r + row + (int64_t)(u0 + u) * ldd] =
            ((red[0][u][row] + red[1][u][row]) + red[2][u][row]) + red[3][u][row];
}

// ------------------------------- launchers ---------------------------------
// NB of the several-right-hand-side kernels: 16 or 32 columns at a time
#define PXA_NB(nrhs, CALL)        \
    do {                          \
        if ((nrhs) <= 16) {       \
            constexpr int NB = 1; \
            CALL;                 \
        } else {                  \
            constexpr int NB = 2; \
            CALL;                 \
        }                         \
    } while (0)

template <typename T, bool UPPER>
static void launch_diag_narrow_m(const DevSymbol &S, const DiagItem *items, int n, const YSlices &ys,
                                 const BwdItem *bitems, const T *pend, int64_t ldp, const T *src, int64_t lds,
                                 T *dst, int64_t ldd, int nrhs, const T *inv, int maxwidth, hipStream_t st) {
    PXA_NB(nrhs, {
        const dim3 g(grid8(n), (nrhs + 16 * NB - 1) / (16 * NB));
        if (maxwidth <= 16)
            hipLaunchKernelGGL((k_diag_narrow_m<T, NB, 1, UPPER>), g, dim3(64), 0, st, S, items, n, ys, bitems, pend,
                               ldp, src, lds, dst, ldd, nrhs, inv);
        else if (maxwidth <= 32)
            hipLaunchKernelGGL((k_diag_narrow_m<T, NB, 2, UPPER>), g, dim3(128), 0, st, S, items, n, ys, bitems, pend,
                               ldp, src, lds, dst, ldd, nrhs, inv);
        else
            hipLaunchKernelGGL((k_diag_narrow_m<T, NB, 4, UPPER>), g, dim3(256), 0, st, S, items, n, ys, bitems, pend,
                               ldp, src, lds, dst, ldd, nrhs, inv);
    });
}

template <typename T>
void launch_fwd_diag(const DevSymbol &S, const DiagItem *items, int n, const YSlices &ys, const T *ybuf,
                     int64_t ldy, T *b, int64_t ldb, T *z, int64_t ldz, int nrhs, const T *w1, const T *w1t,
                     int maxwidth, hipStream_t st) {
    if (n <= 0) return;
    if (nrhs > 1) {
        if (maxwidth <= SOLVE_NARROW) {
            launch_diag_narrow_m<T, false>(S, items, n, ys, nullptr, ybuf, ldy, b, ldb, z, ldz, nrhs, w1, maxwidth, st);
            return;
        }
        hipLaunchKernelGGL(k_fwd_gather<T>, dim3(grid8(n), nrhs), dim3(256), 0, st, S, items, n, ys, ybuf, ldy, b, ldb);
        const dim3 g(grid8(4 * n), (nrhs + 15) / 16);
        if (w1t)
            hipLaunchKernelGGL((k_diag_gemm16<T, false, true>), g, dim3(256), 0, st, S, items, n, (const T *)b, ldb, z,
                               ldz, nrhs, w1t);
        else
            hipLaunchKernelGGL((k_diag_gemm16<T, false, false>), g, dim3(256), 0, st, S, items, n, (const T *)b, ldb,
                               z, ldz, nrhs, w1);
        return;
    }
    if (maxwidth > SOLVE_SPLIT) {
        hipLaunchKernelGGL(k_fwd_gather<T>, dim3(grid8(n), 1), dim3(256), 0, st, S, items, n, ys, ybuf, ldy, b, ldb);
        if (w1t)
            hipLaunchKernelGGL(k_fwd_gemv16t<T>, dim3(grid8(4 * n)), dim3(256), (size_t)maxwidth * sizeof(T), st, S,
                               items, n, (const T *)b, z, w1t);
        else
            hipLaunchKernelGGL((k_diag_gemv16<T, false>), dim3(grid8(4 * n)), dim3(256), (size_t)maxwidth * sizeof(T),
                               st, S, items, n, (const T *)b, z, w1);
        return;
    }
    // levels of narrow cblks (maxwidth = the level's widest) take 4-wave workgroups
    if (maxwidth <= SOLVE_TINY)
        hipLaunchKernelGGL(k_fwd_diag_tiny<T>, dim3(grid8((n + 3) / 4)), dim3(64), 0, st, S, items, n, ys, ybuf, b, z,
                           w1);
    else if (maxwidth <= SOLVE_NARROW)
        hipLaunchKernelGGL((k_fwd_diag<T, 4>), dim3(grid8(n)), dim3(256), (size_t)maxwidth * sizeof(T), st, S, items,
                           n, ys, ybuf, b, z, w1, w1t);
    else
        hipLaunchKernelGGL((k_fwd_diag<T, 16>), dim3(grid8(n)), dim3(1024), (size_t)maxwidth * sizeof(T), st, S,
                           items, n, ys, ybuf, b, z, w1, w1t);
}
template <typename T>
void launch_fwd_prod(const DevSymbol &S, const FwdItem *items, int n, const T *coef, const T *z, int64_t ldz,
                     int nrhs, const int32_t *ydst, T *ybuf, int64_t ldy, int maxwidth, hipStream_t st) {
    if (n <= 0) return;
    if (nrhs > 1)
        PXA_NB(nrhs, hipLaunchKernelGGL((k_fwd_prod_m<T, NB>), dim3(grid8(n), (nrhs + 16 * NB - 1) / (16 * NB)),
                                        dim3(256), 0, st, S, items, n, coef, z, ldz, nrhs, ydst, ybuf, ldy));
    else if (maxwidth <= SOLVE_TINY)
        hipLaunchKernelGGL((k_fwd_prod<T, 1>), dim3(grid8(n)), dim3(64), (size_t)maxwidth * sizeof(T), st, S, items,
                           n, coef, z, ydst, ybuf);
    else if (maxwidth <= SOLVE_NARROW)
        hipLaunchKernelGGL((k_fwd_prod<T, 4>), dim3(grid8(n)), dim3(256), (size_t)maxwidth * sizeof(T), st, S, items,
                           n, coef, z, ydst, ybuf);
    else
        hipLaunchKernelGGL((k_fwd_prod<T, 16>), dim3(grid8(n)), dim3(1024), (size_t)maxwidth * sizeof(T), st, S, items,
                           n, coef, z, ydst, ybuf);
}
template <typename T>
void launch_bwd_prod(const DevSymbol &S, const BwdItem *items, int n, const T *coef, const T *x, int64_t ldx,
                     int nrhs, T *part, int maxwidth, hipStream_t st) {
    if (n <= 0) return;
    if (nrhs > 1) {
        PXA_NB(nrhs, {
            const int gz = (nrhs + 16 * NB - 1) / (16 * NB);
            if (maxwidth <= 16)
                hipLaunchKernelGGL((k_bwd_prod_m<T, NB, 1>), dim3(grid8(n), 1, gz), dim3(256), 0, st, S, items, n,
                                   coef, x, ldx, nrhs, part);
            else if (maxwidth <= 32)
                hipLaunchKernelGGL((k_bwd_prod_m<T, NB, 2>), dim3(grid8(n), 1, gz), dim3(256), 0, st, S, items, n,
                                   coef, x, ldx, nrhs, part);
            else
                hipLaunchKernelGGL((k_bwd_prod_m<T, NB, 4>), dim3(grid8(n), (maxwidth + 63) / 64, gz), dim3(256), 0,
                                   st, S, items, n, coef, x, ldx, nrhs, part);
        });
        return;
    }
    if (maxwidth <= SOLVE_TINY) {
        hipLaunchKernelGGL((k_bwd_prod_narrow<T, SOLVE_TINY>), dim3(grid8((n + 3) / 4)), dim3(64), 0, st, S, items, n,
                           coef, x, part);
        return;
    }
    hipLaunchKernelGGL(k_bwd_prod<T>, dim3(grid8(n), (maxwidth + 63) / 64), dim3(256), 0, st, S, items, n, coef, x,
                       part);
}
template <typename T>
void launch_bwd_diag(const DevSymbol &S, const DiagItem *items, int n, const BwdItem *bitems, T *z,
                     int64_t ldz, T *x, int64_t ldx, int nrhs, const T *part, const T *wb, int maxwidth,
                     hipStream_t st) {
    if (n <= 0) return;
    if (nrhs > 1) {
        if (maxwidth <= SOLVE_NARROW) {
            launch_diag_narrow_m<T, true>(S, items, n, YSlices{}, bitems, part, 0, z, ldz, x, ldx, nrhs, wb, maxwidth,
                                          st);
            return;
        }
        hipLaunchKernelGGL(k_bwd_reduce<T>, dim3(grid8(n), nrhs), dim3(256), 0, st, S, items, n, bitems, z, ldz, part,
                           nrhs);
        hipLaunchKernelGGL((k_diag_gemm16<T, true, false>), dim3(grid8(4 * n), (nrhs + 15) / 16), dim3(256), 0, st, S,
                           items, n, (const T *)z, ldz, x, ldx, nrhs, wb);
        return;
    }
    if (maxwidth > SOLVE_SPLIT) {
        hipLaunchKernelGGL(k_bwd_reduce<T>, dim3(grid8(n), 1), dim3(256), 0, st, S, items, n, bitems, z, ldz, part, 1);
        hipLaunchKernelGGL((k_diag_gemv16<T, true>), dim3(grid8(4 * n)), dim3(256), (size_t)maxwidth * sizeof(T), st,
                           S, items, n, (const T *)z, x, wb);
        return;
    }
    if (maxwidth <= SOLVE_TINY)
        hipLaunchKernelGGL(k_bwd_diag_tiny<T>, dim3(grid8((n + 3) / 4)), dim3(64), 0, st, S, items, n, bitems, z, x,
                           part, wb);
    else if (maxwidth <= SOLVE_NARROW)
        hipLaunchKernelGGL((k_bwd_diag<T, 4>), dim3(grid8(n)), dim3(256), (size_t)maxwidth * sizeof(T), st, S, items,
                           n, bitems, z, x, part, wb);
    else
        hipLaunchKernelGGL((k_bwd_diag<T, 16>), dim3(grid8(n)), dim3(1024), (size_t)maxwidth * sizeof(T), st, S, items,
                           n, bitems, z, x, part, wb);
}


#define INST(T)                                                                                                   \
    template void launch_fwd_diag<T>(const DevSymbol &, const DiagItem *, int, const YSlices &, const T *,       \
                                     int64_t, T *, int64_t, T *, int64_t, int, const T *, const T *, int,        \
                                     hipStream_t);                                                               \
    template void launch_fwd_prod<T>(const DevSymbol &, const FwdItem *, int, const T *, const T *, int64_t, int, \
                                     const int32_t *, T *, int64_t, int, hipStream_t);                           \
    template void launch_bwd_prod<T>(const DevSymbol &, const BwdItem *, int, const T *, const T *, int64_t, int, \
                                     T *, int, hipStream_t);                                                     \
    template void launch_bwd_diag<T>(const DevSymbol &, const DiagItem *, int, const BwdItem *, T *, int64_t,     \
                                     T *, int64_t, int, const T *, const T *, int, hipStream_t);
INST(double)
INST(float)


}  // namespace pxa
