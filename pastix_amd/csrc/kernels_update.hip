// Schur-complement update for CDNA4 (gfx950)
// (reference kernels/core_zgemmsp.c:396-465 and cpucblk_zgemmsp :1337-1409).
//
// One workgroup owns each 64x64 tile of a target cblk's panel and applies, in
// source order, every contribution of the level's sources that lands in it:
// C[f] -= A[s](p rows) * B[s](q rows)^T scattered through the row/column maps
// (no atomics, bitwise-reproducible).
//   k_update_direct : tiles fed by a single source: the product is kept in
//                     registers (computed transposed so that stores walk down
//                     target columns) and subtracted straight into C;
//   k_update_seq    : tiles fed by several sources: each entry's product as
//                     in k_update_direct, subtracted into C in entry order
//                     (FP64) or summed in LDS and subtracted once (FP32);
//   k_update_narrow : the same on levels of narrow sources, a wave per entry;
//   k_update_wgemm, k_update_gather : the products of a level's sources into a
//                     workspace, then summed up tile by tile.
// MODE 0 (LL^t and the L side of LU) keeps pairs with block(p) >= block(q),
// MODE 1 (U side of LU) keeps block(p) > block(q), as the reference's
// iterblok >= blok / iterblok > blok loops.
#include <type_traits>

#include "dev_common.h"
#include "dev_types.h"
#include "dev_update.h"
#include "kernels.h"

namespace pxa {

// The one-pass kernels' entries from the plan's, once per engine: sixteen
// lanes to an item.
__global__ __launch_bounds__(256) void k_update_entries(DevSymbol S, const UpdItem *__restrict__ items, int n,
                                                        const int32_t *__restrict__ from,
                                                        const UpdEntry *__restrict__ ents, UpdX *__restrict__ xs) {
    const int id = blockIdx.x * 16 + (threadIdx.x >> 4);
    if (id >= n || from[id] < 0) return;
    const UpdItem it = items[id];
    const UpdEntry *src = ents + from[id];
    const int64_t c = S.cblk_coef[it.f];
    const int stf = S.cblk_stride[it.f], fcol = S.cblk_fcol[it.f];
    for (int e = threadIdx.x & 15; e < it.e1 - it.e0; e += 16) {
        const UpdEntry en = src[e];
        UpdX x{};
        x.a = S.cblk_coef[en.s] + en.p0;
        x.c = c;
        x.rb = S.cblk_rowbase[en.s] + en.p0;
        x.K = S.cblk_fcol[en.s + 1] - S.cblk_fcol[en.s];
        x.ld = S.cblk_stride[en.s];
        x.stf = stf;
        x.np = en.p1 - en.p0;
        x.nq = en.q1 - en.q0;
        x.dq = en.q0 - en.p0;
        x.sbi = en.sb - en.ib0;
        x.fcol = fcol;
        xs[it.e0 + e] = x;
    }
}
void launch_update_entries(const DevSymbol &S, const UpdItem *items, int n, const int32_t *from, const UpdEntry *ents,
                           UpdX *xs, hipStream_t st) {
    if (n > 0)
        hipLaunchKernelGGL(k_update_entries, dim3((n + 15) / 16), dim3(256), 0, st, S, items, n, from, ents, xs);
}

// K columns staged per LDS chunk in the single-tile GEMMs (16 measured
// faster than 32 on gfx950: the smaller LDS footprint keeps 6 workgroups per
// CU resident; two buffers of 8 columns with one barrier each were no faster,
// two of 16 slower, 24.0 against 21.9 ms).
constexpr int UPD_CH = 16;

// One entry's product minus from the target: up to 64 source rows p x 64
// source columns q, computed transposed, D(j, i) = B(q_j) . A(p_i), so that
// stores walk down target columns.  The row and column maps are fetched
// before the product and published after it: their loads (two deep) run
// under the first chunks.  Bound by the matrix cores (65 to 80 % busy) with
// the rest in the tiles' first and last memory round trips: 80^3 Laplacian,
// FP64, one stream, k_update_direct 20.9 ms (47 TFLOP/s; 21.9 with the maps
// before the product and the descriptors behind three loads), k_update_seq
// 14.0 ms (47 TFLOP/s); FP32 on 61x57x66 2.8 and 1.9 ms (k_update_seq summing
// in LDS 2.1).  Fire-and-forget atomic subtraction instead of the load was
// slower.
template <typename T> struct UpdLds {
    StageBuf<T, UPD_CH> sb;
    int rmap[64], cmap[64], rblk[64], qblk[64];
};
template <typename T>
__device__ __forceinline__ void update_product(Quad<T> &q, const DevSymbol &S, const UpdX &x,
                                               const int32_t *__restrict__ shift, const T *__restrict__ Acoef,
                                               const T *__restrict__ Bcoef, UpdLds<T> &l, int tid) {
    const int lane = tid & 63;
    int mrow = 0, mblk = 0;
    if (tid < 128) {
        const int64_t r = x.rb + (tid < 64 ? min(lane, x.np - 1) : x.dq + min(lane, x.nq - 1));
        mblk = S.panel_blk[r];
        mrow = S.panel_grow[r];
    }
    GemmLds<T, UPD_CH> g;
    g.start(Bcoef + x.a + x.dq, x.nq, x.ld, Acoef + x.a, x.np, x.ld, x.K, tid);
    if (tid < 64) mrow += shift[x.sbi + mblk];
    else mrow -= x.fcol;
    q.zero();
    g.run(q, l.sb, tid);
    if (tid < 64) {
        l.rmap[lane] = mrow;
        l.rblk[lane] = mblk;
    } else if (tid < 128) {
        l.cmap[lane] = mrow;
        l.qblk[lane] = mblk;
    }
    __syncthreads();
}
template <typename T, int MODE>
__device__ __forceinline__ void update_entry(const DevSymbol &S, const UpdX &x, const int32_t *__restrict__ shift,
                                             const T *__restrict__ Acoef, const T *__restrict__ Bcoef,
                                             T *__restrict__ Ccoef, UpdLds<T> &l, int tid) {
    Quad<T> q;
    update_product(q, S, x, shift, Acoef, Bcoef, l, tid);
    const int lane = tid & 63, wave = tid >> 6;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    if (wr < x.nq && wc < x.np) {
        const int64_t stf = x.stf;
        T *C = Ccoef + x.c;
        quad_sub(q, lane, [&](int qrow, int qcol, bool &ok) -> T * {
            const int qj = wr + qrow, pi = wc + qcol;
            ok = qj < x.nq && pi < x.np && ((MODE == 0) ? (l.rblk[pi] >= l.qblk[qj]) : (l.rblk[pi] > l.qblk[qj]));
            return ok ? C + l.rmap[pi] + (int64_t)l.cmap[qj] * stf : C;
        });
    }
}

// register budget held to seven waves per SIMD (72 registers in FP64, no
// spills; the compiler's own choice, 80, allows six): 54.4 -> 53.9 ms FP64
// numfact on the 80^3 Laplacian
template <typename T, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7, 8))) void k_update_direct(
    DevSymbol S, const UpdX *__restrict__ xs, int nitems, const int32_t *__restrict__ shift,
    const T *__restrict__ Acoef, const T *__restrict__ Bcoef, T *__restrict__ Ccoef) {
    __shared__ UpdLds<T> lds;
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    update_entry<T, MODE>(S, xs[id], shift, Acoef, Bcoef, Ccoef, lds, threadIdx.x);
}

// Tiles fed by several sources.  FP64: the entries in order, each one's
// product computed in registers as in k_update_direct and subtracted straight
// into C (C -= p1, then C -= p2, ..., the reference's source order), with a
// barrier between entries so that the next entry's read-modify-write of an
// element another wave wrote sees it (an LDS tile's 52 KB would allow three
// waves per SIMD instead of five: 56.0 against 54.3 ms on the 80^3 Laplacian).
// FP32: the products are summed in an LDS tile that is subtracted at the end:
// one rounding at C's magnitude instead of one per entry (in turn, the FP32
// solution of the 80^3 Laplacian was off by 8.1e-7 instead of 6.1e-7).
template <typename T> struct UpdSum {
    // four groups of sixteen rows, columns four (FP32) or one (FP64) apart:
    // every bank once (twice)
    static constexpr int LD = sizeof(T) == 4 ? 68 : 72;
    T t[64 * LD];
    __device__ __forceinline__ void zero(int tid) {
        for (int k = tid; k < 64 * LD; k += 256) t[k] = (T)0;
    }
    // the entry's product at (row, column) of the panel, the tile's corner at (r0, c0)
    template <int MODE>
    __device__ __forceinline__ void add(const Quad<T> &q, const UpdX &x, int r0, int c0, const UpdLds<T> &l, int tid) {
        const int lane = tid & 63, wave = tid >> 6;
        const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
        if (wr >= x.nq || wc >= x.np) return;
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int n = 0; n < 2; n++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int qj = wr + m * 16 + Mfma<T>::drow(lane, r), pi = wc + n * 16 + (lane & 15);
                    if (qj < x.nq && pi < x.np && ((MODE == 0) ? (l.rblk[pi] >= l.qblk[qj]) : (l.rblk[pi] > l.qblk[qj])))
                        t[(l.cmap[qj] - c0) * LD + l.rmap[pi] - r0] += q.c[m][n][r];
                }
    }
    // the tile (at C, `rows` x `cols` of it in the panel) minus the sums
    __device__ __forceinline__ void apply(T *C, int64_t stf, int64_t rows, int cols, int tid) const {
        const int r = tid & 63, c0 = tid >> 6;
        T v[16];
#pragma unroll
        for (int u = 0; u < 16; u++)
            v[u] = C[min((int64_t)r, rows - 1) + min(c0 + 4 * u, cols - 1) * stf];
#pragma unroll
        for (int u = 0; u < 16; u++) {
            const T w = t[(c0 + 4 * u) * LD + r];
            if (r < rows && c0 + 4 * u < cols && w != (T)0) C[r + (c0 + 4 * u) * stf] = v[u] - w;
        }
    }
};
template <typename T, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5, 8))) void k_update_seq(
    DevSymbol S, const UpdItem *__restrict__ items, int nitems, const UpdX *__restrict__ xs,
    const int32_t *__restrict__ shift, const T *__restrict__ Acoef, const T *__restrict__ Bcoef,
    T *__restrict__ Ccoef) {
    __shared__ UpdLds<T> lds;
    __shared__ std::conditional_t<sizeof(T) == 4, UpdSum<T>, char> sum;
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const UpdItem it = items[id];
    const int tid = threadIdx.x;
    if constexpr (sizeof(T) == 4) sum.zero(tid);
    for (int e = it.e0; e < it.e1; e++) {
        // the previous entry's stores and map reads are done by every wave
        if (e > it.e0) __syncthreads();
        if constexpr (sizeof(T) == 4) {
            Quad<T> q;
            update_product(q, S, xs[e], shift, Acoef, Bcoef, lds, tid);
            sum.template add<MODE>(q, xs[e], it.r0, it.c0, lds, tid);
        } else {
            update_entry<T, MODE>(S, xs[e], shift, Acoef, Bcoef, Ccoef, lds, tid);
        }
    }
    if constexpr (sizeof(T) == 4) {
        __syncthreads();
        const int64_t stf = xs[it.e0].stf;
        sum.apply(Ccoef + xs[it.e0].c + it.r0 + it.c0 * stf, stf, stf - it.r0,
                  S.cblk_fcol[it.f + 1] - S.cblk_fcol[it.f] - it.c0, tid);
    }
}

// The same for levels whose sources have at most NARROW_UPD columns (the
// bottom of the tree), FP32 and FP64.  An entry there is 7 rows by 3 columns
// and 7 source columns (lowest level of a 2D Laplacian) or 13 x 8 and 8 (27
// points on 48^3): one or two 16x16 pieces, too little for a workgroup.  Every
// wave takes an entry, operands straight from memory, and when its turn comes
// adds the product to the tile's sums in LDS; they are subtracted once at the
// end.  Entry order and one subtraction, as with the product workspace
// (k_update_wgemm, k_update_gather), bit for bit.
//
// Bound by latency: descriptor, maps and operands are three loads deep.  So as
// many tiles as possible at a time: only the columns that receive something
// (cm0, cm1) have sums, and the tiles of at most NARROW_COLS of them, nearly
// all, go apart from the others with two waves each.  Lowest level of the
// 701x653 Laplacian, FP64 (35,210 tiles, 135,188 entries): 784 us through the
// workspace, 465 with 64 columns of sums and four waves for every tile, 181 so
// (16 columns 180, 32 columns 232); its five narrow levels 1578 -> 514 us,
// numfact 4.0 -> 3.1 ms.  Subtracting entry by entry without LDS took 485 us,
// but rounds every entry at the target's magnitude.  Source panels of at most
// NARROW_ROWS rows (32-bit lane offsets of up to three columns).
template <typename T, int MODE, int NW, int NC>
__global__ __launch_bounds__(64 * NW) void k_update_narrow(DevSymbol S, const UpdItem *__restrict__ items, int nitems,
                                                       const UpdX *__restrict__ xs, const int32_t *__restrict__ shift,
                                                       const T *__restrict__ Acoef, const T *__restrict__ Bcoef,
                                                       T *__restrict__ Ccoef) {
    // row r of the tile's s-th touched column at [s * LD + r]
    constexpr int LD = UpdSum<T>::LD;
    __shared__ T sum[NC * LD];
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const UpdItem it = items[id];
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr uint32_t SZ = sizeof(T);
    auto at = [](const T *base, uint32_t bytes) -> T {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + bytes);
    };
    typedef typename Mfma<T>::v4 v4;
    const uint64_t mask = ((uint64_t)it.cm1 << 32) | it.cm0;
    const int nc = __popcll(mask);
    for (int o = tid; o < nc * LD; o += 64 * NW) sum[o] = (T)0;
    for (int eb = it.e0; eb < it.e1; eb += NW) {
        const int e = eb + wave, ne = min(NW, it.e1 - eb);
        const UpdX x = xs[min(e, it.e1 - 1)];
        // row and column maps: lane l holds source row p0 + l, column q0 + l
        const int32_t *pblk = S.panel_blk + x.rb, *pgrow = S.panel_grow + x.rb;
        const int rp = min(lane, x.np - 1), rq = x.dq + min(lane, x.nq - 1);
        const int pb = pblk[rp], qb = pblk[rq];
        int pr = pgrow[rp] - it.r0;
        const int qc = __popcll(mask & (((uint64_t)1 << (pgrow[rq] - x.fcol - it.c0)) - 1)) * LD;
        const T *A = Acoef + x.a, *B = Bcoef + x.a + x.dq;
        // 16x16 pieces, columns q by rows p, p first; lane offsets of a
        // step's four source columns and of the last step's
        const int npt = (x.np + 15) >> 4, nt = e < it.e1 ? npt * ((x.nq + 15) >> 4) : 0;
        const int ns = (x.K + 3) >> 2, kl = x.K - 4 * (ns - 1);
        const uint32_t ldb = x.ld * SZ, kv = kq * ldb, kvl = min(kq, kl - 1) * ldb;
        auto product = [&](int q0, int p0) -> v4 {
            const uint32_t ao = min(p0 + i, x.np - 1) * SZ, bo = min(q0 + i, x.nq - 1) * SZ;
            v4 acc = {0, 0, 0, 0};
#pragma unroll 1
            for (int s = 0; s < ns; s += 2) {
                T a[2], b[2];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int su = min(s + u, ns - 1);
                    const uint32_t ko = su == ns - 1 ? kvl : kv;
                    const int64_t so = (int64_t)(4 * su) * x.ld;
                    a[u] = at(A + so, ao + ko);
                    b[u] = at(B + so, bo + ko);
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const bool in = 4 * (s + u) + kq < x.K;
                    acc = Mfma<T>::mma(in ? b[u] : (T)0, in ? a[u] : (T)0, acc);
                }
            }
            return acc;
        };
        auto add = [&](int q0, int p0, const v4 &acc) {
            const int row = __shfl(pr, p0 + i), bp = __shfl(pb, p0 + i);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int j = q0 + Mfma<T>::drow(lane, r);
                const int col = __shfl(qc, j), bq = __shfl(qb, j);
                if (p0 + i < x.np && j < x.nq && (MODE == 0 ? bp >= bq : bp > bq)) sum[col + row] += acc[r];
            }
        };
        constexpr int NT = 4;  // pieces kept in registers until the wave's turn
        v4 acc[NT];
        int q0 = 0, p0 = 0;
        auto next = [&] {
            p0 += 16;
            if (p0 >= x.np) {
                p0 = 0;
                q0 += 16;
            }
        };
#pragma unroll
        for (int t = 0; t < NT; t++)
            if (t < nt) {
                acc[t] = product(q0, p0);
                next();
            }
        pr += shift[x.sbi + pb];
        for (int w = 0; w < ne; w++) {
            __syncthreads();
            if (w != wave) continue;
            q0 = p0 = 0;
#pragma unroll
            for (int t = 0; t < NT; t++)
                if (t < nt) {
                    add(q0, p0, acc[t]);
                    next();
                }
            for (int t = NT; t < nt; t++) {
                add(q0, p0, product(q0, p0));
                next();
            }
        }
    }
    __syncthreads();
    const int64_t stf = xs[it.e0].stf;
    T *C = Ccoef + xs[it.e0].c + it.r0 + lane + it.c0 * stf;
    // the touched columns in turn, wave w every NW-th; zeros are not touched
    uint64_t left = mask;
    for (int w = 0; w < wave; w++) left &= left - 1;
    for (int s = wave; s < nc; s += 4 * NW) {
        T v[4], c[4];
        T *cp[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int su = s + u * NW;
            cp[u] = C + (left ? __builtin_ctzll(left) : 0) * stf;
#pragma unroll
            for (int w = 0; w < NW; w++) left &= left - 1;
            v[u] = su < nc ? sum[min(su, NC - 1) * LD + lane] : (T)0;
            c[u] = (T)0;
            if (v[u] != (T)0) c[u] = *cp[u];
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (v[u] != (T)0) *cp[u] = c[u] - v[u];
    }
}

// Phase 1 of the multi-source tiles: dense 128 (p) x 64 (q) tile of a
// product group in the source's own row space (register budget held to four
// waves per SIMD: one more than the compiler picks unbounded, no spills), P(p, q) = A(p, :) . B(q, :)^T, stored to the
// level workspace.  Computed transposed (quadrant rows index q) so that each
// lane's stores walk down a workspace column.
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_update_wgemm(DevSymbol S, const WTile *__restrict__ items, int nitems,
                                                      const T *__restrict__ Acoef, const T *__restrict__ Bcoef,
                                                      T *__restrict__ W) {
    __shared__ StageBuf2<T, UPD_CH> sb;
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 64;
    const WTile w = items[id];
    const int s = w.s;
    const int K = S.cblk_fcol[s + 1] - S.cblk_fcol[s];
    const int64_t ld = S.cblk_stride[s];
    Quad<T> q0, q1;
    q0.zero();
    q1.zero();
    // 64 q rows (B) x 128 p rows (A) of the group's product
    wg_gemm_lds_64x128<T, UPD_CH>(q0, q1, Bcoef + S.cblk_coef[s] + w.q0, w.mq, ld, Acoef + S.cblk_coef[s] + w.p0,
                                  w.mp, ld, K, sb, tid);
    T *Wt = W + w.wofs;
    if (wr < w.mq && wc < w.mp) {
        UQFOR({
            const int qj = wr + qrow, pi = wc + qcol;
            if (qj < w.mq && pi < w.mp) Wt[pi + (int64_t)qj * w.ldw] = q0.c[m_][n_][r_];
        })
    }
    if (wr < w.mq && wc + 32 < w.mp) {
        UQFOR({
            const int qj = wr + qrow, pi = wc + 32 + qcol;
            if (qj < w.mq && pi < w.mp) Wt[pi + (int64_t)qj * w.ldw] = q1.c[m_][n_][r_];
        })
    }
}

// Phase 2: every multi-source target tile sums, in entry order, the products
// of its entries read from the workspace and subtracts the sum once.
// Thread (r, ph) owns target row r and columns ph, ph+4, ..., ph+60 of the
// tile.  Entries are taken in batches of 8: first the source rows landing on
// each target row / column of every entry of the batch are published in LDS
// tables tagged with the entry index (64 threads per entry, independent
// loads for the whole batch), then the products are accumulated in entry
// order.
template <typename T, int MODE>
__global__ __launch_bounds__(256) void k_update_gather(DevSymbol S, const UpdItem *__restrict__ items, int nitems,
                                                       const UpdEntry *__restrict__ ents,
                                                       const int32_t *__restrict__ shift,
                                                       const WGroup *__restrict__ grp, const T *__restrict__ W,
                                                       T *__restrict__ Ccoef) {
    constexpr int NB = 8;
    __shared__ int rp[NB][64], rs[NB][64], rbk[NB][64];
    __shared__ int cq[NB][64], cs[NB][64], cbk[NB][64];
    __shared__ int64_t wb[NB];
    __shared__ int wl[NB];
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    const int tid = threadIdx.x, r = tid & 63, ph = tid >> 6;
    const UpdItem it = items[id];
    const int f = it.f, r0 = it.r0, c0 = it.c0;
    const int fcol = S.cblk_fcol[f];
    for (int e = tid; e < NB * 64; e += 256) {
        (&rs[0][0])[e] = -1;
        (&cs[0][0])[e] = -1;
    }
    // products: thread (g, cph) owns the E consecutive target rows E*g.. of
    // columns cph + CP*u; when the rows are one run of source rows of the
    // entry, a column's contribution is one 16-byte load
    constexpr int E = Vec<T>::E, RG = 64 / E, CP = 256 / RG, NC = 64 / CP;
    const int rr = E * (tid % RG), cph = tid / RG;
    T acc[NC][E];
#pragma unroll
    for (int u = 0; u < NC; u++)
#pragma unroll
        for (int i = 0; i < E; i++) acc[u][i] = (T)0;
    for (int eb = it.e0; eb < it.e1; eb += NB) {
        const int ne = min(NB, it.e1 - eb);
        __syncthreads();  // previous batch consumed (and the tables initialised)
#pragma unroll
        for (int pass = 0; pass < NB / 4; pass++) {
            const int slot = pass * 4 + ph;
            if (slot < ne) {
                const int e = eb + slot;
                const UpdEntry en = ents[e];
                const int64_t rb = S.cblk_rowbase[en.s];
                const int p = en.p0 + r;
                if (p < en.p1) {
                    const int bk = S.panel_blk[rb + p];
                    const int tr = S.panel_grow[rb + p] + shift[en.sb + bk - en.ib0] - r0;
                    rp[slot][tr] = p;
                    rbk[slot][tr] = bk;
                    rs[slot][tr] = e;
                }
                const int qq = en.q0 + r;
                if (qq < en.q1) {
                    const int tc = S.panel_grow[rb + qq] - fcol - c0;
                    cq[slot][tc] = qq;
                    cbk[slot][tc] = S.panel_blk[rb + qq];
                    cs[slot][tc] = e;
                }
                if (r == 0) {
                    const WGroup G = grp[en.grp];
                    const int base = S.blok_roff[en.ib0];
                    wb[slot] = G.wofs - base - (int64_t)base * G.ldw;
                    wl[slot] = G.ldw;
                }
            }
        }
        __syncthreads();
        for (int slot = 0; slot < ne; slot++) {
            const int e = eb + slot;
            bool cov[E], any = false, run = true;
            int pr[E], bkr[E];
            const int p0 = rp[slot][rr];
#pragma unroll
            for (int i = 0; i < E; i++) {
                cov[i] = rs[slot][rr + i] == e;
                pr[i] = rp[slot][rr + i];
                bkr[i] = rbk[slot][rr + i];
                any |= cov[i];
                run &= cov[i] && pr[i] == p0 + i;
            }
            if (!any) continue;
            const int64_t ldw = wl[slot];
            const T *Wb = W + wb[slot];
#pragma unroll
            for (int u = 0; u < NC; u++) {
                const int c = cph + CP * u;
                if (cs[slot][c] != e) continue;
                const T *Wc = Wb + (int64_t)cq[slot][c] * ldw;
                const int cb = cbk[slot][c];
                T v[E];
                if (run) {
                    const typename Vec<T>::u w = *reinterpret_cast<const typename Vec<T>::u *>(Wc + p0);
#pragma unroll
                    for (int i = 0; i < E; i++) v[i] = w[i];
                } else {
#pragma unroll
                    for (int i = 0; i < E; i++) v[i] = cov[i] ? Wc[pr[i]] : (T)0;
                }
#pragma unroll
                for (int i = 0; i < E; i++) {
                    const bool keep = cov[i] && ((MODE == 0) ? (bkr[i] >= cb) : (bkr[i] > cb));
                    if (keep) acc[u][i] += v[i];
                }
            }
        }
    }
    const int Kf = S.cblk_fcol[f + 1] - fcol;
    const int64_t stf = S.cblk_stride[f];
    T *C = Ccoef + S.cblk_coef[f];
#pragma unroll
    for (int u = 0; u < NC; u++) {
        const int cc = c0 + cph + CP * u;
        if (cc >= Kf) continue;
        bool nz = false;
#pragma unroll
        for (int i = 0; i < E; i++) nz |= acc[u][i] != (T)0;
        if (!nz) continue;
        T *Cp = C + r0 + rr + (int64_t)cc * stf;
        if (r0 + rr + E <= stf) {
            typename Vec<T>::u w = *reinterpret_cast<const typename Vec<T>::u *>(Cp);
#pragma unroll
            for (int i = 0; i < E; i++) w[i] -= acc[u][i];
            *reinterpret_cast<typename Vec<T>::u *>(Cp) = w;
        } else {
#pragma unroll
            for (int i = 0; i < E; i++)
                if (r0 + rr + i < stf && acc[u][i] != (T)0) Cp[i] -= acc[u][i];
        }
    }
}

static inline int grid8(int n) { return ((n + 7) / 8) * 8; }

// LDS of an update workgroup that runs beside the panel kernels (`beside`,
// the second stream): unused space rounds it up so that five of them fill a
// CU.  At the seven that the registers allow, a panel kernel of a few
// workgroups (a diagonal block takes 42 KB and a wave of 124 registers on
// every SIMD) waits for a CU to drain: k_potrf64 took 90-186 us beside the
// updates, 22 us alone, and the level's other panels wait for it.
// Factorisation of an 80^3 Laplacian with 7 / 6 / 5 / 3 workgroups per CU:
// 49.9 / 49.1 / 48.4 / 50.0 ms; in FP32 (61x57x66), with 8 / 6 / 5: 10.05 /
// 9.88 / 9.69 ms; LU of 48^3 13.7 ms with either.
constexpr size_t BESIDE_LDS = 32768;

template <typename T>
void launch_update_direct(const DevSymbol &S, int mode, const UpdX *xs, int n, const int32_t *shift, const T *A,
                          const T *B, T *C, bool beside, hipStream_t st) {
    if (n <= 0) return;
    const dim3 g(grid8(n)), b(256);
    const size_t lds = beside ? BESIDE_LDS - sizeof(UpdLds<T>) : 0;
    if (mode == 0) hipLaunchKernelGGL((k_update_direct<T, 0>), g, b, lds, st, S, xs, n, shift, A, B, C);
    else hipLaunchKernelGGL((k_update_direct<T, 1>), g, b, lds, st, S, xs, n, shift, A, B, C);
}

template <typename T>
void launch_update_seq(const DevSymbol &S, int mode, const UpdItem *items, int n, const UpdX *xs,
                       const int32_t *shift, const T *A, const T *B, T *C, bool beside, hipStream_t st) {
    if (n <= 0) return;
    const dim3 g(grid8(n)), b(256);
    const size_t own = sizeof(UpdLds<T>) + (sizeof(T) == 4 ? sizeof(UpdSum<T>) : 0);
    const size_t lds = beside ? BESIDE_LDS - own : 0;
    if (mode == 0) hipLaunchKernelGGL((k_update_seq<T, 0>), g, b, lds, st, S, items, n, xs, shift, A, B, C);
    else hipLaunchKernelGGL((k_update_seq<T, 1>), g, b, lds, st, S, items, n, xs, shift, A, B, C);
}

template <typename T>
void launch_update_narrow(const DevSymbol &S, int mode, const UpdItem *items, int n, bool few, const UpdX *xs,
                          const int32_t *shift, const T *A, const T *B, T *C, hipStream_t st) {
    if (n <= 0) return;
    auto run = [&](auto kernel, int waves) {
        hipLaunchKernelGGL(kernel, dim3(grid8(n)), dim3(64 * waves), 0, st, S, items, n, xs, shift, A, B, C);
    };
    constexpr int W = NARROW_COLS;
    if (few) mode == 0 ? run(k_update_narrow<T, 0, 2, W>, 2) : run(k_update_narrow<T, 1, 2, W>, 2);
    else mode == 0 ? run(k_update_narrow<T, 0, 4, 64>, 4) : run(k_update_narrow<T, 1, 4, 64>, 4);
}

template <typename T>
void launch_update_wgemm(const DevSymbol &S, const WTile *items, int n, const T *A, const T *B, T *W, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL((k_update_wgemm<T>), dim3(grid8(n)), dim3(256), 0, st, S, items, n, A, B, W);
}

template <typename T>
void launch_update_gather(const DevSymbol &S, int mode, const UpdItem *items, int n, const UpdEntry *ents,
                          const int32_t *shift, const WGroup *grp, const T *W, T *C, hipStream_t st) {
    if (n <= 0) return;
    const dim3 g(grid8(n)), b(256);
    if (mode == 0) hipLaunchKernelGGL((k_update_gather<T, 0>), g, b, 0, st, S, items, n, ents, shift, grp, W, C);
    else hipLaunchKernelGGL((k_update_gather<T, 1>), g, b, 0, st, S, items, n, ents, shift, grp, W, C);
}

#define PXA_UPD_INST(T)                                                                                           \
    template void launch_update_direct<T>(const DevSymbol &, int, const UpdX *, int, const int32_t *, const T *,  \
                                          const T *, T *, bool, hipStream_t);                                     \
    template void launch_update_seq<T>(const DevSymbol &, int, const UpdItem *, int, const UpdX *,                \
                                       const int32_t *, const T *, const T *, T *, bool, hipStream_t);            \
    template void launch_update_narrow<T>(const DevSymbol &, int, const UpdItem *, int, bool, const UpdX *,       \
                                          const int32_t *, const T *, const T *, T *, hipStream_t);               \
    template void launch_update_wgemm<T>(const DevSymbol &, const WTile *, int, const T *, const T *, T *,        \
                                         hipStream_t);                                                            \
    template void launch_update_gather<T>(const DevSymbol &, int, const UpdItem *, int, const UpdEntry *,         \
                                          const int32_t *, const WGroup *, const T *, T *, hipStream_t);
PXA_UPD_INST(double)
PXA_UPD_INST(float)

}  // namespace pxa
