// Device helpers shared by the CDNA4 kernels: MFMA wrappers and the
// wave-level 32x32 tile product used by every GEMM-shaped kernel.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace pxa {

// v_mfma_{f64,f32}_16x16x4: A is 16x4, B is 4x16, D is 16x16.  Lane l holds
// A[l%16][l/16] and B[l/16][l%16] for both types; the accumulator layouts
// differ (measured on gfx950):
//   f32: D[4*(l/16) + r][l%16] in register r
//   f64: D[4*r + l/16][l%16]   in register r
template <typename T> struct Mfma;
template <> struct Mfma<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int drow(int lane, int r) { return 4 * r + (lane >> 4); }
};
template <> struct Mfma<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int drow(int lane, int r) { return 4 * (lane >> 4) + r; }
};

// 32x32 accumulator of one wave, as 2x2 MFMA blocks of 16x16.
template <typename T> struct Quad {
    typename Mfma<T>::v4 c[2][2];
    __device__ __forceinline__ void zero() {
        for (int m = 0; m < 2; m++)
            for (int n = 0; n < 2; n++)
                for (int r = 0; r < 4; r++) c[m][n][r] = (T)0;
    }
    // Element of block (m,n), register r, owned by `lane`:
    //   row = m*16 + Mfma<T>::drow(lane, r), col = n*16 + (lane&15)
};

// Operand staging moves 16 bytes per lane: E = 16 / sizeof(T) consecutive
// rows of one column (4 floats or 2 doubles).  Vec<T>::u has the alignment
// of one panel element (panels start and lead at any element), Vec<T>::a is
// fully aligned (LDS staging rows, whose pitch is a multiple of 16 bytes).
template <typename T> struct Vec;
template <> struct Vec<float> {
    static constexpr int E = 4;
    typedef float u __attribute__((ext_vector_type(4), aligned(4)));
    typedef float a __attribute__((ext_vector_type(4)));
};
template <> struct Vec<double> {
    static constexpr int E = 2;
    typedef double u __attribute__((ext_vector_type(2), aligned(8)));
    typedef double a __attribute__((ext_vector_type(2)));
};
// E rows [r, r+E) of column p (rows >= m read as zero) into o
template <typename T> __device__ __forceinline__ void ld_rows(const T *p, int r, int m, T *o) {
    constexpr int E = Vec<T>::E;
    if (r + E <= m) {
        const typename Vec<T>::u v = *reinterpret_cast<const typename Vec<T>::u *>(p);
#pragma unroll
        for (int e = 0; e < E; e++) o[e] = v[e];
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) o[e] = (r + e < m) ? p[e] : (T)0;
    }
}
// E consecutive elements at p, unconditionally
template <typename T> __device__ __forceinline__ void ld_vec(const T *p, T *o) {
    const typename Vec<T>::u v = *reinterpret_cast<const typename Vec<T>::u *>(p);
#pragma unroll
    for (int e = 0; e < Vec<T>::E; e++) o[e] = v[e];
}
template <typename T> __device__ __forceinline__ void st_rows(T *p, const T *o) {
    typename Vec<T>::a v;
#pragma unroll
    for (int e = 0; e < Vec<T>::E; e++) v[e] = o[e];
    *reinterpret_cast<typename Vec<T>::a *>(p) = v;
}

// Workgroup-level D(64x64) = X(64xK) * Y(64xK)^T with operands staged through
// LDS in chunks of CH columns (16 or 32): the 256 threads fetch each chunk
// once with coalesced column segments (rows contiguous in memory), the 4
// waves read their MFMA fragments from LDS.  Global loads of chunk c+1 are in
// flight while chunk c is multiplied, so a chunk's MFMA time (CH/4 * 4
// MFMAs per wave) is the latency the prefetch can hide.  X(r, k) =
// X[r + k*ldx].  Wave w owns the 32x32 quadrant (w>>1, w&1); output rows >=
// mx and columns >= my are not defined.  Must be called by all 256 threads
// (contains barriers).
//
// The loads carry no row masks: a row >= mx of X only reaches output rows >=
// mx, which nobody stores, so a lane past the last row reads row 0 again and
// the lane that straddles it up to E - 1 elements more (every device
// allocation ends in LOAD_PAD bytes of padding for the last column).  With
// masks the compiler waited for all outstanding loads before every partial
// one: up to four memory round trips per chunk on a tile with an odd row
// count.  Columns >= K must count as zero; the last chunk clears them on
// their way to LDS.  80^3 Laplacian, FP64, together with quad_sub below, one
// stream: k_update_direct 23.6 -> 21.9 ms, k_update_seq 17.8 -> 14.2 ms,
// panel steps 19.0 -> 16.2 ms.
template <typename T, int CH = 16> struct StageBuf {
    T xs[CH][68];
    T ys[CH][68];
};

// one chunk's MFMAs of a 32x32 quadrant, X fragments at xs[.][xr], Y at
// ys[.][yr]; left columns of the chunk (and later) exist.  A rolled loop:
// unrolled four times the direct update ran 21.7 instead of 20.9 ms,
// straight through 22.4.  Rows i and i + 16 to a lane, so that a lane group
// stores sixteen rows side by side; rows 2i and 2i + 1 would come in one LDS
// read but store every other row (21.4 ms).
template <typename T, int CH, int PX, int PY>
__device__ __forceinline__ void quad_chunk(Quad<T> &q, const T (*xs)[PX], const T (*ys)[PY], int xr, int yr, int left,
                                           int kq) {
    const int ns = (min(CH, left) + 3) / 4;
#pragma unroll 1
    for (int s = 0; s < ns; s++) {
        const int kr = 4 * s + kq;
        const T x0 = xs[kr][xr], x1 = xs[kr][xr + 16];
        const T y0 = ys[kr][yr], y1 = ys[kr][yr + 16];
        q.c[0][0] = Mfma<T>::mma(x0, y0, q.c[0][0]);
        q.c[0][1] = Mfma<T>::mma(x0, y1, q.c[0][1]);
        q.c[1][0] = Mfma<T>::mma(x1, y0, q.c[1][0]);
        q.c[1][1] = Mfma<T>::mma(x1, y1, q.c[1][1]);
    }
}

// One operand's chunk loads: R rows (64 or 128) of CH columns by the 256
// threads, 16 bytes per lane.  The column a wave's first lanes read is
// uniform, so the address is a scalar base plus a 32-bit lane offset of at
// most CPW - 1 columns and R rows.  It fits: a panel's rows are a clique of
// the factor, so its leading dimension squared is at most twice the stored
// entries.  No branches around the loads: with one for the last chunk the
// compiler waited between them.
template <typename T, int R, int CH> struct Stager {
    static constexpr int E = Vec<T>::E, LPC = R / E, CPW = 64 / LPC, NP = CH / (4 * CPW);
    static_assert(NP >= 1 && CH % (4 * CPW) == 0, "chunk of whole passes");
    const char *base;
    int64_t ldb;  // bytes from column to column
    unsigned row;
    int r, kl, kw;
    T g[NP][E];
    // rows [0, m) of P, column k at P + k*ld
    __device__ __forceinline__ void init(const T *P, int m, int64_t ld, int lane, int wave) {
        r = E * (lane % LPC);
        kl = lane / LPC;
        kw = CPW * wave;
        ldb = ld * (int64_t)sizeof(T);
        base = reinterpret_cast<const char *>(P);
        row = (unsigned)((r < m ? r : 0) * sizeof(T));
    }
    // columns [k0, k0 + CH); those at and after K read column K - 1 again
    __device__ __forceinline__ void load(int k0, int K) {
#pragma unroll
        for (int u = 0; u < NP; u++) {
            const int c = min(k0 + kw + 4 * CPW * u, K - 1);  // uniform
            const unsigned off = row + (unsigned)min(kl, K - 1 - c) * (unsigned)ldb;
            ld_vec(reinterpret_cast<const T *>(base + (int64_t)c * ldb + off), g[u]);
        }
    }
    // into s, columns at and after K as zeros
    template <int P> __device__ __forceinline__ void store(T (*s)[P], int k0, int K) {
        if (k0 + CH > K) {  // uniform
#pragma unroll
            for (int u = 0; u < NP; u++)
#pragma unroll
                for (int e = 0; e < E; e++)
                    if (k0 + kw + 4 * CPW * u + kl >= K) g[u][e] = (T)0;
        }
#pragma unroll
        for (int u = 0; u < NP; u++) st_rows(&s[kw + 4 * CPW * u + kl][r], g[u]);
    }
};

template <typename T, int CH> struct GemmLds {
    Stager<T, 64, CH> gx, gy;
    int mx, my, K;
    // the first chunk's loads go out
    __device__ __forceinline__ void start(const T *X, int mx_, int64_t ldx, const T *Y, int my_, int64_t ldy, int K_,
                                          int tid) {
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        mx = mx_;
        my = my_;
        K = K_;
        gx.init(X, mx, ldx, lane, wave);
        gy.init(Y, my, ldy, lane, wave);
        gx.load(0, K);
        gy.load(0, K);
    }
    __device__ __forceinline__ void run(Quad<T> &q, StageBuf<T, CH> &sb, int tid) {
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
        const int i = lane & 15, kq = lane >> 4;
        const bool active = (wr < mx) && (wc < my);
        gx.store(sb.xs, 0, K);
        gy.store(sb.ys, 0, K);
        __syncthreads();
        for (int k0 = 0; k0 < K; k0 += CH) {
            const bool more = k0 + CH < K;
            if (more) {
                gx.load(k0 + CH, K);
                gy.load(k0 + CH, K);
            }
            if (active) quad_chunk<T, CH>(q, sb.xs, sb.ys, wr + i, wc + i, K - k0, kq);
            __syncthreads();
            if (more) {
                gx.store(sb.xs, k0 + CH, K);
                gy.store(sb.ys, k0 + CH, K);
            }
            __syncthreads();
        }
    }
};

template <typename T, int CH>
__device__ __forceinline__ void wg_gemm_lds(Quad<T> &q, const T *X, int mx, int64_t ldx, const T *Y, int my,
                                            int64_t ldy, int K, StageBuf<T, CH> &sb, int tid) {
    GemmLds<T, CH> g;
    g.start(X, mx, ldx, Y, my, ldy, K, tid);
    g.run(q, sb, tid);
}

// The same product for a 64 x 128 tile: q0, q1 += X[0:64, 0:K] * Y[0:128,
// 0:K]^T, wave w owning X rows (w>>1)*32 + [0, 32) against Y rows (w&1)*64 +
// [0, 32) (q0) and [32, 64) (q1).  Each staged X fragment feeds twice as
// many MFMAs as in the 64 x 64 form.  Must be called by all 256 threads.
template <typename T, int CH = 16> struct StageBuf2 {
    T xs[CH][68];
    T ys[CH][132];
};

template <typename T, int CH>
__device__ __forceinline__ void wg_gemm_lds_64x128(Quad<T> &q0, Quad<T> &q1, const T *X, int mx, int64_t ldx,
                                                   const T *Y, int my, int64_t ldy, int K, StageBuf2<T, CH> &sb,
                                                   int tid) {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 64;
    const int i = lane & 15, kq = lane >> 4;
    Stager<T, 64, CH> gx;
    Stager<T, 128, CH> gy;
    gx.init(X, mx, ldx, lane, wave);
    gy.init(Y, my, ldy, lane, wave);
    const bool act0 = (wr < mx) && (wc < my), act1 = act0 && (wc + 32 < my);
    gx.load(0, K);
    gy.load(0, K);
    gx.store(sb.xs, 0, K);
    gy.store(sb.ys, 0, K);
    __syncthreads();
    for (int k0 = 0; k0 < K; k0 += CH) {
        const bool more = k0 + CH < K;
        if (more) {
            gx.load(k0 + CH, K);
            gy.load(k0 + CH, K);
        }
        if (act0) {
#pragma unroll
            for (int s = 0; s < CH / 4; s++) {
                if (k0 + 4 * s < K) {
                    const T x[2] = {sb.xs[4 * s + kq][wr + i], sb.xs[4 * s + kq][wr + 16 + i]};
                    const T y[2] = {sb.ys[4 * s + kq][wc + i], sb.ys[4 * s + kq][wc + 16 + i]};
                    q0.c[0][0] = Mfma<T>::mma(x[0], y[0], q0.c[0][0]);
                    q0.c[0][1] = Mfma<T>::mma(x[0], y[1], q0.c[0][1]);
                    q0.c[1][0] = Mfma<T>::mma(x[1], y[0], q0.c[1][0]);
                    q0.c[1][1] = Mfma<T>::mma(x[1], y[1], q0.c[1][1]);
                    if (act1) {
                        const T z[2] = {sb.ys[4 * s + kq][wc + 32 + i], sb.ys[4 * s + kq][wc + 48 + i]};
                        q1.c[0][0] = Mfma<T>::mma(x[0], z[0], q1.c[0][0]);
                        q1.c[0][1] = Mfma<T>::mma(x[0], z[1], q1.c[0][1]);
                        q1.c[1][0] = Mfma<T>::mma(x[1], z[0], q1.c[1][0]);
                        q1.c[1][1] = Mfma<T>::mma(x[1], z[1], q1.c[1][1]);
                    }
                }
            }
        }
        __syncthreads();
        if (more) {
            gx.store(sb.xs, k0 + CH, K);
            gy.store(sb.ys, k0 + CH, K);
        }
        __syncthreads();
    }
}

// The quadrant subtracted from memory: at(row, col, ok) gives the address of
// element (row, col) of the quadrant and whether it exists (the address must
// be readable either way).  Eight elements' loads go out together: written as
// C -= q one element at a time, every load waited for the store before it
// (they may alias), sixteen memory round trips in a row per tile.
template <typename T, class At> __device__ __forceinline__ void quad_sub(const Quad<T> &q, int lane, At at) {
#pragma unroll
    for (int m = 0; m < 2; m++) {
        T *p[2][4], v[2][4];
        bool ok[2][4];
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                p[n][r] = at(m * 16 + Mfma<T>::drow(lane, r), n * 16 + (lane & 15), ok[n][r]);
                v[n][r] = *p[n][r];
            }
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (ok[n][r]) *p[n][r] = v[n][r] - q.c[m][n][r];
    }
}

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous range of work items so neighbouring items share its L2.  The grid
// size must be a multiple of 8 (the map is then a bijection of [0, grid));
// callers drop ids beyond their item count.
__device__ __forceinline__ int xcd_remap(int bid, int grid) {
    int per = grid >> 3;
    return (bid & 7) * per + (bid >> 3);
}

}  // namespace pxa
