// Blocked right-looking panel factorisation for CDNA4 (gfx950).
//
// A cblk's panel (stride x K, column-major) is factored by 64-column steps,
// each step being three launches over all cblks of the level:
//   k_potrf64   : Cholesky of the 64x64 diagonal sub-block with static
//                 pivoting (reference kernels/core_zpotrfsp.c:66-108), the
//                 block in registers, plus its inverse;
//   k_panel_trsm: every panel row below the sub-block times inv(L_kk)^T
//                 (core_zpotrfsp.c:166-176 and core_ztrsmsp.c:147-181);
//   k_panel_upd : the in-cblk products (core_zpotrfsp.c:178-185 applied
//                 column block by column block): before the step, of the
//                 blocks before it into the step's block (left-looking), or,
//                 on levels with few rows, after the step, of the step's block
//                 into every later block (right-looking).
// k_winv_merge completes the inverses of the solve nodes' diagonal blocks
// once the panels are factored.  Inverses are stored twice: W (lower,
// column-major) for the forward sweep and WT = W^T for the backward sweep.
#include <algorithm>
#include <type_traits>

#include "dev_common.h"
#include "dev_types.h"
#include "dev_update.h"
#include "kernels.h"

namespace pxa {

#define QFOR(...)                                                        \
    for (int m_ = 0; m_ < 2; m_++)                                       \
        for (int n_ = 0; n_ < 2; n_++)                                   \
            for (int r_ = 0; r_ < 4; r_++) {                             \
                const int qrow = m_ * 16 + Mfma<T>::drow(lane, r_);       \
                const int qcol = n_ * 16 + (lane & 15);                   \
                __VA_ARGS__                                              \
            }

template <typename T> __device__ __forceinline__ T pabs(T v) { return v < (T)0 ? -v : v; }

// Square root and its reciprocal of a positive pivot, and reciprocals, from
// the hardware estimates refined until about one ulp: for the FP64 inverse
// square root one third-order step, y <- y + y e (1/2 + 3/8 e) with
// e = 1 - d y^2, which triples the correct bits of the estimate; Newton steps
// y <- y + y(1/2 - d y^2/2) and y <- y + y(1 - d y), each doubling them,
// elsewhere.  Fewer dependent instructions than the correctly rounded sqrt
// and division on the diagonal block's critical path.
__device__ __forceinline__ void sqrt_rsqrt(double d, double &L, double &r) {
    double y = __builtin_amdgcn_rsq(d);
    const double e = __builtin_fma(-(d * y), y, 1.0);
    y = __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
    r = y;
    L = d * y;
}
__device__ __forceinline__ void sqrt_rsqrt(float d, float &L, float &r) {
    float y = __builtin_amdgcn_rsqf(d);
    const float h = 0.5f * d * y;
    y = __builtin_fmaf(y, __builtin_fmaf(-h, y, 0.5f), y);
    r = y;
    L = d * y;
}
__device__ __forceinline__ double recip(double d) {
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
    return __builtin_fma(y, __builtin_fma(-d, y, 1.0), y);
}
__device__ __forceinline__ float recip(float d) {
    const float y = __builtin_amdgcn_rcpf(d);
    return __builtin_fmaf(y, __builtin_fmaf(-d, y, 1.0f), y);
}

__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmax_(double a, double b) { return __builtin_fmax(a, b); }
__device__ __forceinline__ float fmax_(float a, float b) { return __builtin_fmaxf(a, b); }

// Static pivoting of one Cholesky pivot (reference
// kernels/core_zpotrfsp.c:78-81: |d| < crit is replaced by crit, a negative
// pivot is an error): max(|d|, crit), one instruction on the dependency
// chain; the counts are kept off the chain.  Identity padding columns (pivot
// exactly 1) pass through too: they stay decoupled from the real columns, and
// the caller removes them from the count when crit > 1.
template <typename T> __device__ __forceinline__ T piv_max(T d, T crit, int &npiv, int &neg) {
    npiv += (pabs(d) < crit) ? 1 : 0;
    neg |= (d < (T)0 && d <= -crit) ? 1 : 0;
    return fmax_(pabs(d), crit);
}

// Value of v in lane `lane` (wave-uniform) of the calling wave.
__device__ __forceinline__ double rlane(double v, int lane) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ float rlane(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// One joining level of the recursive-doubling inverse below, on the vector
// units: for every pair of inverted diagonal blocks of size B (X11 at
// [base, base+B), X22 at [base+B, base+2B)), X21 = -X22 (M21 X11).
template <typename T, int B> __device__ __forceinline__ void inv_join_valu(T (*Xs)[65], T *Ts, int tid) {
    constexpr int NO = 32 * B;  // outputs of the level: 64/(2B) pairs of B x B
    const int o = tid;
    const int p = o / (B * B), rem = o % (B * B), r = rem / B, cc = rem % B, base = 2 * B * p;
    if (o < NO) {
        T s = (T)0;
#pragma unroll
        for (int m = 0; m < B; m++) s = fma_(Xs[base + B + r][base + m], Xs[base + m][base + cc], s);
        Ts[o] = s;
    }
    __syncthreads();
    if (o < NO) {
        T s = (T)0;
#pragma unroll
        for (int m = 0; m < B; m++) s = fma_(Xs[base + B + r][base + B + m], Ts[p * B * B + m * B + cc], s);
        Xs[base + B + r][base + cc] = -s;
    }
    __syncthreads();
}

// The same on the matrix cores for B = 16, 32: one 16x16 tile per wave.
template <typename T, int B> __device__ __forceinline__ void inv_join_mfma(T (*Xs)[65], T *Ts, int lane, int w) {
    constexpr int TPP = (B / 16) * (B / 16), NT = (64 / (2 * B)) * TPP;
    const int i = lane & 15, kq = lane >> 4;
    const int p = w / TPP, ti = (w % TPP) / (B / 16), tj = w % (B / 16), base = 2 * B * p;
    if (w < NT) {
        typename Mfma<T>::v4 acc = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < B / 4; s++) {
            const int k = 4 * s + kq;
            acc = Mfma<T>::mma(Xs[base + B + ti * 16 + i][base + k], Xs[base + k][base + tj * 16 + i], acc);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) Ts[p * B * B + (ti * 16 + Mfma<T>::drow(lane, r)) * B + tj * 16 + i] = acc[r];
    }
    __syncthreads();
    if (w < NT) {
        typename Mfma<T>::v4 acc = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < B / 4; s++) {
            const int k = 4 * s + kq;
            acc = Mfma<T>::mma(Xs[base + B + ti * 16 + i][base + B + k], Ts[p * B * B + k * B + tj * 16 + i], acc);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) Xs[base + B + ti * 16 + Mfma<T>::drow(lane, r)][base + tj * 16 + i] = -acc[r];
    }
    __syncthreads();
}

// X = inv(M) in place for the lower-triangular 64x64 M held in Xs, zeros
// above the diagonal (1/M(r, r) = dinv[r]), by recursive doubling: the
// sixteen 4x4 diagonal blocks are inverted directly, then pairs of inverted
// blocks of size 4, 8, 16 and 32 are joined
// (inv([M11 0; M21 M22]) = [X11 0; -X22 M21 X11 X22]): 4 levels of small
// products instead of a 64-step substitution.  Every join overwrites the
// block M21 it has consumed, and only M21 blocks are read from M after the
// 4x4 blocks.  Ts (1024 entries) is scratch.  Only X[0:nb, 0:nb] is complete:
// levels that would join blocks of the identity padding only are skipped.
// All 256 threads (nb uniform), barriers inside; Xs and dinv must be visible
// to all threads on entry.
template <typename T>
__device__ __forceinline__ void lower_inverse(T (*Xs)[65], T *Ts, const T *dinv, int nb, int tid, int w) {
    if (tid < 64) {
        // one wave; the block's strict lower entries are read before any write
        const int b0 = 4 * (tid >> 2), cc = tid & 3;
        auto M = [&](int r, int k) -> T { return Xs[b0 + r][b0 + k]; };
        const T m10 = M(1, 0), m20 = M(2, 0), m21 = M(2, 1), m30 = M(3, 0), m31 = M(3, 1), m32 = M(3, 2);
        const T d0 = dinv[b0], d1 = dinv[b0 + 1], d2 = dinv[b0 + 2], d3 = dinv[b0 + 3];
        const T x0 = (cc == 0) ? d0 : (T)0;
        const T x1 = (cc > 1) ? (T)0 : (cc == 1) ? d1 : -(m10 * x0) * d1;
        const T x2 = (cc > 2) ? (T)0 : (cc == 2) ? d2 : -fma_(m21, x1, m20 * x0) * d2;
        const T x3 = (cc == 3) ? d3 : -fma_(m32, x2, fma_(m31, x1, m30 * x0)) * d3;
        Xs[b0][b0 + cc] = x0;
        Xs[b0 + 1][b0 + cc] = x1;
        Xs[b0 + 2][b0 + cc] = x2;
        Xs[b0 + 3][b0 + cc] = x3;
    }
    __syncthreads();
    // a level whose joined blocks start at or beyond nb only builds padding
    if (nb > 4) inv_join_valu<T, 4>(Xs, Ts, tid);
    if (nb > 8) inv_join_valu<T, 8>(Xs, Ts, tid);
    if (nb > 16) inv_join_mfma<T, 16>(Xs, Ts, tid & 63, w);
    if (nb > 32) inv_join_mfma<T, 32>(Xs, Ts, tid & 63, w);
}

// Cholesky and inverse of one 64-column diagonal sub-block.
//
// Thread (i, w) = (tid % 64, tid / 64) keeps the entries (i, j), j = w mod 4,
// of row i in registers.  Columns are taken 4 at a time with one barrier per
// block: the block's 4 columns are published through LDS (two buffers by
// parity), every thread factors the 4x4 diagonal block, replacing pivots
// below the threshold (reference kernels/core_zpotrfsp.c:78-81), and forms
// its row's 4 multipliers.  The multipliers of the rows a wave's columns
// belong to are held by lanes of the same wave (every wave forms all rows'
// multipliers), so the rank-4 update reads them across lanes (readlane)
// rather than through LDS.  Only the next block's columns are updated before
// they are published; the update of the columns after them is deferred into
// the next block, where it overlaps that block's 4x4 dependency chain.  Rows
// beyond the block width are padded with the identity, which the updates
// leave untouched.
//
// The inverse X = inv(L) comes from lower_inverse (recursive doubling, in
// place of L in LDS).  W receives X (lower, column-major, ld = K) and WT its
// transpose, both with explicit zeros in the other triangle of the sub-block.
// LDS of one diagonal-block factorisation: the published columns (then the
// inverse's scratch), the factor and the pivots' reciprocals.
template <typename T> struct PotrfLds {
    T fac[1024];
    T Ls[64][65];
    T dinv[64];
};

template <typename T>
__device__ __forceinline__ void potrf64_block(const DevSymbol &S, const int c, int kb, T *__restrict__ coef,
                                              T *__restrict__ winv, T *__restrict__ winvt, double thr, int *stat,
                                              PotrfLds<T> &lds) {
    T *fac = lds.fac;
    T(*colb)[4][64] = reinterpret_cast<T(*)[4][64]>(fac);  // [parity][w][row]
    T(*Ls)[65] = lds.Ls;
    T *dinv = lds.dinv;
    T *Ts = fac;  // inverse scratch once the factor is done
    const int tid = threadIdx.x, i = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = S.cblk_fcol[c + 1] - S.cblk_fcol[c];
    const int k0 = kb * 64;
    const int nb = min(64, K - k0);
    const int64_t ld = S.cblk_stride[c];
    T *P = coef + S.cblk_coef[c] + k0 + (int64_t)k0 * ld;
    T a[16];
#pragma unroll
    for (int jj = 0; jj < 16; jj++) {
        const int j = 4 * jj + w;
        T v = (i == j) ? (T)1 : (T)0;
        if (i < nb && j < nb && j <= i) v = P[i + (int64_t)j * ld];
        a[jj] = v;
    }
    const T crit = (T)thr;
    int npiv = 0, neg = 0;
    T pl0 = 0, pl1 = 0, pl2 = 0, pl3 = 0;  // this row's multipliers of the last block (0 above it)
    colb[0][w][i] = a[0];
#pragma unroll
    for (int b4 = 0; b4 < 16; b4++) {
        const int k = 4 * b4;
        if (k >= nb) break;  // uniform: the padding needs no elimination
        __syncthreads();
        // the row index as an opaque value: keeps the compiler from hoisting
        // the 16 blocks' row masks out of the loop (they would hold registers
        // for the whole factorisation)
        int ii = i;
        asm volatile("" : "+v"(ii));
        T(*cb)[64] = colb[b4 & 1];
        const T c00 = cb[0][k], c10 = cb[0][k + 1], c20 = cb[0][k + 2], c30 = cb[0][k + 3];
        const T c11 = cb[1][k + 1], c21 = cb[1][k + 2], c31 = cb[1][k + 3];
        const T c22 = cb[2][k + 2], c32 = cb[2][k + 3], c33 = cb[3][k + 3];
        const T r0 = cb[0][ii], r1 = cb[1][ii], r2 = cb[2][ii], r3 = cb[3][ii];
        // deferred rank-4 update by the previous block of the columns after this block's
        if (b4 >= 1) {
#pragma unroll
            for (int jj = b4 + 1; jj < 16; jj++) {
                const int lj = 4 * jj + w;
                a[jj] = fma_(-pl3, rlane(pl3, lj), fma_(-pl2, rlane(pl2, lj),
                        fma_(-pl1, rlane(pl1, lj), fma_(-pl0, rlane(pl0, lj), a[jj]))));
            }
        }
        // 4x4 Cholesky of the diagonal block (same in every thread)
        T L00, i00, L11, i11, L22, i22, L33, i33;
        sqrt_rsqrt(piv_max(c00, crit, npiv, neg), L00, i00);
        const T L10 = c10 * i00, L20 = c20 * i00, L30 = c30 * i00;
        sqrt_rsqrt(piv_max(fma_(-L10, L10, c11), crit, npiv, neg), L11, i11);
        const T L21 = fma_(-L20, L10, c21) * i11, L31 = fma_(-L30, L10, c31) * i11;
        sqrt_rsqrt(piv_max(fma_(-L21, L21, fma_(-L20, L20, c22)), crit, npiv, neg), L22, i22);
        const T L32 = fma_(-L31, L21, fma_(-L30, L20, c32)) * i22;
        sqrt_rsqrt(piv_max(fma_(-L32, L32, fma_(-L31, L31, fma_(-L30, L30, c33))), crit, npiv, neg), L33, i33);
        // take the counts now: left to the end, they would keep every pivot in registers
        asm volatile("" : "+v"(npiv), "+v"(neg));
        // multipliers of row i (rows of the block take the block's L)
        const T m0 = r0 * i00;
        const T m1 = (r1 - m0 * L10) * i11;
        const T m2 = (r2 - m0 * L20 - m1 * L21) * i22;
        const T m3 = (r3 - m0 * L30 - m1 * L31 - m2 * L32) * i33;
        const int t = ii - k;
        const bool below = t > 3;
        const T l0 = below ? m0 : (t == 0) ? L00 : (t == 1) ? L10 : (t == 2) ? L20 : L30;
        const T l1 = below ? m1 : (t == 1) ? L11 : (t == 2) ? L21 : L31;
        const T l2 = below ? m2 : (t == 2) ? L22 : L32;
        const T l3 = below ? m3 : L33;
        const T lw = (w == 0) ? l0 : (w == 1) ? l1 : (w == 2) ? l2 : l3;
        if (t >= w) a[b4] = lw;
        pl0 = below ? l0 : (T)0;
        pl1 = below ? l1 : (T)0;
        pl2 = below ? l2 : (T)0;
        pl3 = below ? l3 : (T)0;
        if (b4 < 15) {
            const int jn = b4 + 1, lj = 4 * jn + w;
            a[jn] = fma_(-pl3, rlane(pl3, lj), fma_(-pl2, rlane(pl2, lj),
                    fma_(-pl1, rlane(pl1, lj), fma_(-pl0, rlane(pl0, lj), a[jn]))));
            colb[jn & 1][w][ii] = a[jn];
        }
    }
#pragma unroll
    for (int jj = 0; jj < 16; jj++) {
        const int j = 4 * jj + w;
        Ls[i][j] = (j <= i) ? a[jj] : (T)0;
        if (i < nb && j < nb && j <= i) P[i + (int64_t)j * ld] = a[jj];
    }
    if (crit > (T)1) npiv -= ((nb + 3) & ~3) - nb;  // the identity padding's pivots
    if (tid == 0) {
        if (npiv) atomicAdd(&stat[0], npiv);
        if (neg) atomicOr(&stat[1], 1);
    }
    __syncthreads();
    if (tid < 64) dinv[tid] = recip(Ls[tid][tid]);
    __syncthreads();
    lower_inverse<T>(Ls, Ts, dinv, nb, tid, w);
    T *W = winv + S.cblk_winv[c] + k0 + (int64_t)k0 * K;
    T *WT = winvt + S.cblk_winv[c] + k0 + (int64_t)k0 * K;
    for (int e = tid; e < 64 * 64; e += 256) {
        const int lo = e & 63, hi = e >> 6;
        if (lo < nb && hi < nb) {
            W[lo + (int64_t)hi * K] = Ls[lo][hi];
            WT[lo + (int64_t)hi * K] = Ls[hi][lo];
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_potrf64(DevSymbol S, const int32_t *__restrict__ cblks, int kb,
                                                 T *__restrict__ coef, T *__restrict__ winv, T *__restrict__ winvt,
                                                 double thr, int *stat) {
    __builtin_amdgcn_s_setprio(3);  // panel steps lead the critical path
    __shared__ PotrfLds<T> lds;
    potrf64_block<T>(S, cblks[blockIdx.x], kb, coef, winv, winvt, thr, stat, lds);
}

// Narrow supernodes.  k_potrf64 gives each one a 256-thread workgroup and 42 KB
// of LDS whatever its width: a leaf level of thousands of supernodes of 4 to
// 10 columns was three workgroups to a compute unit, each padding to 64 rows
// (701x653 grid, FP64: 16,384 of at most 5 columns 523 us; 80^3: 21,293 of at
// most 8).  Below, a row is a lane with its columns in registers, the pivot
// column crosses lanes without LDS, and nothing waits on a barrier.  The
// elimination is k_potrf64's, operation for operation; the inverse comes from
// forward substitution, lane c solving for column c.

// f(integral_constant<int, I>) for I = B .. E - 1
template <int B, int E, class F> __device__ __forceinline__ void static_for(F f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// v of lane N of the calling lane's row of sixteen
template <int N> __device__ __forceinline__ int row16(int v) {
    return __builtin_amdgcn_mov_dpp(v, 0x150 + N, 0xf, 0xf, true);  // row_newbcast:N
}
template <int N> __device__ __forceinline__ float row16(float v) {
    return __builtin_bit_cast(float, row16<N>(__builtin_bit_cast(int, v)));
}
template <int N> __device__ __forceinline__ double row16(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)row16<N>((int)(unsigned)u), hi = (unsigned)row16<N>((int)(unsigned)(u >> 32));
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Lane exchange of one supernode of at most KM columns: sixteen lanes and
// four supernodes to a wave (KM = 16), or the whole wave (KM = 32, uniform
// reads of one lane).
template <typename T, int KM, int N> __device__ __forceinline__ T from_row(T v) {
    if constexpr (KM == 16) return row16<N>(v);
    else return rlane(v, N);
}

template <typename T, int KM>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(KM == 16 ? 4 : 3))) void k_potrf_narrow(DevSymbol S, const int32_t *__restrict__ cblks, int n,
                                                     T *__restrict__ coef, T *__restrict__ winv,
                                                     T *__restrict__ winvt, double thr, int *stat) {
    __builtin_amdgcn_s_setprio(3);
    constexpr int PW = KM == 16 ? 4 : 1;  // supernodes of a wave
    const int lane = threadIdx.x, i = KM == 16 ? (lane & 15) : lane;
    const int id = blockIdx.x * PW + (KM == 16 ? (lane >> 4) : 0);
    int K = 0;
    int64_t ld = 0, wo = 0;
    T *P = coef;
    if (id < n) {
        const int c = cblks[id];
        K = S.cblk_fcol[c + 1] - S.cblk_fcol[c];
        ld = S.cblk_stride[c];
        P = coef + S.cblk_coef[c];
        wo = S.cblk_winv[c];
    }
    T a[KM];
#pragma unroll
    for (int j = 0; j < KM; j++) a[j] = (i < K && j <= i) ? P[i + (int64_t)j * ld] : (i == j) ? (T)1 : (T)0;
    // columns of the wave's widest supernode: the padding after them is skipped
    int km = __builtin_amdgcn_readfirstlane(K);
    if constexpr (KM == 16)
        for (int g = 1; g < 4; g++) km = max(km, __builtin_amdgcn_readlane(K, 16 * g));
    const T crit = (T)thr;
    int npiv = 0, neg = 0;
    T dia = (T)1;  // this row's diagonal entry
    static_for<0, KM>([&](auto kk) {
        constexpr int k = kk;
        if (k >= km) return;  // uniform
        const T d = from_row<T, KM, k>(a[k]);
        int np = 0, ng = 0;
        T L, r;
        sqrt_rsqrt(piv_max(d, crit, np, ng), L, r);
        npiv += (k < K) ? np : 0;
        neg |= (k < K) ? ng : 0;
        if (i == k) dia = L;
        a[k] = (i == k) ? L : a[k] * r;
        static_for<k + 1, KM>([&](auto jj) {
            constexpr int j = jj;
            a[j] = fma_(-a[k], from_row<T, KM, j>(a[k]), a[j]);
        });
    });
#pragma unroll
    for (int j = 0; j < KM; j++)
        if (i < K && j <= i) P[i + (int64_t)j * ld] = a[j];
    if (i == 0) {
        if (npiv) atomicAdd(&stat[0], npiv);
        if (neg) atomicOr(&stat[1], 1);
    }
    const T di = recip(dia);
    T x[KM];
    static_for<0, KM>([&](auto rr) {
        constexpr int r = rr;
        if (r >= km) return;  // uniform
        T v = (i == r) ? (T)1 : (T)0;
        static_for<0, r>([&](auto kk) {
            constexpr int k = kk;
            v = fma_(-from_row<T, KM, r>(a[k]), x[k], v);
        });
        x[r] = v * from_row<T, KM, r>(di);
    });
    if (i < K) {
        T *W = winv + wo, *WT = winvt + wo;
#pragma unroll
        for (int r = 0; r < KM; r++)
            if (r < K) {
                W[r + (int64_t)i * K] = x[r];
                WT[i + (int64_t)r * K] = x[r];
            }
    }
}

// rows [r0, r0+64) of cblk c below the diagonal sub-block kb: X = A * W_kk^T
// (all 256 threads; contains barriers)
template <typename T>
__device__ __forceinline__ void panel_trsm_tile(const DevSymbol &S, const int c, const int r0, int kb,
                                                T *__restrict__ coef, const T *__restrict__ winv,
                                                StageBuf<T, 16> &sb) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    const int K = S.cblk_fcol[c + 1] - S.cblk_fcol[c];
    const int stride = S.cblk_stride[c];
    const int64_t ld = stride;
    const int k0 = kb * 64, nb = min(64, K - k0);
    T *P = coef + S.cblk_coef[c];
    const T *W = winv + S.cblk_winv[c];
    const int mr = min(64, stride - r0);
    Quad<T> q;
    q.zero();
    // the row tile is read completely (staged through LDS) before it is overwritten
    wg_gemm_lds<T, 16>(q, P + r0 + (int64_t)k0 * ld, mr, ld, W + k0 + (int64_t)k0 * K, nb, K, nb, sb, tid);
    if (wr < mr && wc < nb) {
        QFOR(if (qrow < mr - wr && qcol < nb - wc) P[(r0 + wr + qrow) + (int64_t)(k0 + wc + qcol) * ld] = q.c[m_][n_][r_];)
    }
}

// blockIdx.y selects the side: (coef, winv), or (coef2, winv2) for the
// second panel of LU (both sides of a step in one launch: they write
// different panels and read only the step's diagonal inverses)
template <typename T>
__global__ __launch_bounds__(256) void k_panel_trsm(DevSymbol S, const PanelItem *__restrict__ items, int nitems,
                                                    int kb, T *__restrict__ coef, const T *__restrict__ winv,
                                                    T *__restrict__ coef2, const T *__restrict__ winv2) {
    __builtin_amdgcn_s_setprio(3);
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    __shared__ StageBuf<T, 16> sb;
    const PanelItem it = items[id];
    if (blockIdx.y == 0) panel_trsm_tile<T>(S, it.c, it.r0, kb, coef, winv, sb);
    else panel_trsm_tile<T>(S, it.c, it.r0, kb, coef2, winv2, sb);
}

// In-cblk update of column block c0 of the panel (item), 64-row tile r0:
//   C[r, c0+j] -= sum_{k in Kr} X[r, k] . Y[c0+j, k]
// left-looking (right = 0: c0 is the step's block kb, Kr = [0, c0), before
// the step) or right-looking (right = 1: c0 is a later block, Kr = the
// columns of block kb, after the step).  C, X, Y are panels of the same cblk:
// all L for LL^t; L, L, U and U, U, L for the two sides of LU; the
// reference's blocked potrf/getrf applies the same products,
// kernels/core_zpotrfsp.c:178-185.  On a block's diagonal tile (r0 == c0)
// only r >= c (strict = 0) or r > c (strict = 1) is written: the L side of LU
// keeps the lower part and the diagonal, the U side (transposed) the strict
// upper part.
template <typename T>
__device__ __forceinline__ void panel_upd_tile(const DevSymbol &S, const PanelItem it, int kb, int right,
                                               T *__restrict__ ccoef, const T *__restrict__ xcoef,
                                               const T *__restrict__ ycoef, int strict) {
    __shared__ StageBuf<T, 16> sb;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    const int c = it.c, r0 = it.r0, c0 = it.c0;
    const int K = S.cblk_fcol[c + 1] - S.cblk_fcol[c];
    const int stride = S.cblk_stride[c];
    const int64_t ld = stride;
    const int ks = right ? kb * 64 : 0, kn = right ? min(64, K - ks) : c0;
    T *P = ccoef + S.cblk_coef[c];
    const T *X = xcoef + S.cblk_coef[c] + (int64_t)ks * ld, *Y = ycoef + S.cblk_coef[c] + (int64_t)ks * ld;
    const int mr = min(64, stride - r0), mc = min(64, K - c0);
    Quad<T> q;
    q.zero();
    wg_gemm_lds<T, 16>(q, X + r0, mr, ld, Y + c0, mc, ld, kn, sb, tid);
    if (wr < mr && wc < mc) {
        const bool diag = r0 == c0;
        T *C = P + (r0 + wr) + (int64_t)(c0 + wc) * ld;
        quad_sub(q, lane, [&](int qrow, int qcol, bool &ok) -> T * {
            ok = qrow < mr - wr && qcol < mc - wc && (!diag || wr + qrow > wc + qcol - (strict ? 0 : 1));
            return ok ? C + qrow + (int64_t)qcol * ld : C;
        });
    }
}

// blockIdx.y = 1: the other side of LU, C = Y = ycoef's panel, X = xcoef's,
// strict (the two sides write different panels and read only the blocks
// the step does not write)
template <typename T>
__global__ __launch_bounds__(256) void k_panel_upd(DevSymbol S, const PanelItem *__restrict__ items, int nitems,
                                                   int kb, int right, T *__restrict__ ccoef,
                                                   const T *__restrict__ xcoef, T *__restrict__ ycoef,
                                                   int strict) {
    __builtin_amdgcn_s_setprio(3);
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    if (id >= nitems) return;
    if (blockIdx.y == 0) panel_upd_tile<T>(S, items[id], kb, right, ccoef, xcoef, ycoef, strict);
    else panel_upd_tile<T>(S, items[id], kb, right, ycoef, ycoef, xcoef, 1);
}

// One launch for an LL^t panel step's in-cblk update and the diagonal
// factorisation that waits on it.  Right-looking (right = 1): step kb's
// update of the later blocks, and the factorisation of block kb+1;
// left-looking (right = 0): the update of block kb by the blocks before it,
// and the factorisation of block kb.  Workgroups [0, npot) update the
// diagonal tile of the block to factor for cblk cblks[i] and factor it at
// once (potrf64_block); the others apply the rest of the update (items; the
// diagonal tiles of that block are skipped, their workgroup above has them).
// The factorisation no longer waits for the whole update, only for its tile.
template <typename T>
__global__ __launch_bounds__(256) void k_panel_upd_potrf(DevSymbol S, const int32_t *__restrict__ cblks, int npot,
                                                         const PanelItem *__restrict__ items, int nitems, int kb,
                                                         int right, T *__restrict__ coef, T *__restrict__ winv,
                                                         T *__restrict__ winvt, double thr, int *stat) {
    __builtin_amdgcn_s_setprio(3);
    const int id = blockIdx.x;
    const int kf = right ? kb + 1 : kb;  // the block factored here
    const int k1 = 64 * kf;
    if (id < npot) {
        const int c = cblks[id];
        panel_upd_tile<T>(S, PanelItem{c, k1, k1, 0}, kb, right, coef, coef, coef, 0);
        __syncthreads();  // the tile's stores reach the whole workgroup
        __shared__ PotrfLds<T> lds;
        potrf64_block<T>(S, c, kf, coef, winv, winvt, thr, stat, lds);
        return;
    }
    if (id - npot >= nitems) return;
    const PanelItem it = items[id - npot];
    if (it.r0 == k1 && it.c0 == k1) return;
    panel_upd_tile<T>(S, it, kb, right, coef, coef, coef, 0);
}

// Inverses of the solve nodes' diagonal blocks, by recursive doubling.  The
// diagonal-block kernels leave the inverse of every 64-column sub-block of a
// cblk in place (W, and WT = W^T); a merge round joins adjacent column runs
// [a, m) and [m, b) of a node whose inverses X11 and X22 are known:
//   X21 = -X22 M21 X11
// (M21: rows [m, b), columns [a, m) of the node's lower-triangular diagonal
// block), on 64x64 tiles of X21 in two phases: T = M21 X11, stored
// transposed, then X21 = -X22 T, written to W (column-major, lower) and to
// WT.  M is read in the members' panels: node column j lies in member c
// (o = its first node column), node row i >= o is panel row i - o of c
// (a node's members are coupled by full blocks).  k_winv_leaves first copies
// the members' 64-column inverses into the W and WT of nodes of several
// cblks (a node of one cblk already holds them in place).

// D(64x64) += X(64xK) Y(64xK)^T as wg_gemm_lds (K >= 1), where xcol(k) points
// at X(0, k) (rows contiguous; called with increasing k, also for k >= K,
// where it must still point at readable rows) and Y(r, k) = Y[k + r*ldy] (consecutive k contiguous)
template <typename T, int CH, class XCol>
__device__ __forceinline__ void wg_gemm_lds_xcol_yt(Quad<T> &q, XCol &xcol, int mx, const T *Y, int my, int64_t ldy,
                                                    int K, StageBuf<T, CH> &sb, int tid) {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    const int i = lane & 15, kq = lane >> 4;
    constexpr int E = Vec<T>::E, NP = CH / (4 * E), NY = CH / 4;
    const int re = E * (tid % (64 / E)), ke = tid / (64 / E);
    // Y: thread (row yr, k group yk) fetches NY consecutive k of its row
    const int yr = tid & 63, yk = (tid >> 6) * NY;
    const int rx = re < mx ? re : 0;
    const T *py = Y + (int64_t)min(yr, my - 1) * ldy;
    T gx[NP][E], gy[NY];
    auto gload = [&](int k0) {
#pragma unroll
        for (int u = 0; u < NP; u++) ld_vec(xcol(k0 + ke + 4 * E * u) + rx, gx[u]);
#pragma unroll
        for (int e = 0; e < NY; e++) gy[e] = py[min(k0 + yk + e, K - 1)];
    };
    auto sstore = [&](int k0) {
        if (k0 + CH > K) {  // uniform: the last chunk, columns >= K cleared
#pragma unroll
            for (int u = 0; u < NP; u++)
#pragma unroll
                for (int e = 0; e < E; e++)
                    if (k0 + ke + 4 * E * u >= K) gx[u][e] = (T)0;
#pragma unroll
            for (int e = 0; e < NY; e++)
                if (k0 + yk + e >= K) gy[e] = (T)0;
        }
#pragma unroll
        for (int u = 0; u < NP; u++) st_rows(&sb.xs[ke + 4 * E * u][re], gx[u]);
#pragma unroll
        for (int e = 0; e < NY; e++) sb.ys[yk + e][yr] = gy[e];
    };
    const bool active = (wr < mx) && (wc < my);
    gload(0);
    sstore(0);
    __syncthreads();
    for (int k0 = 0; k0 < K; k0 += CH) {
        const bool more = k0 + CH < K;
        if (more) gload(k0 + CH);
        if (active) quad_chunk<T, CH>(q, sb.xs, sb.ys, wr + i, wc + i, K - k0, kq);
        __syncthreads();
        if (more) sstore(k0 + CH);
        __syncthreads();
    }
}

// One workgroup per leaf (64-column block ib of member c of node nd, a node
// of several cblks): the leaf's inverse block into the node's W (and WT).
template <typename T>
__global__ __launch_bounds__(256) void k_winv_leaves(DevSymbol S, const WinvLeaf *__restrict__ leaves,
                                                     T *__restrict__ w, T *__restrict__ wt) {
    const WinvLeaf lf = leaves[blockIdx.x];
    const int tid = threadIdx.x;
    const int nd = lf.nd, c = lf.c;
    const int f0 = S.cblk_fcol[S.node_cblk[nd]];
    const int K = S.cblk_fcol[S.node_cblk[nd + 1]] - f0;
    const int o = S.cblk_fcol[c] - f0, wc = S.cblk_fcol[c + 1] - S.cblk_fcol[c];
    const int j0 = 64 * lf.ib, bw = min(64, wc - j0);
    const int64_t xo = S.node_winv[nd] + (o + j0) + (int64_t)(o + j0) * K;
    const int64_t mo = S.cblk_winv[c] + j0 + (int64_t)j0 * wc;
    // 16 entries per thread, loads first
    T v[16], vt[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int t = tid + 256 * u, i = t & 63, j = t >> 6;
        const bool ok = i < bw && j < bw;
        v[u] = ok ? w[mo + i + (int64_t)j * wc] : (T)0;
        vt[u] = (ok && wt) ? wt[mo + i + (int64_t)j * wc] : (T)0;
    }
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int t = tid + 256 * u, i = t & 63, j = t >> 6;
        if (i < bw && j < bw) {
            w[xo + i + (int64_t)j * K] = v[u];
            if (wt) wt[xo + i + (int64_t)j * K] = vt[u];
        }
    }
}

// columns staged per chunk of the merges' products
constexpr int WINV_CH = 16;

template <typename T, int PHASE>
__global__ __launch_bounds__(256) void k_winv_merge(DevSymbol S, const WinvTile *__restrict__ tiles,
                                                    const T *__restrict__ coef, T *__restrict__ w,
                                                    T *__restrict__ wt, T *__restrict__ tbuf) {
    __shared__ StageBuf<T, WINV_CH> sb;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    const WinvTile t = tiles[blockIdx.x];
    const int nd = t.nd, c0 = S.node_cblk[nd];
    const int f0 = S.cblk_fcol[c0];
    const int K = S.cblk_fcol[S.node_cblk[nd + 1]] - f0;
    const int h1 = t.m - t.a, h2 = t.b - t.m;
    const int mi = min(64, h2 - t.i0), mj = min(64, h1 - t.j0);
    T *X = w + S.node_winv[nd];
    Quad<T> q;
    q.zero();
    if constexpr (PHASE == 1) {
        // T[i0+i, j0+j] = sum_{k >= j0} M[m+i0+i, a+k] X[a+k, a+j0+j], M in
        // the members' panels (the member of a column followed as k grows)
        const int row0 = t.m + t.i0;
        int mc = c0, mend = S.cblk_fcol[c0 + 1] - f0, mo = 0;
        const T *mbase = coef + S.cblk_coef[c0] + row0;
        int64_t mld = S.cblk_stride[c0];
        auto xcol = [&](int k) -> const T * {
            const int gc = min(t.a + t.j0 + k, t.m - 1);
            while (gc >= mend) {
                mc++;
                mo = mend;
                mend = S.cblk_fcol[mc + 1] - f0;
                mbase = coef + S.cblk_coef[mc] + (row0 - mo);
                mld = S.cblk_stride[mc];
            }
            return mbase + (int64_t)(gc - mo) * mld;
        };
        wg_gemm_lds_xcol_yt<T, WINV_CH>(q, xcol, mi, X + (t.a + t.j0) + (int64_t)(t.a + t.j0) * K, mj, K, h1 - t.j0, sb,
                                   tid);
        T *Tt = tbuf + t.toff;
        QFOR(if (wr + qrow < mi && wc + qcol < mj)
                 Tt[(t.j0 + wc + qcol) + (int64_t)(t.i0 + wr + qrow) * h1] = q.c[m_][n_][r_];)
    } else {
        // X[m+i0+i, a+j0+j] = -sum_{k <= i0+i} X[m+i0+i, m+k] T[k, j0+j]
        wg_gemm_lds<T, WINV_CH>(q, X + (t.m + t.i0) + (int64_t)t.m * K, mi, K, tbuf + t.toff + t.j0, mj, h1,
                           min(t.i0 + 64, h2), sb, tid);
        T *XT = wt ? wt + S.node_winv[nd] : nullptr;
        QFOR(if (wr + qrow < mi && wc + qcol < mj) {
            const int gi = t.m + t.i0 + wr + qrow, gj = t.a + t.j0 + wc + qcol;
            const T v = -q.c[m_][n_][r_];
            X[gi + (int64_t)gj * K] = v;
            if (XT) XT[gj + (int64_t)gi * K] = v;
        })
    }
}

// Entry (r, c) of a lower-triangular matrix of the LU pair packed in X: the
// unit lower L (strictly below the diagonal), or with UT the transpose of U
// (U on and above the diagonal).
template <typename T, bool UT> __device__ __forceinline__ T &lu_at(T (*X)[65], int r, int c) {
    return UT ? X[c][r] : X[r][c];
}
template <typename T, bool UT> __device__ __forceinline__ T lu_tri(T (*X)[65], int r, int c) {
    const T v = lu_at<T, UT>(X, r, c);
    return r > c ? v : r < c ? (T)0 : UT ? v : (T)1;
}

// One joining level for one of the two matrices (see lower_inverse):
// PHASE 1: Ts = M21 X11, PHASE 2: X21 = -X22 Ts; output o of 32 B on the
// vector units, 16x16 tile t on the matrix cores.
template <typename T, bool UT, int B, int PHASE>
__device__ __forceinline__ void lu_join_valu(T (*X)[65], T *Ts, int o) {
    const int p = o / (B * B), rem = o % (B * B), r = rem / B, cc = rem % B, base = 2 * B * p;
    T s = (T)0;
#pragma unroll
    for (int m = 0; m < B; m++) {
        if (PHASE == 1) s = fma_(lu_at<T, UT>(X, base + B + r, base + m), lu_tri<T, UT>(X, base + m, base + cc), s);
        else s = fma_(lu_tri<T, UT>(X, base + B + r, base + B + m), Ts[p * B * B + m * B + cc], s);
    }
    if (PHASE == 1) Ts[o] = s;
    else lu_at<T, UT>(X, base + B + r, base + cc) = -s;
}
template <typename T, bool UT, int B, int PHASE>
__device__ __forceinline__ void lu_join_mfma(T (*X)[65], T *Ts, int lane, int t) {
    constexpr int TPP = (B / 16) * (B / 16);
    const int i = lane & 15, kq = lane >> 4;
    const int p = t / TPP, ti = (t % TPP) / (B / 16) * 16, tj = t % (B / 16) * 16, base = 2 * B * p;
    typename Mfma<T>::v4 acc = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < B / 4; s++) {
        const int k = 4 * s + kq;
        if (PHASE == 1)
            acc = Mfma<T>::mma(lu_at<T, UT>(X, base + B + ti + i, base + k), lu_tri<T, UT>(X, base + k, base + tj + i),
                               acc);
        else
            acc = Mfma<T>::mma(lu_tri<T, UT>(X, base + B + ti + i, base + B + k), Ts[p * B * B + k * B + tj + i], acc);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int row = ti + Mfma<T>::drow(lane, r);
        if (PHASE == 1) Ts[p * B * B + row * B + tj + i] = acc[r];
        else lu_at<T, UT>(X, base + B + row, base + tj + i) = -acc[r];
    }
}

// The 4x4 diagonal blocks of one of the two (lane: 4 columns of 16 blocks).
template <typename T, bool UT> __device__ __forceinline__ void lu_inv4(T (*X)[65], const T *dinv, int lane) {
    const int b0 = 4 * (lane >> 2), cc = lane & 3;
    auto M = [&](int r, int c) -> T { return lu_at<T, UT>(X, b0 + r, b0 + c); };
    const T m10 = M(1, 0), m20 = M(2, 0), m21 = M(2, 1), m30 = M(3, 0), m31 = M(3, 1), m32 = M(3, 2);
    const T d0 = UT ? dinv[b0] : (T)1, d1 = UT ? dinv[b0 + 1] : (T)1;
    const T d2 = UT ? dinv[b0 + 2] : (T)1, d3 = UT ? dinv[b0 + 3] : (T)1;
    const T x0 = (cc == 0) ? d0 : (T)0;
    const T x1 = (cc > 1) ? (T)0 : (cc == 1) ? d1 : -(m10 * x0) * d1;
    const T x2 = (cc > 2) ? (T)0 : (cc == 2) ? d2 : -fma_(m21, x1, m20 * x0) * d2;
    const T x3 = (cc == 3) ? d3 : -fma_(m32, x2, fma_(m31, x1, m30 * x0)) * d3;
    const int first = UT ? cc : cc + 1;  // L's unit diagonal is implied
    if (first <= 0) lu_at<T, UT>(X, b0, b0 + cc) = x0;
    if (first <= 1) lu_at<T, UT>(X, b0 + 1, b0 + cc) = x1;
    if (first <= 2) lu_at<T, UT>(X, b0 + 2, b0 + cc) = x2;
    if (first <= 3) lu_at<T, UT>(X, b0 + 3, b0 + cc) = x3;
}

// inv(L) and inv(U)^T of the LU pair packed in X, in place, by the steps of
// lower_inverse: the two go side by side, so that together they take the
// barriers of one (the unit diagonal of L and the zeros beyond the triangles
// are implied).  Ts: 2048 entries of scratch.
template <typename T>
__device__ __forceinline__ void lu_inverse(T (*X)[65], T *Ts, const T *dinv, int nb, int tid, int w) {
    T *const TL = Ts, *const TU = Ts + 1024;
    const int lane = tid & 63;
    if (w == 0) lu_inv4<T, false>(X, dinv, lane);
    else if (w == 1) lu_inv4<T, true>(X, dinv, lane);
    __syncthreads();
#define LU_JOIN(PHASE)                                                        \
    if (w < 2) lu_join_valu<T, false, 4, PHASE>(X, TL, tid);                  \
    else lu_join_valu<T, true, 4, PHASE>(X, TU, tid - 128);                   \
    __syncthreads();
    if (nb > 4) {
        LU_JOIN(1)
        LU_JOIN(2)
    }
#undef LU_JOIN
#define LU_JOIN(PHASE)                                \
    lu_join_valu<T, false, 8, PHASE>(X, TL, tid);     \
    lu_join_valu<T, true, 8, PHASE>(X, TU, tid);      \
    __syncthreads();
    if (nb > 8) {
        LU_JOIN(1)
        LU_JOIN(2)
    }
#undef LU_JOIN
#define LU_JOIN(PHASE)                                               \
    if (w < 2) lu_join_mfma<T, false, 16, PHASE>(X, TL, lane, w);    \
    else lu_join_mfma<T, true, 16, PHASE>(X, TU, lane, w - 2);       \
    __syncthreads();
    if (nb > 16) {
        LU_JOIN(1)
        LU_JOIN(2)
    }
#undef LU_JOIN
#define LU_JOIN(PHASE)                                   \
    lu_join_mfma<T, false, 32, PHASE>(X, TL, lane, w);   \
    lu_join_mfma<T, true, 32, PHASE>(X, TU, lane, w);    \
    __syncthreads();
    if (nb > 32) {
        LU_JOIN(1)
        LU_JOIN(2)
    }
#undef LU_JOIN
}

// LU without pivoting of one 64-column diagonal sub-block (reference
// kernels/core_zgetrfsp.c:63-106, getf2 with static pivoting +-thr).  During
// the factorisation the square part of a cblk keeps its lower triangle
// (diagonal included) in the L panel and its strict upper triangle,
// transposed, in the U panel.  Thread (i, w) keeps the entries (i, j),
// j = w mod 4, of row i of the full sub-block; the elimination runs by
// blocks of four columns with one barrier each.  Outputs: L (unit, strict lower) and the diagonal of U
// in the L panel, the strict upper part of U transposed in the U panel,
// W1 = inv(L) (lower, unit diagonal), W2 = inv(U)^T (lower) and WB = inv(U)
// (upper), with explicit zeros in the other triangles of the sub-block; the
// inverses come from lu_inverse.
//
// Bound by the latency of its 16 steps and the joins.  With the rows of U
// published through LDS and read back per column, the two inverses one after
// the other and the U panel's triangle walked across columns, 16 blocks took
// 44.7 us in FP64 and 35.9 in FP32, 2048 blocks 173 and 95; now 31.5 and
// 26.6, 136 and 79 (same roundings).
template <typename T>
__global__ __launch_bounds__(256) void k_getrf64(DevSymbol S, const int32_t *__restrict__ cblks, int kb,
                                                 T *__restrict__ lcoef, T *__restrict__ ucoef, T *__restrict__ w1,
                                                 T *__restrict__ w2, T *__restrict__ wb, double thr, int *stat) {
    __builtin_amdgcn_s_setprio(3);
    __shared__ T fac[2048];
    T(*colb)[4][64] = reinterpret_cast<T(*)[4][64]>(fac);  // [parity][w][row]
    __shared__ T Ls[64][65];                               // L below the diagonal, U from it
    __shared__ T dinv[64];
    const int tid = threadIdx.x, i = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = cblks[blockIdx.x];
    const int K = S.cblk_fcol[c + 1] - S.cblk_fcol[c];
    const int k0 = kb * 64;
    const int nb = min(64, K - k0);
    const int64_t ld = S.cblk_stride[c];
    T *PL = lcoef + S.cblk_coef[c] + k0 + (int64_t)k0 * ld;
    T *PU = ucoef + S.cblk_coef[c] + k0 + (int64_t)k0 * ld;
    // both triangles walked down columns, into rows through LDS; the padding
    // up to 64 is the identity
    {
        T vl[16], vu[16];
        const int64_t row = min(i, nb - 1);
#pragma unroll
        for (int u = 0; u < 16; u++) {
            const int64_t o = row + min(4 * u + w, nb - 1) * ld;
            vl[u] = PL[o];
            vu[u] = PU[o];
        }
#pragma unroll
        for (int u = 0; u < 16; u++) {
            const int j = 4 * u + w;
            const bool pad = i >= nb || j >= nb;
            if (i >= j) Ls[i][j] = !pad ? vl[u] : (i == j) ? (T)1 : (T)0;
            if (i > j) Ls[j][i] = !pad ? vu[u] : (T)0;
        }
    }
    __syncthreads();
    T a[16];
#pragma unroll
    for (int jj = 0; jj < 16; jj++) a[jj] = Ls[i][4 * jj + w];
    const T crit = (T)thr;
    int npiv = 0;
    auto piv = [&](T d, int col) -> T {
        const bool small = col < nb && pabs(d) < crit;
        npiv += small;
        return small ? ((d < (T)0) ? -crit : crit) : d;
    };
    // Blocks of 4 columns k..k+3, as in potrf64_block: the columns are
    // published through LDS, every thread eliminates the 4x4 diagonal block,
    // and row i forms its 4 multipliers.  The block's rows of U in a column
    // are held by lanes k..k+3 of the wave that owns the column: with the
    // multipliers of those rows being the block's own L (0 in the rows above),
    // one formula leaves U in them and the Schur complement below, reading
    // each pivot row across lanes once it is done.  The four products are
    // summed before they are subtracted: every entry is rounded once per
    // block (four subtractions in turn doubled the factor's error).  The next
    // block's columns go first, the others overlap its 4x4 chain.
    T p0 = 0, p1 = 0, p2 = 0, p3 = 0;  // this row's multipliers of the last block
    auto rank4 = [&](T x, int k) -> T {
        T s = p0 * rlane(x, k);
        s = fma_(p1, rlane(x - s, k + 1), s);
        s = fma_(p2, rlane(x - s, k + 2), s);
        s = fma_(p3, rlane(x - s, k + 3), s);
        return x - s;
    };
    colb[0][w][i] = a[0];
#pragma unroll
    for (int b4 = 0; b4 < 16; b4++) {
        const int k = 4 * b4;
        if (k >= nb) break;  // uniform: the padding needs no elimination
        __syncthreads();
        int ii = i;  // opaque: see potrf64_block
        asm volatile("" : "+v"(ii));
        T(*cb)[64] = colb[b4 & 1];
        // D(t, u) = cb[u][k + t]
        const T d00 = cb[0][k], d10 = cb[0][k + 1], d20 = cb[0][k + 2], d30 = cb[0][k + 3];
        const T u01 = cb[1][k], d11 = cb[1][k + 1], d21 = cb[1][k + 2], d31 = cb[1][k + 3];
        const T u02 = cb[2][k], d12 = cb[2][k + 1], d22 = cb[2][k + 2], d32 = cb[2][k + 3];
        const T u03 = cb[3][k], d13 = cb[3][k + 1], d23 = cb[3][k + 2], d33 = cb[3][k + 3];
        const T e0 = cb[0][ii], e1 = cb[1][ii], e2 = cb[2][ii], e3 = cb[3][ii];
        if (b4 >= 1) {
#pragma unroll
            for (int jj = b4 + 1; jj < 16; jj++) a[jj] = rank4(a[jj], k - 4);
        }
        const T u00 = piv(d00, k), r0 = recip(u00);
        const T l10 = d10 * r0, l20 = d20 * r0, l30 = d30 * r0;
        const T u11 = piv(d11 - l10 * u01, k + 1), r1 = recip(u11);
        const T u12 = d12 - l10 * u02, u13 = d13 - l10 * u03;
        const T l21 = (d21 - l20 * u01) * r1, l31 = (d31 - l30 * u01) * r1;
        const T u22 = piv(d22 - l20 * u02 - l21 * u12, k + 2), r2 = recip(u22);
        const T u23 = d23 - l20 * u03 - l21 * u13;
        const T l32 = (d32 - l30 * u02 - l31 * u12) * r2;
        const T u33 = piv(d33 - l30 * u03 - l31 * u13 - l32 * u23, k + 3), r3 = recip(u33);
        asm volatile("" : "+v"(npiv));
        const T m0 = e0 * r0;
        const T m1 = (e1 - m0 * u01) * r1;
        const T m2 = (e2 - m0 * u02 - m1 * u12) * r2;
        const T m3 = (e3 - m0 * u03 - m1 * u13 - m2 * u23) * r3;
        const int t = ii - k;
        const bool below = t > 3;
        p0 = below ? m0 : (t == 1) ? l10 : (t == 2) ? l20 : (t == 3) ? l30 : (T)0;
        p1 = below ? m1 : (t == 2) ? l21 : (t == 3) ? l31 : (T)0;
        p2 = below ? m2 : (t == 3) ? l32 : (T)0;
        p3 = below ? m3 : (T)0;
        // the block's own columns: L strictly left of the diagonal, U from it
        T f;
        if (w == 0) f = (t == 0) ? u00 : p0;
        else if (w == 1) f = (t == 0) ? u01 : (t == 1) ? u11 : p1;
        else if (w == 2) f = (t == 0) ? u02 : (t == 1) ? u12 : (t == 2) ? u22 : p2;
        else f = (t == 0) ? u03 : (t == 1) ? u13 : (t == 2) ? u23 : (t == 3) ? u33 : p3;
        if (t >= 0) a[b4] = f;
        if (b4 < 15) {
            a[b4 + 1] = rank4(a[b4 + 1], k);
            colb[(b4 + 1) & 1][w][ii] = a[b4 + 1];
        }
    }
#pragma unroll
    for (int jj = 0; jj < 16; jj++) Ls[i][4 * jj + w] = a[jj];
    if (tid == 0 && npiv) atomicAdd(&stat[0], npiv);
    __syncthreads();
    if (w == 0) dinv[i] = recip(Ls[i][i]);
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int j = 4 * u + w;
        if (i < nb && j < nb) {
            if (i >= j) PL[i + j * ld] = Ls[i][j];
            if (i > j) PU[i + j * ld] = Ls[j][i];
        }
    }
    __syncthreads();
    lu_inverse<T>(Ls, fac, dinv, nb, tid, w);
    T *W1 = w1 + S.cblk_winv[c] + k0 + (int64_t)k0 * K;
    T *W2 = w2 + S.cblk_winv[c] + k0 + (int64_t)k0 * K;
    T *WB = wb + S.cblk_winv[c] + k0 + (int64_t)k0 * K;
#pragma unroll 4
    for (int u = 0; u < 16; u++) {
        const int j = 4 * u + w;
        if (i < nb && j < nb) {
            W1[i + (int64_t)j * K] = lu_tri<T, false>(Ls, i, j);
            W2[i + (int64_t)j * K] = lu_tri<T, true>(Ls, i, j);
            WB[i + (int64_t)j * K] = lu_tri<T, true>(Ls, j, i);
        }
    }
}

// The square parts of the LU panels, by 64x64 tiles on and below the
// diagonal (item: rows [r0, r0+64), columns [c0, c0+64) of cblk c's square,
// r0 >= c0) and their mirror images above it.  Bound by memory: each tile
// crosses LDS so that both the tile and its mirror are walked down columns.
// One workgroup per cblk with the transposed side read across columns took
// 135 us per level and 353 us for the layout on the 48^3 27-point operator
// (FP64, beside the updates of the second stream); these take 21 and 71 us.

// Before the LU panel of a cblk: the square part's upper triangle arrives
// split between the L panel (same-block Schur contributions, written above
// the diagonal as the reference does) and the U panel (transposed): the
// reference adds them (core_zgeadd, kernels/core_zgetrfsp.c:240-242); here
// the sum goes to the U panel and the L panel keeps the lower triangle only.
template <typename T>
__global__ __launch_bounds__(256) void k_lu_square_merge(DevSymbol S, const PanelItem *__restrict__ items,
                                                         T *__restrict__ lcoef, T *__restrict__ ucoef) {
    __shared__ T tile[64][65];
    const PanelItem it = items[blockIdx.x];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int K = S.cblk_fcol[it.c + 1] - S.cblk_fcol[it.c];
    const int64_t ld = S.cblk_stride[it.c];
    T *PL = lcoef + S.cblk_coef[it.c], *PU = ucoef + S.cblk_coef[it.c];
    // L(r, cc), r < cc: rows r = c0 + lane of columns cc = r0 + j
    const int r = it.c0 + lane;
    T v[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int cc = it.r0 + w + 4 * u;
        v[u] = (r < cc && cc < K) ? PL[r + (int64_t)cc * ld] : (T)0;
    }
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int cc = it.r0 + w + 4 * u;
        if (r < cc && cc < K) PL[r + (int64_t)cc * ld] = (T)0;
        tile[w + 4 * u][lane] = v[u];
    }
    __syncthreads();
    // added to U^T(cc, r): rows cc = r0 + lane of columns r = c0 + i
    const int cc = it.r0 + lane;
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int q = it.c0 + w + 4 * u;
        v[u] = (q < cc && cc < K) ? PU[cc + (int64_t)q * ld] : (T)0;
    }
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int q = it.c0 + w + 4 * u;
        if (q < cc && cc < K) PU[cc + (int64_t)q * ld] = v[u] + tile[lane][w + 4 * u];
    }
}

// Final layout of the LU diagonal blocks (reference core_zgetrfsp.c:240-251):
// the L panel's square receives the whole LU (strict upper part from the U
// panel, where it was kept transposed) and the U panel's square its
// transpose (core_zgetmo).  The lower triangles stay, so every entry moves
// once: L(j, i) = U^T(i, j) and U^T(j, i) = L(i, j) for i > j, and the
// diagonal of U^T is L's.
template <typename T>
__global__ __launch_bounds__(256) void k_lu_square_layout(DevSymbol S, const PanelItem *__restrict__ items,
                                                          T *__restrict__ lcoef, T *__restrict__ ucoef) {
    __shared__ T tl[64][65], tu[64][65];
    const PanelItem it = items[blockIdx.x];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int K = S.cblk_fcol[it.c + 1] - S.cblk_fcol[it.c];
    const int64_t ld = S.cblk_stride[it.c];
    T *PL = lcoef + S.cblk_coef[it.c], *PU = ucoef + S.cblk_coef[it.c];
    // the lower tile: rows i = r0 + lane of columns j
    const int i = it.r0 + lane;
    T a[16], b[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int j = it.c0 + w + 4 * u;
        const bool ok = i < K && j <= i;
        a[u] = ok ? PL[i + (int64_t)j * ld] : (T)0;
        b[u] = ok ? PU[i + (int64_t)j * ld] : (T)0;
    }
#pragma unroll
    for (int u = 0; u < 16; u++) {
        tl[w + 4 * u][lane] = a[u];
        tu[w + 4 * u][lane] = b[u];
    }
    __syncthreads();
    // its mirror: rows j = c0 + lane of columns i
    const int j = it.c0 + lane;
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int q = it.r0 + w + 4 * u;
        if (q < K && j <= q) {
            PU[j + (int64_t)q * ld] = tl[lane][w + 4 * u];
            if (j < q) PL[j + (int64_t)q * ld] = tu[lane][w + 4 * u];
        }
    }
}

// ---------------------------------------------------------------------------
// Leaf region: one persistent launch whose tasks are driven by device-side
// dependency counters (reference kernels/cpucblk_zmpi_coeftab.c:482-562,
// cpucblk_zincoming_deps / cpucblk_zrelease_deps, with counters as
// blend/solver_backup.c:95-101 sets them, and the ready queue of the dynamic
// scheduler, sopalin/sequential_zpotrf.c:129-234).
//
// A task is one region cblk c (at most 64 columns): it pulls the updates of
// every region cblk facing it (its incoming tiles, entries in source order,
// owner computes: no other workgroup writes c), factors the diagonal block
// with its inverse, solves the rows below, then decrements the counter of
// every region cblk it faces; the decrement that reaches zero appends that
// cblk to the ready queue.  Workgroups take queue slots in order with one
// atomic; a slot's cblk is published with a release store once its counter
// reaches zero.  Every cblk enters the queue exactly once, and a taken slot
// whose cblk is not yet published waits only for tasks taken before it, all
// of them running on workgroups that wait for nothing: the queue drains
// whatever the number of resident workgroups.  Every wait is bounded: after
// `maxwait` ticks of the constant-rate wall clock without its slot being
// published a workgroup sets stat[2], every workgroup leaves, and the host
// reports the error.
//
// Memory ordering: a task's stores are released at agent scope by every wave
// (the writes of other compute units' L2 become visible to the consumer),
// the counter decrement a release, the last decrement's thread acquires the
// earlier ones before the release store of the queue slot, and the consumer
// polls the slot with relaxed loads, then takes one acquire fence; the other
// waves of its workgroup are ordered after that fence by the barrier.
// sync[0]: next queue slot to take, sync[1]: next slot to publish.
template <typename T> union LeafLds {
    UpdAccLds<T> u;
    PotrfLds<T> p;
};

__global__ __launch_bounds__(256) void k_leaf_init(LeafDev LP, int32_t *__restrict__ ctr,
                                                   int32_t *__restrict__ queue, int32_t *__restrict__ sync) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < LP.cblknbr) ctr[i] = LP.ctr0[i];
    if (i < LP.nregion) queue[i] = (i < LP.ninit) ? LP.init[i] : -1;
    if (i == 0) {
        sync[0] = 0;
        sync[1] = LP.ninit;
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_leaf_tasks(DevSymbol S, LeafDev LP, const UpdEntry *__restrict__ ents,
                                                    const int32_t *__restrict__ shift, T *__restrict__ coef,
                                                    T *__restrict__ winv, T *__restrict__ winvt, double thr,
                                                    int *stat, int32_t *__restrict__ ctr,
                                                    int32_t *__restrict__ queue, int32_t *__restrict__ sync,
                                                    long long maxwait) {
    __shared__ LeafLds<T> lds;
    __shared__ int task;
    const int tid = threadIdx.x;
    for (;;) {
        if (tid == 0) {
            int c = -1;
            const int t = __hip_atomic_fetch_add(&sync[0], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (t < LP.nregion) {
                // relaxed polls (an acquire load would invalidate the L2 on
                // every poll), one acquire fence once the slot is published;
                // the wait is bounded in time (constant-rate wall clock)
                const unsigned long long t0 = wall_clock64();
                for (;;) {
                    c = __hip_atomic_load(&queue[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (c >= 0) break;
                    if (__hip_atomic_load(&stat[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
                        wall_clock64() - t0 > (unsigned long long)maxwait) {
                        __hip_atomic_store(&stat[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        c = -1;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(8);
                }
                if (c >= 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            }
            task = c;
        }
        __syncthreads();
        const int c = task;
        __syncthreads();  // every thread holds the task before thread 0 takes the next one
        if (c < 0 || c >= LP.cblknbr) break;
        // incoming updates (each tile ends with a barrier after its stores)
        for (int k = LP.in_ptr[c]; k < LP.in_ptr[c + 1]; k++)
            update_acc_tile<T, 0>(S, LP.in[k], ents, shift, coef, coef, coef, lds.u);
        // the diagonal block and its inverse, then the rows below it
        potrf64_block<T>(S, c, 0, coef, winv, winvt, thr, stat, lds.p);
        __syncthreads();
        const int K = S.cblk_fcol[c + 1] - S.cblk_fcol[c];
        const int stride = S.cblk_stride[c];
        for (int r0 = K; r0 < stride; r0 += 64) {
            panel_trsm_tile<T>(S, c, r0, 0, coef, winv, lds.u.sb);
            __syncthreads();
        }
        // release the panel and the inverse, then the counters it feeds
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __syncthreads();
        if (tid == 0) {
            for (int k = LP.tgt_ptr[c]; k < LP.tgt_ptr[c + 1]; k++) {
                const int f = LP.tgt[k];
                // release: this task's writes (fenced above by every wave);
                // the last decrement also acquires the earlier ones before it
                // publishes f
                if (__hip_atomic_fetch_add(&ctr[f], -1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT) == 1) {
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                    const int pos = __hip_atomic_fetch_add(&sync[1], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (pos < LP.nregion) __hip_atomic_store(&queue[pos], f, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
                    else __hip_atomic_store(&stat[2], 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
    }
}

// ------------------------------- launchers ---------------------------------
static inline int grid8(int n) { return ((n + 7) / 8) * 8; }

template <typename T>
void launch_potrf64(const DevSymbol &S, const int32_t *cblks, int n, int kb, int maxwidth, T *coef, T *winv, T *winvt,
                    double thr, int *stat, hipStream_t st) {
    if (n <= 0) return;
    // at most 16 columns: 8 to 40 us (16,384 supernodes), k_potrf64 17 to 523
    if (kb == 0 && maxwidth <= 16) {
        hipLaunchKernelGGL((k_potrf_narrow<T, 16>), dim3((n + 3) / 4), dim3(64), 0, st, S, cblks, n, coef, winv, winvt,
                           thr, stat);
        return;
    }
    // up to 32 columns the whole wave takes one: 30 us however few there are
    // (its 32 pivots follow each other), where k_potrf64 takes 20 us for up to
    // some 500 supernodes and 40 us more for every 1024 (FP64)
    if (kb == 0 && maxwidth <= 32 && n >= 1024) {
        hipLaunchKernelGGL((k_potrf_narrow<T, 32>), dim3(n), dim3(64), 0, st, S, cblks, n, coef, winv, winvt, thr,
                           stat);
        return;
    }
    hipLaunchKernelGGL(k_potrf64<T>, dim3(n), dim3(256), 0, st, S, cblks, kb, coef, winv, winvt, thr, stat);
}
template <typename T>
void launch_getrf64(const DevSymbol &S, const int32_t *cblks, int n, int kb, T *lcoef, T *ucoef, T *w1, T *w2, T *wb,
                    double thr, int *stat, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_getrf64<T>, dim3(n), dim3(256), 0, st, S, cblks, kb, lcoef, ucoef, w1, w2, wb, thr, stat);
}
template <typename T>
void launch_lu_square_merge(const DevSymbol &S, const PanelItem *items, int n, T *lcoef, T *ucoef, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_lu_square_merge<T>, dim3(n), dim3(256), 0, st, S, items, lcoef, ucoef);
}
template <typename T>
void launch_lu_square_layout(const DevSymbol &S, const PanelItem *items, int n, T *lcoef, T *ucoef, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_lu_square_layout<T>, dim3(n), dim3(256), 0, st, S, items, lcoef, ucoef);
}
template <typename T>
void launch_panel_trsm(const DevSymbol &S, const PanelItem *items, int n, int kb, T *coef, const T *winv,
                       hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_panel_trsm<T>, dim3(grid8(n)), dim3(256), 0, st, S, items, n, kb, coef, winv, coef, winv);
}
template <typename T>
void launch_panel_trsm2(const DevSymbol &S, const PanelItem *items, int n, int kb, T *coef, const T *winv, T *coef2,
                        const T *winv2, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_panel_trsm<T>, dim3(grid8(n), 2), dim3(256), 0, st, S, items, n, kb, coef, winv, coef2,
                       winv2);
}
template <typename T>
void launch_panel_upd(const DevSymbol &S, const PanelItem *items, int n, int kb, bool right, T *C, const T *X,
                      const T *Y, bool strict, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_panel_upd<T>, dim3(grid8(n)), dim3(256), 0, st, S, items, n, kb, right ? 1 : 0, C, X,
                       const_cast<T *>(Y), strict ? 1 : 0);
}
template <typename T>
void launch_panel_upd_lu(const DevSymbol &S, const PanelItem *items, int n, int kb, bool right, T *L, T *U,
                         hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_panel_upd<T>, dim3(grid8(n), 2), dim3(256), 0, st, S, items, n, kb, right ? 1 : 0, L, L, U,
                       0);
}
template <typename T>
void launch_panel_upd_potrf(const DevSymbol &S, const int32_t *cblks, int npot, const PanelItem *items, int n, int kb,
                            bool right, T *coef, T *winv, T *winvt, double thr, int *stat, hipStream_t st) {
    if (npot + n <= 0) return;
    hipLaunchKernelGGL(k_panel_upd_potrf<T>, dim3(npot + n), dim3(256), 0, st, S, cblks, npot, items, n, kb,
                       right ? 1 : 0, coef, winv, winvt, thr, stat);
}
template <typename T>
void launch_winv_nodes(const DevSymbol &S, const WinvLeaf *leaves, int nleaves, const WinvTile *tiles,
                       const int32_t *round_ptr, int nrounds, const T *coef, T *w, T *wt, T *tbuf, hipStream_t st) {
    if (nleaves > 0) hipLaunchKernelGGL(k_winv_leaves<T>, dim3(nleaves), dim3(256), 0, st, S, leaves, w, wt);
    for (int r = 0; r < nrounds; r++) {
        const int t0 = round_ptr[r], nt = round_ptr[r + 1] - t0;
        if (nt <= 0) continue;
        hipLaunchKernelGGL((k_winv_merge<T, 1>), dim3(nt), dim3(256), 0, st, S, tiles + t0, coef, w, wt, tbuf);
        hipLaunchKernelGGL((k_winv_merge<T, 2>), dim3(nt), dim3(256), 0, st, S, tiles + t0, coef, w, wt, tbuf);
    }
}

void launch_leaf_init(const LeafDev &LP, int32_t *ctr, int32_t *queue, int32_t *sync, hipStream_t st) {
    const int n = std::max(std::max(LP.cblknbr, LP.nregion), 1);
    hipLaunchKernelGGL(k_leaf_init, dim3((n + 255) / 256), dim3(256), 0, st, LP, ctr, queue, sync);
}
template <typename T>
void launch_leaf_tasks(const DevSymbol &S, const LeafDev &LP, const UpdEntry *ents, const int32_t *shift, T *coef,
                       T *winv, T *winvt, double thr, int *stat, int32_t *ctr, int32_t *queue, int32_t *sync,
                       int grid, long long maxwait, hipStream_t st) {
    if (LP.nregion <= 0) return;
    const int g = std::max(1, std::min(grid, LP.nregion));
    hipLaunchKernelGGL(k_leaf_tasks<T>, dim3(g), dim3(256), 0, st, S, LP, ents, shift, coef, winv, winvt, thr, stat,
                       ctr, queue, sync, maxwait);
}

#define INST(T)                                                                                                    \
    template void launch_leaf_tasks<T>(const DevSymbol &, const LeafDev &, const UpdEntry *, const int32_t *, T *, \
                                       T *, T *, double, int *, int32_t *, int32_t *, int32_t *, int, long long,   \
                                       hipStream_t);                                                               \
    template void launch_getrf64<T>(const DevSymbol &, const int32_t *, int, int, T *, T *, T *, T *, T *, double, \
                                    int *, hipStream_t);                                                           \
    template void launch_lu_square_layout<T>(const DevSymbol &, const PanelItem *, int, T *, T *, hipStream_t);      \
    template void launch_lu_square_merge<T>(const DevSymbol &, const PanelItem *, int, T *, T *, hipStream_t);       \
    template void launch_potrf64<T>(const DevSymbol &, const int32_t *, int, int, int, T *, T *, T *, double, int *,    \
                                    hipStream_t);                                                                  \
    template void launch_panel_trsm<T>(const DevSymbol &, const PanelItem *, int, int, T *, const T *, hipStream_t); \
    template void launch_panel_trsm2<T>(const DevSymbol &, const PanelItem *, int, int, T *, const T *, T *,         \
                                        const T *, hipStream_t);                                                 \
    template void launch_panel_upd<T>(const DevSymbol &, const PanelItem *, int, int, bool, T *, const T *,       \
                                      const T *, bool, hipStream_t);                                             \
    template void launch_panel_upd_lu<T>(const DevSymbol &, const PanelItem *, int, int, bool, T *, T *,          \
                                         hipStream_t);                                                           \
    template void launch_panel_upd_potrf<T>(const DevSymbol &, const int32_t *, int, const PanelItem *, int, int,  \
                                            bool, T *, T *, T *, double, int *, hipStream_t);                    \
    template void launch_winv_nodes<T>(const DevSymbol &, const WinvLeaf *, int, const WinvTile *,               \
                                       const int32_t *, int, const T *, T *, T *, T *, hipStream_t);
INST(double)
INST(float)

}  // namespace pxa
