// small_kernels.hpp -- gfx950 kernels of the PCGPME iteration
// (src2LOWNS/pcgpme_para.F90:148-247) for operators of a few hundred to some
// hundred thousand rows.
//
// There a kernel takes 1.5 us of work and as much again to start and to end,
// and an iteration of 14 launches is bound by their number: 54 us at 78
// thousand rows.  So an iteration here is five launches:
//   k_small_spmv<1>  the scalars of the iteration before (k_fin_beta), P = R +
//                    BETA (P - AMU Q) at every row and neighbour, Y = A P
//   k_small_pm       the whole of LDUSUB (all six stages) and its dots
//   k_small_spmv<2>  ALP, E = R - ALP Q, Y = A E
//   k_small_pm
//   k_small_update   AMU, X, R and their dots
// Work is repeated to save launches: every workgroup sums the dot partials
// (some hundred) and computes the scalars itself; P and E are formed from
// their terms at each neighbour; stages 1 to 4 are computed at each point that
// stage 6 reads, from records that hold the neighbours of the neighbours.
//
// What bounds them is the chain of dependent loads: a kernel finds its XCD's L2
// without the other XCDs' results, so a trip costs some 0.7 us; k_small_pm
// makes four (its last stage's record, that of stage 3/4, of stage 1/2, the
// vector), the others two.  An iteration at 78 thousand rows: 54 us in 14
// launches, 29 in five; FP32 60 and 33.
//
// Dot partials are one a wavefront's worth of rows (128 FP64, 256 FP32), which
// the consumer adds up in the order of block_sum and fin_sums.  Values and the
// order of operations are those of the single kernels: results are
// bit-identical.
#pragma once
#include "pcg_kernels.hpp"

namespace clowns {

// Stages s, s + 1 (a pair of slots) of a row: t(i) = (x(i) - c0 x(j0)) - c1 (x(m) -
// cm x(f)), f the slot-s neighbour of m.  Ghosts are row N, whose record is zero.
template <typename T> struct alignas(16) SmallPair {
    T c0, c1, cm;
    int j0, m, f;
};
template <typename T> struct alignas(16) SmallLast {  // stage 5/6
    T c0, c1;
    int j0, j1;
};
template <typename T> struct SmallOp {
    const T *AL, *D;
    const int *LL;
    int lda;
    const SmallPair<T> *p01, *p23;
    const SmallLast<T> *p45;
};
constexpr int SMALL_MAX_G = 2048;  // row blocks

// Records of rows 0 .. N from the preconditioner's columns (C: as stored).
template <typename T, typename C>
__global__ void __launch_bounds__(BS)
k_small_build(int N, int lda, const C *__restrict__ a, const int *__restrict__ LL, SmallPair<T> *__restrict__ p01,
              SmallPair<T> *__restrict__ p23, SmallLast<T> *__restrict__ p45) {
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i > N) return;
    SmallPair<T> p[2];
    SmallLast<T> q = {T(0), T(0), N, N};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        p[s] = {T(0), T(0), T(0), N, N, N};
        if (i == N) continue;
        const size_t k0 = (size_t)(2 * s) * lda, k1 = k0 + lda;
        p[s].c0 = (T)a[k0 + i];
        p[s].c1 = (T)a[k1 + i];
        p[s].j0 = min(LL[k0 + i] - 1, N);
        const int m = min(LL[k1 + i] - 1, N);
        p[s].m = m;
        if (m < N) {
            p[s].cm = (T)a[k0 + m];
            p[s].f = min(LL[k0 + m] - 1, N);
        }
    }
    if (i < N) {
        q.c0 = (T)a[4 * (size_t)lda + i];
        q.c1 = (T)a[5 * (size_t)lda + i];
        q.j0 = min(LL[4 * (size_t)lda + i] - 1, N);
        q.j1 = min(LL[5 * (size_t)lda + i] - 1, N);
    }
    p01[i] = p[0];
    p23[i] = p[1];
    p45[i] = q;
}

// Sums of NA arrays of W G partials (W = 4: a wavefront's each; 1: a row
// block's), in every thread, in the order of block_sum and fin_sums.  BS
// threads; lds: 16 NA doubles.
template <int NA, int W>
__device__ __forceinline__ void small_sums(const double *__restrict__ wp, int G, double *lds, double *out) {
    const int t = threadIdx.x, w = t >> 6;
    const int nv = min((G + 63) >> 6, FIN_BS / 64);  // fin_sums' wavefronts that have partials
    for (int v = w; v < nv; v += BS / 64) {
        const int k = 64 * v + (t & 63);
        double s[NA];
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            s[a] = 0.0;
            for (int kk = k; kk < G; kk += FIN_BS) {
                const double *p = wp + W * ((size_t)a * G + kk);
                if (W == 1) {
                    s[a] += *p;
                    continue;
                }
                const double2 u0 = *reinterpret_cast<const double2 *>(p), u1 = *reinterpret_cast<const double2 *>(p + 2);
                double b = 0.0;
                b += u0.x;
                b += u0.y;
                b += u1.x;
                b += u1.y;
                s[a] += b;
            }
        }
#pragma unroll
        for (int a = 0; a < NA; ++a) {
            s[a] = wave_sum(s[a]);
            if ((t & 63) == 0) lds[16 * a + v] = s[a];
        }
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        out[a] = 0.0;
        for (int v = 0; v < nv; ++v) out[a] += lds[16 * a + v];
    }
}

// The scalars after the iteration whose update left the partials (k_fin_beta),
// to nxt, whose copy the next iteration uses; false: the run has ended.
template <int W, typename T>
__device__ __forceinline__ bool small_beta(const Scal *sc, Scal *nxt, unsigned long long *host, const double *wp,
                                           int G, double *lds, T &beta, T &amu) {
    Scal s = *sc;
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (!s.done) {
        double r[2];
        small_sums<2, W>(wp, G, lds, r);
        beta_step(s, r[0], r[1]);
        if (first) post_word(host, s.K, s.done, s.ERR);
    }
    if (first) *nxt = s;
    beta = (T)s.BETA;
    amu = (T)s.AMU;
    return !s.done;
}
// ALP from the partials of (R^,Q) (k_fin_alpha), to sc.
template <int W, typename T>
__device__ __forceinline__ bool small_alpha(Scal *sc, const double *wp, int G, double *lds, T &alp) {
    if (sc->done) return false;
    const double C1 = sc->C1;
    double rq;
    small_sums<1, W>(wp, G, lds, &rq);
    const double alpha = C1 / rq;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->RQ = rq;
        sc->ALP = alpha;
    }
    alp = (T)alpha;
    return true;
}

// Y = A v.  STEP 0: v = a.  STEP 1: v = a + BETA (b - AMU c).  STEP 2: v =
// a - ALP c.  v at the rows goes to o (STEP 1, 2).  One row a thread.
template <typename T, int STEP, int W>
__global__ void __launch_bounds__(BS)
k_small_spmv(Scal *sc, Scal *nxt, unsigned long long *host, int N, const double *__restrict__ wp, int G,
             SmallOp<T> A, const T *__restrict__ a, const T *__restrict__ b, const T *__restrict__ c,
             T *__restrict__ o, T *__restrict__ y) {
    __shared__ double lds[32];
    const int i = logical_block() * BS + threadIdx.x, ii = min(i, N - 1);
    int j[6];
    T co[7];
#pragma unroll
    for (int k = 0; k < 6; ++k) j[k] = A.LL[(size_t)k * A.lda + ii] - 1;
#pragma unroll
    for (int k = 0; k < 6; ++k) co[k] = A.AL[(size_t)k * A.lda + ii];
    co[6] = A.D[ii];
    T va[7], vb[7], vc[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        const int n = k ? j[k ? k - 1 : 0] : ii;
        va[k] = a[n];
        if (STEP == 1) vb[k] = b[n];
        if (STEP != 0) vc[k] = c[n];
    }
    if (STEP == 0) {
        if (sc->done) return;
    } else if (STEP == 1) {
        T beta, amu;
        if (!small_beta<W>(sc, nxt, host, wp, G, lds, beta, amu)) return;
#pragma unroll
        for (int k = 0; k < 7; ++k) va[k] = va[k] + beta * (vb[k] - amu * vc[k]);
    } else {
        T alp;
        if (!small_alpha<W>(sc, wp, G, lds, alp)) return;
#pragma unroll
        for (int k = 0; k < 7; ++k) va[k] = va[k] - alp * vc[k];
    }
    if (i >= N) return;
    if (STEP != 0) o[i] = va[0];
    T acc = va[0] * co[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) acc = acc + co[k] * (STEP == 0 || j[k] < N ? va[k + 1] : T(0));
    y[i] = acc;
}

// Stages 1 and 2 at row j, 1 to 4 at row j (a ghost's values are zero: its
// record's coefficients are, and its vectors).
template <typename T>
__device__ __forceinline__ T small_12(const SmallPair<T> *__restrict__ p, const T *__restrict__ x, int j) {
    const SmallPair<T> r = p[j];
    const T xj = x[j], xm = x[r.m], x0 = x[r.j0];
    T xf = xj;
    if (r.f != j) xf = x[r.f];
    const T om = xm - r.cm * xf;
    return (xj - r.c0 * x0) - r.c1 * om;
}
template <typename T> __device__ __forceinline__ T small_14(const SmallOp<T> &A, const T *__restrict__ x, int j) {
    const SmallPair<T> r = A.p23[j];
    const T tj = small_12(A.p01, x, j), tm = small_12(A.p01, x, r.m), t0 = small_12(A.p01, x, r.j0);
    T tf = tj;
    if (r.f != j) tf = small_12(A.p01, x, r.f);
    const T om = tm - r.cm * tf;
    return (tj - r.c0 * t0) - r.c1 * om;
}

// out = PM in, with the dots of k_pm_v2 / k_pm_v4 (DOT 1: (w,out); 2: those and
// (out,out)) as wavefront partials, one a workgroup of 64 R
// rows (R rows a thread of those kernels), gridDim.x an array.  One row a
// thread.
template <typename T, int DOT>
__global__ void __launch_bounds__(256)
k_small_pm(const Scal *__restrict__ sc, int N, SmallOp<T> A, const T *__restrict__ in, T *__restrict__ out,
           const T *__restrict__ w, double *__restrict__ wp) {
    constexpr int R = sizeof(T) == 8 ? 2 : 4;
    __shared__ double pr[DOT][64 * R];
    const int done = sc->done;
    const int lb = logical_block(), t = threadIdx.x, i = lb * 64 * R + t;
    double s0 = 0.0, s1 = 0.0;
    if (i < N) {
        const SmallLast<T> q = A.p45[i];
        const T wi = w[i];
        const T t4 = small_14(A, in, i), u0 = small_14(A, in, q.j0), u1 = small_14(A, in, q.j1);
        T r = t4 - q.c0 * u0;
        r = r - q.c1 * u1;
        if (!done) out[i] = r;
        s0 = (double)wi * (double)r;
        s1 = (double)r * (double)r;
    }
    pr[0][t] = s0;
    if (DOT == 2) pr[DOT - 1][t] = s1;
    __syncthreads();
    if (t >= 64 || done) return;
#pragma unroll
    for (int a = 0; a < DOT; ++a) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (i - t + R * t + k < N) s += pr[a][R * t + k];
        s = wave_sum(s);
        if (t == 0) wp[(size_t)a * gridDim.x + lb] = s;
    }
}

// AMU from the partials of (E,V), (V,V) into sc; x += ALP p + AMU e; r = e - AMU
// v; (r,r), (r^,r) as wavefront partials wo (k_update_vec's rows a thread).
template <typename T, int W>
__global__ void __launch_bounds__(BS)
k_small_update(Scal *sc, int N, const double *__restrict__ wp, int Gp, T *__restrict__ x, const T *__restrict__ p,
               const T *__restrict__ e, const T *__restrict__ v, T *__restrict__ r, const T *__restrict__ rh,
               double *__restrict__ wo) {
    using VT = typename VecOf<T>::t;
    constexpr int RV = VecOf<T>::R;
    __shared__ double lds[32];
    const int lb = logical_block();
    const int i = (lb * BS + threadIdx.x) * RV;
    VT xv = {}, pv = {}, ev = {}, vv = {}, hv = {};
    if (i < N) {  // the vectors' zero rows after row N - 1 hold a vector more
        xv = *reinterpret_cast<const VT *>(x + i);
        pv = *reinterpret_cast<const VT *>(p + i);
        ev = *reinterpret_cast<const VT *>(e + i);
        vv = *reinterpret_cast<const VT *>(v + i);
        hv = *reinterpret_cast<const VT *>(rh + i);
    }
    if (sc->done) return;
    const T alp = (T)sc->ALP;
    double s[2];
    small_sums<2, W>(wp, Gp, lds, s);
    const double omega = s[0] / s[1];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->SS = s[1];
        sc->AMU = omega;
    }
    const T amu = (T)omega;
    double rn = 0.0, c1 = 0.0;
    VT xo, ro;
#pragma unroll
    for (int k = 0; k < RV; ++k) {
        T t = ev[k];
        xo[k] = xv[k] + alp * pv[k] + amu * t;
        t = t - amu * vv[k];
        ro[k] = t;
        if (i + k < N) {
            rn += (double)t * (double)t;
            c1 += (double)t * (double)hv[k];
        }
    }
    if (i + RV - 1 < N) {
        *reinterpret_cast<VT *>(x + i) = xo;
        *reinterpret_cast<VT *>(r + i) = ro;
    } else {
        for (int k = 0; k < RV; ++k)
            if (i + k < N) {
                x[i + k] = xo[k];
                r[i + k] = ro[k];
            }
    }
    const double a = wave_sum(rn), b = wave_sum(c1);
    if ((threadIdx.x & 63) == 0) {
        wo[4 * lb + (threadIdx.x >> 6)] = a;
        wo[4 * ((size_t)gridDim.x + lb) + (threadIdx.x >> 6)] = b;
    }
}

} // namespace clowns
