// run_kernels.hpp -- gfx950 kernels of the PCGPME solve for operators whose
// rows come in runs: SpMV (AXSUB, src2LOWNS/pcgpme_para.F90:323-352) and the
// stages of LDUSUB (:279-318).
//
// An assembled pressure operator numbers its rows along grid lines, so over
// long runs of rows the neighbours' offsets from the row repeat, and mostly
// the coefficients too (the row patterns of pcg_kernels.hpp).  The runs are
// cut into tasks of up to 128 rows for one wavefront, two consecutive rows a
// lane.  A task's description (rows, offsets, coefficients) is one small load
// and then lives in scalar registers: no row reads an index, and where the
// coefficients repeat none reads a coefficient.  Rows outside long enough runs
// (at walls and partial cells) stand in a list, one a lane, with their
// neighbours and coefficients packed in list order.
//
// The description also holds the second level of a pair of stages: stage s+1
// of row i needs stage s of its neighbour m,
//   t(m) = in(m) - a_s(m) in(f),  f = m's neighbour in slot s,
// and on a grid f is mostly i itself (m lies across the face that stage s+1
// crosses, and stage s crosses the opposite one).  So a pair of stages is one
// pass with two gathers (k_pm_pair_run) in place of two.  Where the last two
// slots are the adjacent rows, the two-term stage with its dots
// (k_pm_dot_run) takes them from the neighbouring lanes and gathers nothing.
//
// What bounds gathers here is the L1 cache's rate, which counts four lanes an
// access whatever their width, and the chain of dependent memory round trips.
// So a neighbour is loaded as the aligned pair its row pair falls on; where
// the offset is odd the lanes hand the elements on (one DPP move a dword); the
// adjacent rows' values are the neighbouring lanes' own; and a wavefront makes
// two round trips, its descriptions and its gathers, without a barrier.
//
// Work vectors carry RUN_PAD zero rows after row N - 1: lanes past a task's
// end read them or neighbouring rows and store nothing, and a ghost slot reads
// there.
//
// Values and order of operations are those of k_spmv_v2, k_pm_v2, k_pm_v4 and
// k_spmv_rows32: results, dot partials included, are bit-identical.
#pragma once
#include "pcg_kernels.hpp"

namespace clowns {

constexpr int RUN_ROWS = 512;       // rows of a block (k_pm_v2's)
constexpr int RUN_W = 128;          // rows of a task's window
constexpr int RUN_MIN = 16;         // rows a run needs to be tasks; shorter ones go to the list
constexpr int RUN_TASKS = RUN_ROWS / RUN_MIN;  // tasks a block can have
constexpr int RUN_U = 2;            // tasks of a wavefront, both in flight at once
constexpr int RUN_PAD = 256;        // zero rows after row N - 1: a window, its neighbours', an edge
constexpr int RUN_MAX_N = 1 << 28;  // rows up to here: byte offsets of FP64 vectors fit 32 bits
constexpr int RUN_GHOST = 1 << 30;  // offset of a ghost slot while a block is described

// Task descriptions.  a: the window's first row (even), rows [lo, hi) of it
// are the task's.  b: the element a neighbour of row a is (N: ghost); its even
// part is where the pairs are loaded, its lowest bit whether they hand on.
enum : int {
    RF_FAR = 1,     // bf: the partner's slot s leads elsewhere than back to the row
    RF_GHOST = 2,   // the partner is a ghost row (its stage value is 0)
    RF_K4 = 4, RF_K5 = 6  // bits of the classes of slots 4 and 5 (RK_*)
};
template <typename T> struct alignas(16) RunPair {  // stages s, s + 1
    int a, lo, hi, flags, b0, b1, bf, pad_;
    T c0, c1, cm;  // a_s, a_s+1; a_s of the partner
};
template <typename T> struct alignas(16) RunSpmv {
    int a, lo, hi, flags, b[6];
    T c[6], d;
};
constexpr int RK_LEFT = 0, RK_RIGHT = 1, RK_GHOST = 2, RK_OTHER = 3;
// Two-term stage: a byte a row, pattern | class of slot 4 << 4 | class of slot
// 5 << 6; RC_REC: the row has a record (its own coefficients, or a slot that
// leads elsewhere), packed in row order, those of a 128-row quarter q of block
// b rq[4 b + q].y from rq[4 b + q].x on.  Each wavefront of a launch reads its
// first record, their number and its row block (RunWave).
constexpr int RC_REC = 0xf0;

typedef int4 RunWave;

// List entry (SoA): the row, its six neighbours, the slot-0 neighbour of its
// slot-1 neighbour and the slot-2 neighbour of its slot-3 neighbour (0-based,
// N: ghost); coefficients lc[k][entry], k = 0..5 a_k, 6 D, 7 a_0 of the slot-1
// neighbour, 8 a_2 of the slot-3 neighbour.
constexpr int RUN_LC = 9;
// The tasks and the list as the kernels of one precision read them: nt[0]
// tasks of table coefficients, then nt[1] tasks of the rows' own.
template <typename T> struct RunOp {
    const RunPair<T> *pair[2];
    const RunSpmv<T> *spmv;
    const int4 *lj0, *lj1;        // {row, n0, n1, n2}, {n3, n4, n5, 0}
    const int2 *lj2;              // {f of slot 1, f of slot 3}
    const T *sc, *lc;             // list coefficients of the operator and of the preconditioner
    const T *AL, *D;              // the operator's columns (tasks of the rows' own coefficients)
    const uint8_t *cid;           // two-term stage (null: not in this form)
    const RunWave *wave;
    const int2 *rj;               // records: neighbours of slots 4, 5 ...
    const T *rc;                  // ... and a_4, a_5
    const double *ptab;
    int lda, lcap, nl, nt[2];
};

// ------------------------------------------------------------------ build --
struct RunBuild {
    int *nt0, *nt1;               // per block: tasks of table and of own coefficients
    RunPair<double> *pair0, *pair1;  // [block][RUN_TASKS], table tasks from the front, own ones from the back
    RunSpmv<double> *spmv;
    int4 *lj0, *lj1;
    int2 *lj2;
    double *lc;
    uint8_t *cid;                 // null: no two-term form
    int2 *rq;
    int2 *rj;
    double *rc;
    int lcap, rcap;
};

__device__ __forceinline__ int run_class(int off) {
    return off == -1 ? RK_LEFT : (off == 1 ? RK_RIGHT : (off == RUN_GHOST ? RK_GHOST : RK_OTHER));
}

// Runs of a block's rows: heads (bit u of the 512) given, the run of row u.
__device__ __forceinline__ void run_bounds(const unsigned long long *heads, int u, int &rs, int &re) {
    int w = u >> 6;
    unsigned long long b = heads[w] & (~0ull >> (63 - (u & 63)));
    while (b == 0) b = heads[--w];  // row 0 is a head
    rs = 64 * w + 63 - __clzll((long long)b);
    w = u >> 6;
    b = (u & 63) == 63 ? 0ull : heads[w] & (~0ull << ((u & 63) + 1));
    while (b == 0 && ++w < RUN_ROWS / 64) b = heads[w];
    re = b ? 64 * w + __ffsll((unsigned long long)b) - 1 : RUN_ROWS;
}

// One workgroup describes one block.  pid: the rows' pattern ids.  Rows run
// together while the six offsets and the partners' repeat: first the runs of
// one pattern (the row's and its partners'), then, over what is left, those of
// any coefficients.  List entries and records come from an atomic
// allocation (their place depends on the run, their contents do not; past lcap
// and rcap none are written).  cnt: list entries, records << 32: one atomic a
// block (the four counters of a first form, of which atomics on one address
// are some 6 ns each, were its time: 613 us at 6.6M rows, now 224).
__global__ void __launch_bounds__(BS)
k_run_build(int N, int lda, const double *__restrict__ AL, const double *__restrict__ D, const int *__restrict__ LL,
            const uint8_t *__restrict__ pid, RunBuild o, unsigned long long *__restrict__ cnt) {
    const int r0 = blockIdx.x * RUN_ROWS, t = threadIdx.x;
    constexpr int KW = 9;  // six offsets, the partners' two, patterns
    __shared__ int key[KW][RUN_ROWS];
    __shared__ unsigned long long heads[RUN_ROWS / 64], inp[RUN_ROWS / 64];
    __shared__ int pre[RUN_ROWS];
    __shared__ int start[2];
    int off[2][6], fo[2][2], info[2];  // fo: offset of the partner's slot from the row
    bool one[2];                       // is on one pattern with its partners
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int u = t + 256 * h, r = r0 + u;
        one[h] = false;
        info[h] = 255;
#pragma unroll
        for (int k = 0; k < 6; ++k) off[h][k] = RUN_GHOST;
        fo[h][0] = fo[h][1] = 0;
        if (r < N) {
            int l[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) l[k] = LL[(size_t)k * lda + r];
#pragma unroll
            for (int k = 0; k < 6; ++k) off[h][k] = l[k] > N ? RUN_GHOST : l[k] - 1 - r;
            const int p = pid[r];
            info[h] = p;
            one[h] = p < PAT_MAX;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int m = l[2 * s + 1] - 1;
                int q = 255;  // ghost
                if (m < N) {
                    q = pid[m];
                    const int f = LL[(size_t)(2 * s) * lda + m];
                    fo[h][s] = f > N ? RUN_GHOST : f - 1 - r;
                    one[h] = one[h] && q < PAT_MAX;
                }
                info[h] |= q << (8 + 8 * s);
            }
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) key[k][u] = off[h][k];
        key[6][u] = fo[h][0];
        key[7][u] = fo[h][1];
        key[8][u] = one[h] ? info[h] : -1;
    }
    __syncthreads();
    // same offsets as the row before; a run of one pattern starts where that,
    // or the pattern, changes
    bool same[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int u = t + 256 * h;
        same[h] = u > 0 && r0 + u < N;
        if (same[h]) {
#pragma unroll
            for (int k = 0; k < 6; ++k) same[h] = same[h] && key[k][u - 1] == off[h][k];
            same[h] = same[h] && key[6][u - 1] == fo[h][0] && key[7][u - 1] == fo[h][1];
        }
        const unsigned long long b = __ballot(!(same[h] && one[h] && key[8][u ? u - 1 : 0] == info[h]));
        if ((t & 63) == 0) heads[u >> 6] = b;
    }
    __syncthreads();
    int rs[2], re[2];
    bool run[2], own[2] = {false, false};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int u = t + 256 * h;
        run_bounds(heads, u, rs[h], re[h]);
        run[h] = one[h] && re[h] - rs[h] >= RUN_MIN;
        const unsigned long long b = __ballot(run[h]);
        if ((t & 63) == 0) inp[u >> 6] = b;
    }
    __syncthreads();
    // what is left: runs of any coefficients (rows past N are runs of one)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int u = t + 256 * h;
        const bool pin = u > 0 && (inp[(u - 1) >> 6] >> ((u - 1) & 63) & 1);
        const unsigned long long b = __ballot(run[h] || pin || !same[h]);
        if ((t & 63) == 0) heads[u >> 6] = b;
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (run[h]) continue;
        int a, b;
        run_bounds(heads, t + 256 * h, a, b);
        if (b - a >= RUN_MIN) {
            run[h] = own[h] = true;
            rs[h] = a;
            re[h] = b;
        }
    }
    // prefix over the rows: list rows (bits 0-9), records (10-19), table tasks
    // (20-25), own tasks (26-).  A run's windows start at its first row rounded
    // down to an even one.
    bool nw[2], rec[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int u = t + 256 * h;
        const bool in = r0 + u < N;
        const bool list = !run[h] && in;
        const int k4 = run_class(off[h][4]), k5 = run_class(off[h][5]), p = info[h] & 255;
        rec[h] = in && (p >= PAT_MAX || k4 == RK_OTHER || k5 == RK_OTHER);
        if (o.cid) o.cid[(size_t)r0 + u] = (uint8_t)(!in ? RK_GHOST << 4 | RK_GHOST << 6 : (rec[h] ? RC_REC : p | k4 << 4 | k5 << 6));
        nw[h] = run[h] && (u == rs[h] || (u - (rs[h] & ~1)) % RUN_W == 0);
        pre[u] = (int)list | (int)rec[h] << 10 | (int)(nw[h] && !own[h]) << 20 | (int)(nw[h] && own[h]) << 26;
    }
    __syncthreads();
    for (int st = 1; st < RUN_ROWS; st <<= 1) {  // inclusive scan
        int w[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) w[h] = t + 256 * h >= st ? pre[t + 256 * h - st] : 0;
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) pre[t + 256 * h] += w[h];
        __syncthreads();
    }
    const unsigned tot = pre[RUN_ROWS - 1];
    if (t == 0) {
        const int nl = tot & 1023, nr = tot >> 10 & 1023;
        const unsigned long long at = nl | nr ? atomicAdd(cnt, (unsigned long long)nr << 32 | nl) : 0;
        start[0] = (int)(unsigned)at;
        start[1] = (int)(at >> 32);
        o.nt0[blockIdx.x] = tot >> 20 & 63;
        o.nt1[blockIdx.x] = tot >> 26;
    }
    __syncthreads();
    if (o.cid && t < 4) {
        const int before = t ? pre[128 * t - 1] >> 10 & 1023 : 0;
        o.rq[4 * (size_t)blockIdx.x + t] = make_int2(start[1] + before, (pre[128 * t + 127] >> 10 & 1023) - before);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int u = t + 256 * h, r = r0 + u;
        if (r >= N) continue;
        const int ex = u ? pre[u - 1] : 0;
        int n[6];
#pragma unroll
        for (int s = 0; s < 6; ++s) n[s] = off[h][s] == RUN_GHOST ? N : r + off[h][s];
        const int er = start[1] + (ex >> 10 & 1023);
        if (o.cid && rec[h] && er < o.rcap) {
            o.rj[er] = make_int2(n[4], n[5]);
            o.rc[2 * (size_t)er] = AL[4 * (size_t)lda + r];
            o.rc[2 * (size_t)er + 1] = AL[5 * (size_t)lda + r];
        }
        if (run[h]) {
            if (!nw[h]) continue;
            const int k0 = own[h] ? RUN_TASKS - 1 - (ex >> 26) : ex >> 20 & 63;
            const size_t k = (size_t)blockIdx.x * RUN_TASKS + k0;
            const int a = r & ~1, hi = r0 + min(re[h], (u & ~1) + RUN_W);
            double c[6];
#pragma unroll
            for (int s = 0; s < 6; ++s) c[s] = AL[(size_t)s * lda + r];
            int b[6];
#pragma unroll
            for (int s = 0; s < 6; ++s) b[s] = off[h][s] == RUN_GHOST ? N : a + off[h][s];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int mo = off[h][2 * s + 1];
                int fl = 0, bf = a;
                double cm = 0.0;
                if (mo == RUN_GHOST) {
                    fl |= RF_GHOST;
                } else {
                    cm = AL[(size_t)(2 * s) * lda + r + mo];
                    if (fo[h][s] != 0) {
                        fl |= RF_FAR;
                        bf = fo[h][s] == RUN_GHOST ? N : a + fo[h][s];
                    }
                }
                RunPair<double> p = {a, r, hi, fl, b[2 * s], b[2 * s + 1], bf, 0, c[2 * s], c[2 * s + 1], cm};
                (s ? o.pair1 : o.pair0)[k] = p;
            }
            RunSpmv<double> q = {a, r, hi, run_class(off[h][4]) << RF_K4 | run_class(off[h][5]) << RF_K5,
                                 {b[0], b[1], b[2], b[3], b[4], b[5]}, {c[0], c[1], c[2], c[3], c[4], c[5]}, D[r]};
            o.spmv[k] = q;
        } else {
            const int e = start[0] + (ex & 1023);
            if (e >= o.lcap) continue;
            int f[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) f[s] = n[2 * s + 1] >= N || fo[h][s] == RUN_GHOST ? N : r + fo[h][s];
            o.lj0[e] = make_int4(r, n[0], n[1], n[2]);
            o.lj1[e] = make_int4(n[3], n[4], n[5], 0);
            o.lj2[e] = make_int2(f[0], f[1]);
            const size_t c = o.lcap;
#pragma unroll
            for (int s = 0; s < 6; ++s) o.lc[s * c + e] = AL[(size_t)s * lda + r];
            o.lc[6 * c + e] = D[r];
            o.lc[7 * c + e] = n[1] < N ? AL[n[1]] : 0.0;
            o.lc[8 * c + e] = n[3] < N ? AL[2 * (size_t)lda + n[3]] : 0.0;
        }
    }
}

// A coefficient of the preconditioner: through C (half precision, as the FP32
// inner solve's columns hold it).
template <typename C, typename T> __device__ __forceinline__ T run_coef(double v) {
    if constexpr (sizeof(T) == 8)
        return v;
    else
        return (T)(C)(T)v;
}
// Task counts of the blocks in launch order (order null: natural), for the
// scans: out[0..G) table tasks, out[G+1..2G+1) own ones.
__global__ void __launch_bounds__(BS)
k_run_counts(int G, int nblk, const int *__restrict__ order, const int *__restrict__ nt0,
             const int *__restrict__ nt1, int *__restrict__ out) {
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i >= G) return;
    const int rb = order ? order[i] : i;
    out[i] = rb < nblk ? nt0[rb] : 0;
    out[G + 1 + i] = rb < nblk ? nt1[rb] : 0;
}
// Tasks of both kinds from the scanned counts.
__global__ void k_run_totals(int G, const int *__restrict__ pos, int *__restrict__ out) {
    if (threadIdx.x < 2) out[threadIdx.x] = pos[threadIdx.x ? 2 * G + 1 : G];
}
// The wavefronts of k_pm_dot_run (R rows a lane) in launch order.
template <int R>
__global__ void __launch_bounds__(BS)
k_run_waves(int n, int nblk, const int *__restrict__ order, const int2 *__restrict__ rq, RunWave *__restrict__ out) {
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i >= n) return;
    const int lb = order ? order[i >> 2] : i >> 2;
    const int q = (4 * lb + (i & 3)) * (R / 2);  // its 128-row quarters, 4 nblk of them
    int2 a = {0, 0};
    if (q < 4 * nblk) {
        a = rq[q];
        if (R == 4) a.y += rq[q + 1].y;
    }
    out[i] = make_int4(a.x, a.y, lb, 0);
}
// The blocks' tasks packed in launch order, as T: coefficients of the
// preconditioner go through C (half precision, as the FP32 inner solve's
// columns hold them), the operator's do not.  pos: the scanned counts.
template <typename T, typename C>
__global__ void __launch_bounds__(BS)
k_run_pack(int G, int nblk, const int *__restrict__ order, const int *__restrict__ nt0, const int *__restrict__ nt1,
           const int *__restrict__ pos, const RunPair<double> *__restrict__ p0, const RunPair<double> *__restrict__ p1,
           const RunSpmv<double> *__restrict__ sp, RunPair<T> *__restrict__ q0, RunPair<T> *__restrict__ q1,
           RunSpmv<T> *__restrict__ qs) {
    const int i = (blockIdx.x * BS + threadIdx.x) / RUN_TASKS, j = threadIdx.x % RUN_TASKS;
    if (i >= G) return;
    const int rb = order ? order[i] : i;
    if (rb >= nblk) return;
    size_t o;
    if (j < nt0[rb])
        o = (size_t)pos[i] + j;
    else if (RUN_TASKS - 1 - j < nt1[rb])
        o = (size_t)pos[G] + pos[G + 1 + i] + (RUN_TASKS - 1 - j);
    else
        return;
    const size_t k = (size_t)rb * RUN_TASKS + j;
    auto c = [](double v) -> T { return run_coef<C, T>(v); };
    auto pr = [&](const RunPair<double> &a) {
        RunPair<T> r = {a.a, a.lo, a.hi, a.flags, a.b0, a.b1, a.bf, 0, c(a.c0), c(a.c1), c(a.cm)};
        return r;
    };
    q0[o] = pr(p0[k]);
    q1[o] = pr(p1[k]);
    const RunSpmv<double> a = sp[k];
    RunSpmv<T> r;
    r.a = a.a;
    r.lo = a.lo;
    r.hi = a.hi;
    r.flags = a.flags;
    for (int e = 0; e < 6; ++e) {
        r.b[e] = a.b[e];
        r.c[e] = (T)a.c[e];
    }
    r.d = (T)a.d;
    qs[o] = r;
}
// n values of each of W arrays (stride cap).
template <typename C>
__global__ void __launch_bounds__(BS)
k_run_list32(int n, int W, int cap, const double *__restrict__ a, float *__restrict__ b) {
    const int i = blockIdx.x * BS + threadIdx.x;
    if (i >= n) return;
    for (int k = 0; k < W; ++k) b[(size_t)k * cap + i] = (float)(C)(float)a[(size_t)k * cap + i];
}

// ---------------------------------------------------------------- kernels --
// Lane e's value.
__device__ __forceinline__ int run_pull(int v, int e) { return __builtin_amdgcn_ds_bpermute(e << 2, v); }
__device__ __forceinline__ float run_pull(float v, int e) { return __int_as_float(run_pull(__float_as_int(v), e)); }
__device__ __forceinline__ double run_pull(double v, int e) {
    return __hiloint2double(run_pull(__double2hiint(v), e), run_pull(__double2loint(v), e));
}
// Element j >= 0 through a 32-bit byte offset (RUN_MAX_N).
template <typename T> __device__ __forceinline__ T ldx(const T *p, int j) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + (unsigned)j * (unsigned)sizeof(T));
}
template <typename T> using Run2 = T __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int run_readlane(int v, int k) { return __builtin_amdgcn_readlane(v, k); }
__device__ __forceinline__ float run_readlane(float v, int k) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
}
__device__ __forceinline__ double run_readlane(double v, int k) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), k),
                            __builtin_amdgcn_readlane(__double2loint(v), k));
}
// The value of the lane before (after); the first (last) lane of the
// wavefront gets edge.  All lanes active.
template <bool PREV> __device__ __forceinline__ int run_dpp(int v, int edge) {
    return PREV ? __builtin_amdgcn_update_dpp(edge, v, 0x138, 0xf, 0xf, false)   // wave_shr:1
                : __builtin_amdgcn_update_dpp(edge, v, 0x130, 0xf, 0xf, false);  // wave_shl:1
}
template <bool PREV> __device__ __forceinline__ float run_lane(float v, float edge) {
    return __int_as_float(run_dpp<PREV>(__float_as_int(v), __float_as_int(edge)));
}
template <bool PREV> __device__ __forceinline__ double run_lane(double v, double edge) {
    return __hiloint2double(run_dpp<PREV>(__double2hiint(v), __double2hiint(edge)),
                            run_dpp<PREV>(__double2loint(v), __double2loint(edge)));
}

// Descriptions: a wavefront's RUN_U are one load, dword k in lane k, then
// scalar registers.
template <typename D> __device__ __forceinline__ int run_desc(const D *tab, int unit, int n, int l) {
    constexpr int W = sizeof(D) / 4;
    static_assert(RUN_U * W <= 64, "a lane a dword");
    const int *p = reinterpret_cast<const int *>(tab + unit);
    return l < W * min(RUN_U, n - unit) ? p[l] : 0;
}
template <typename T> __device__ __forceinline__ T run_field(int v, int k) {
    if constexpr (sizeof(T) == 8)
        return __hiloint2double(run_readlane(v, k + 1), run_readlane(v, k));
    else if constexpr (std::is_same<T, float>::value)
        return __int_as_float(run_readlane(v, k));
    else
        return run_readlane(v, k);
}

// The aligned pairs of a neighbour (element b of row a's); a lane whose pair
// would start before the vector (half a pair no row needs) reads its start.
template <typename T> __device__ __forceinline__ Run2<T> run_pairs(const T *x, int b, int l) {
    return ldx(reinterpret_cast<const Run2<T> *>(x), max((b >> 1) + l, 0));
}
// The two rows' elements from the loaded pairs: edge is the element after the
// last lane's pair.
template <typename T> __device__ __forceinline__ void run_align(Run2<T> &v, int b, T edge) {
    if (b & 1) {
        const T nx = run_lane<false>((T)v.x, edge);
        v.x = v.y;
        v.y = nx;
    }
}
// The task's rows of a lane's pair into y (by row).
template <bool ST, typename T> __device__ __forceinline__ void run_store(T *y, int a, int lo, int hi, int l, Run2<T> o) {
    const int r = a + 2 * l;
    if (r >= lo && r + 1 < hi) {
        stv<ST>(reinterpret_cast<Run2<T> *>(y + r), o);
    } else {
        if (r >= lo && r < hi) y[r] = o.x;
        if (r + 1 >= lo && r + 1 < hi) y[r + 1] = o.y;
    }
}

// A pair of stages of one task: loads, then value and store.  OWN: the rows'
// own coefficients, the columns' through C.
template <typename T> struct RunV {
    Run2<T> xi, g0, g1, gf;
    T ed;  // lanes 0, 1, 2: the elements after the pairs of b0, b1, bf
};
template <typename T>
__device__ __forceinline__ void run_pair_load(int v, int o, const T *__restrict__ in, int l, RunV<T> &w) {
    const int a = run_readlane(v, o), hi = run_readlane(v, o + 2), fl = run_readlane(v, o + 3);
    const int b0 = run_readlane(v, o + 4), b1 = run_readlane(v, o + 5), bf = run_readlane(v, o + 6);
    w.xi = w.g0 = w.g1 = T(0);
    w.ed = T(0);
    if (a + 2 * l <= hi) {  // a lane more than the rows: the last one's odd neighbours
        w.xi = run_pairs(in, a, l);
        w.g0 = run_pairs(in, b0, l);
        w.g1 = run_pairs(in, b1, l);
    }
    if (l < 3) w.ed = ldx(in, ((l == 0 ? b0 : (l == 1 ? b1 : bf)) & ~1) + RUN_W);
    w.gf = w.xi;
    if (fl & RF_FAR) w.gf = run_pairs(in, bf, l);
}
template <bool OWN, typename C, bool ST, typename T>
__device__ __forceinline__ void run_pair_finish(int v, int o, RunV<T> &w, T *__restrict__ out,
                                                const T *__restrict__ c, int lda, int l) {
    const int a = run_readlane(v, o), lo = run_readlane(v, o + 1), hi = run_readlane(v, o + 2);
    const int fl = run_readlane(v, o + 3), b0 = run_readlane(v, o + 4), b1 = run_readlane(v, o + 5);
    Run2<T> c0, c1, cm;
    if (OWN) {
        c0 = run_pairs(c, a, l);
        c1 = run_pairs(c + lda, a, l);
        cm = run_pairs(c, b1, l);
        run_align(cm, b1, ldx(c, (b1 & ~1) + RUN_W));
        if constexpr (!std::is_same<C, T>::value) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                c0[h] = (T)(C)c0[h];
                c1[h] = (T)(C)c1[h];
                cm[h] = (T)(C)cm[h];
            }
        }
    } else {
        constexpr int W = sizeof(T) / 4;
        c0 = run_field<T>(v, o + 8);
        c1 = run_field<T>(v, o + 8 + W);
        cm = run_field<T>(v, o + 8 + 2 * W);
    }
    run_align(w.g0, b0, run_readlane(w.ed, 0));
    run_align(w.g1, b1, run_readlane(w.ed, 1));
    if (fl & RF_FAR) run_align(w.gf, run_readlane(v, o + 6), run_readlane(w.ed, 2));
    Run2<T> r;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const T om = fl & RF_GHOST ? T(0) : w.g1[h] - cm[h] * w.gf[h];
        r[h] = (w.xi[h] - c0[h] * w.g0[h]) - c1[h] * om;
    }
    run_store<ST>(out, a, lo, hi, l, r);
}

// The workgroups of a launch: nw[1] of own tasks, then the list's, then nw[0]
// of table tasks (XCD-contiguous, a multiple of 8), 4 RUN_U tasks or 256
// entries each.
struct RunGrid {
    int own, list, tab;
};
// At 12.2M rows (wavy bed): FP64 37.5 us, 5.2 TB/s of the vectors read and
// written (k_pm2_v2: 93; two single stages: 79); FP32 26 (65; 51).  At 13.1M rows
// of a bathymetry 61 and 40 us: by the counters 23.0 and 12.9 bytes a row (16 and
// 8 of them the vectors'), 4.9 and 4.2 TB/s, and 11 million L1 accesses where
// k_pm2_v2 makes 33.
template <typename T, int S, bool ST, typename C>
__global__ void __launch_bounds__(BS)
k_pm_pair_run(const Scal *__restrict__ sc, int N, const T *__restrict__ in, T *__restrict__ out, RunOp<T> d,
              RunGrid g) {
    const int done = sc->done;
    const int t = threadIdx.x, q = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63;
    constexpr int W = sizeof(RunPair<T>) / 4;
    int b = blockIdx.x - g.own - g.list;
    if (b >= 0) {
        b = (b & 7) * (g.tab >> 3) + (b >> 3);
        const int u = (4 * b + q) * RUN_U;
        if (u >= d.nt[0]) return;
        const int v = run_desc(d.pair[S], u, d.nt[0], l);
        if (done) return;
        RunV<T> w[RUN_U];
#pragma unroll
        for (int k = 0; k < RUN_U; ++k) run_pair_load(v, k * W, in, l, w[k]);
#pragma unroll
        for (int k = 0; k < RUN_U; ++k) run_pair_finish<false, C, ST>(v, k * W, w[k], out, (const T *)nullptr, 0, l);
    } else if (b < -g.list) {
        const int u = (4 * blockIdx.x + q) * RUN_U;
        if (u >= d.nt[1]) return;
        const int v = run_desc(d.pair[S] + d.nt[0], u, d.nt[1], l);
        if (done) return;
        for (int k = 0; k < RUN_U; ++k) {
            RunV<T> w;
            run_pair_load(v, k * W, in, l, w);
            run_pair_finish<true, C, ST>(v, k * W, w, out, d.AL + (size_t)(2 * S) * d.lda, d.lda, l);
        }
    } else {
        const int i = (blockIdx.x - g.own) * BS + t;
        if (i >= d.nl) return;
        const int4 a = d.lj0[i];
        const int2 ff = d.lj2[i];
        const T *co = d.lc + i;
        const size_t cap = d.lcap;
        const T c0 = co[2 * S * cap], c1 = co[(2 * S + 1) * cap], cm = co[(7 + S) * cap];
        const int n0 = S ? a.w : a.y, m = S ? d.lj1[i].x : a.z, f = S ? ff.y : ff.x;
        if (done) return;
        const T x = ldx(in, a.x);
        const T om = m < N ? ldx(in, m) - cm * (f == a.x ? x : ldx(in, f)) : T(0);
        out[a.x] = (x - c0 * ldx(in, n0)) - c1 * om;
    }
}

// The SpMV of one task.  Lanes 0 .. 5 of ed: the elements after the pairs of
// b[0..5]; lanes 6, 7: the rows before and after the window.
template <typename T> struct RunVS {
    Run2<T> xi, g[4], g4, g5;
    T ed;
};
template <typename T>
__device__ __forceinline__ void run_spmv_load(int v, int o, const T *__restrict__ x, int l, RunVS<T> &w) {
    const int a = run_readlane(v, o), hi = run_readlane(v, o + 2), fl = run_readlane(v, o + 3);
    int b[6];
#pragma unroll
    for (int e = 0; e < 6; ++e) b[e] = run_readlane(v, o + 4 + e);
    w.xi = T(0);
#pragma unroll
    for (int e = 0; e < 4; ++e) w.g[e] = T(0);
    w.ed = T(0);
    w.g4 = w.g5 = T(0);
    if (a + 2 * l <= hi) {
        w.xi = run_pairs(x, a, l);
#pragma unroll
        for (int e = 0; e < 4; ++e) w.g[e] = run_pairs(x, b[e], l);
    }
    if (l < 8) {
        int i = l == 6 ? max(a - 1, 0) : a + RUN_W;
#pragma unroll
        for (int e = 0; e < 6; ++e) i = l == e ? (b[e] & ~1) + RUN_W : i;
        w.ed = ldx(x, i);
    }
    if ((fl >> RF_K4 & 3) == RK_OTHER) w.g4 = run_pairs(x, b[4], l);
    if ((fl >> RF_K5 & 3) == RK_OTHER) w.g5 = run_pairs(x, b[5], l);
}
template <bool OWN, int MODE, typename T>
__device__ __forceinline__ void run_spmv_finish(int v, int o, RunVS<T> &w, const T *__restrict__ v1,
                                                T *__restrict__ y, const RunOp<T> &d, int l) {
    const int a = run_readlane(v, o), lo = run_readlane(v, o + 1), hi = run_readlane(v, o + 2);
    const int fl = run_readlane(v, o + 3), k4 = fl >> RF_K4 & 3, k5 = fl >> RF_K5 & 3;
    const T prev = run_lane<true>((T)w.xi.y, run_readlane(w.ed, 6));
    const T next = run_lane<false>((T)w.xi.x, run_readlane(w.ed, 7));
#pragma unroll
    for (int e = 0; e < 4; ++e) run_align(w.g[e], run_readlane(v, o + 4 + e), run_readlane(w.ed, e));
    if (k4 == RK_OTHER) run_align(w.g4, run_readlane(v, o + 8), run_readlane(w.ed, 4));
    if (k5 == RK_OTHER) run_align(w.g5, run_readlane(v, o + 9), run_readlane(w.ed, 5));
    const Run2<T> gl = {prev, w.xi.x}, gr = {w.xi.y, next};
    if (k4 == RK_LEFT) w.g4 = gl;
    if (k4 == RK_RIGHT) w.g4 = gr;
    if (k5 == RK_LEFT) w.g5 = gl;
    if (k5 == RK_RIGHT) w.g5 = gr;
    constexpr int W = sizeof(T) / 4, C0 = 10;
    auto co = [&](int e) -> Run2<T> {
        if (OWN) return run_pairs(e < 6 ? d.AL + (size_t)e * d.lda : d.D, a, l);
        return (Run2<T>)run_field<T>(v, o + C0 + e * W);
    };
    Run2<T> acc = w.xi * co(6);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = acc + co(e) * w.g[e];
    acc = acc + co(4) * w.g4;
    acc = acc + co(5) * w.g5;
    if (MODE == 3) acc = run_pairs(v1, a, l) - acc;
    run_store<false>(y, a, lo, hi, l, acc);
}

// y = A x (MODE 0) or y = v1 - A x (MODE 3), NL = 6.  At 12.2M rows (wavy bed):
// FP64 55 us, 3.5 TB/s of x and y (k_spmv_v2: 78); FP32 32 (k_spmv_rows32: 46).
// At 13.1M rows of a bathymetry 88 and 53 (105 and 76): its listed rows, 3% of
// all, each fetch six cache lines of their own; 28.9 and 18.3 bytes a row by the
// counters, 4.3 and 4.5 TB/s, and 17.6 million L1 accesses (k_spmv_v2: 33.5).
template <typename T, int MODE>
__global__ void __launch_bounds__(BS)
k_spmv_run(const Scal *__restrict__ sc, int N, const T *__restrict__ x, const T *__restrict__ v1, T *__restrict__ y,
           RunOp<T> d, RunGrid g) {
    const int done = sc->done;
    const int t = threadIdx.x, q = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63;
    constexpr int W = sizeof(RunSpmv<T>) / 4;
    int b = blockIdx.x - g.own - g.list;
    if (b >= 0) {
        b = (b & 7) * (g.tab >> 3) + (b >> 3);
        const int u = (4 * b + q) * RUN_U;
        if (u >= d.nt[0]) return;
        const int v = run_desc(d.spmv, u, d.nt[0], l);
        if (done) return;
        RunVS<T> w[RUN_U];
#pragma unroll
        for (int k = 0; k < RUN_U; ++k) run_spmv_load(v, k * W, x, l, w[k]);
#pragma unroll
        for (int k = 0; k < RUN_U; ++k) run_spmv_finish<false, MODE>(v, k * W, w[k], v1, y, d, l);
    } else if (b < -g.list) {
        const int u = (4 * blockIdx.x + q) * RUN_U;
        if (u >= d.nt[1]) return;
        const int v = run_desc(d.spmv + d.nt[0], u, d.nt[1], l);
        if (done) return;
        for (int k = 0; k < RUN_U; ++k) {
            RunVS<T> w;
            run_spmv_load(v, k * W, x, l, w);
            run_spmv_finish<true, MODE>(v, k * W, w, v1, y, d, l);
        }
    } else {
        const int i = (blockIdx.x - g.own) * BS + t;
        if (i >= d.nl) return;
        const int4 a = d.lj0[i], c = d.lj1[i];
        T co[7];
#pragma unroll
        for (int k = 0; k < 7; ++k) co[k] = d.sc[(size_t)k * d.lcap + i];
        if (done) return;
        const int n[6] = {a.y, a.z, a.w, c.x, c.y, c.z};
        T acc = ldx(x, a.x) * co[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) acc = acc + co[k] * ldx(x, n[k]);
        y[a.x] = MODE == 3 ? v1[a.x] - acc : acc;
    }
}

// The two-term stage 5/6 with k_pm_v2's (FP64: two rows a lane) or k_pm_v4's
// (FP32: four) dots, for operators whose last two slots are mostly the
// adjacent rows: those come from the lanes beside, coefficients from the
// pattern table, whose row p lane p holds; rows with a record take theirs by
// rank from the lane that loaded it, while the ids are still on their way (a
// load by rank after them was a dependent trip more: 74.6 against 70.4 us).
// FP64: block order as k_pm_v2's; FP32: natural.  What bounds it is HBM: 26.8
// bytes a row by the counters (14.1 FP32), 5.1 TB/s at 13.1M rows (69 us; k_pm_p2
// 76; FP32 44.5, 4.1 TB/s; k_pm_v4 46).
template <typename T, int DOT, bool ST, typename C>
__global__ void __launch_bounds__(BS)
k_pm_dot_run(const Scal *__restrict__ sc, int N, const T *__restrict__ in, T *__restrict__ out,
             const T *__restrict__ w, double *__restrict__ part, RunOp<T> d) {
    constexpr int R = sizeof(T) == 8 ? 2 : 4;
    typedef T vR __attribute__((ext_vector_type(R)));
    typedef typename std::conditional<R == 2, uint16_t, uint32_t>::type Ids;
    const int done = sc->done;
    const int t = threadIdx.x, l = t & 63;
    const RunWave rq = d.wave[4 * logical_block() + __builtin_amdgcn_readfirstlane(t >> 6)];
    const int lb = rq.z;
    const int i = (lb * BS + t) * R;
    const int i0 = __builtin_amdgcn_readfirstlane(i);
    double s0 = 0.0, s1 = 0.0;
    if (i0 < N) {
        // the wavefront's rows; lane p's table row p; lane e's record e
        vR x = {}, wv = {};
        Ids id = 0;
        T edge = T(0);
        if (i < N) {
            x = *reinterpret_cast<const vR *>(in + i);
            id = ldv<ST>(reinterpret_cast<const Ids *>(d.cid + i));
            if (DOT == 1 || DOT == 2) wv = ldv<ST>(reinterpret_cast<const vR *>(w + i));
            if ((l == 0 && i > 0) || l == 63) edge = in[l == 0 ? i - 1 : i + R];
        }
        const double *row = d.ptab + (l & (PAT_MAX - 1)) * PAT_W;
        const double p4 = row[4], p5 = row[5];
        int2 rj = {0, 0};
        Run2<T> rc = {0, 0};
        if (l < rq.y) {
            rj = d.rj[rq.x + l];
            rc = reinterpret_cast<const Run2<T> *>(d.rc)[rq.x + l];
        }
        if (done) return;
        const T t4 = run_coef<C, T>(p4), t5 = run_coef<C, T>(p5);
        const T prev = run_lane<true>((T)x[R - 1], edge), next = run_lane<false>((T)x[0], edge);
        T c4[R], c5[R], v4[R], v5[R];
        int k4[R], k5[R], before = 0;
        bool has[R];
        const unsigned long long below = (1ull << l) - 1;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int e = (int)(id >> (8 * k)) & 255;
            const T lv = k ? x[k ? k - 1 : 0] : prev, rv = k < R - 1 ? x[k < R - 1 ? k + 1 : 0] : next;
            has[k] = e == RC_REC && i + k < N;
            k4[k] = e >> 4 & 3;
            k5[k] = e >> 6;
            c4[k] = run_pull(t4, e & 15);
            c5[k] = run_pull(t5, e & 15);
            v4[k] = k4[k] == RK_LEFT ? lv : (k4[k] == RK_RIGHT ? rv : T(0));
            v5[k] = k5[k] == RK_LEFT ? lv : (k5[k] == RK_RIGHT ? rv : T(0));
            before += __popcll(__ballot(has[k]) & below);
        }
        if (rq.y) {
            int e = before;
#pragma unroll
            for (int k = 0; k < R; ++k) {
                int2 j = {run_pull(rj.x, e), run_pull(rj.y, e)};
                T a4 = run_pull((T)rc.x, e), a5 = run_pull((T)rc.y, e);
                if (has[k]) {
                    if (e >= 64) {
                        j = d.rj[rq.x + e];
                        a4 = d.rc[2 * (size_t)(rq.x + e)];
                        a5 = d.rc[2 * (size_t)(rq.x + e) + 1];
                    }
                    ++e;
                    const T lv = k ? x[k ? k - 1 : 0] : prev, rv = k < R - 1 ? x[k < R - 1 ? k + 1 : 0] : next;
                    const int d4 = j.x - (i + k), d5 = j.y - (i + k);
                    c4[k] = a4;
                    c5[k] = a5;
                    v4[k] = d4 == -1 ? lv : rv;
                    v5[k] = d5 == -1 ? lv : rv;
                    if (d4 != -1 && d4 != 1) v4[k] = ldx(in, j.x);
                    if (d5 != -1 && d5 != 1) v5[k] = ldx(in, j.y);
                }
            }
        }
        vR o;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            T r = x[k] - c4[k] * v4[k];
            r = r - c5[k] * v5[k];
            o[k] = r;
            if (i + k < N) {
                if (DOT == 1 || DOT == 2) s0 += (double)wv[k] * (double)r;
                if (DOT == 2) s1 += (double)r * (double)r;
                if (DOT == 3) s0 += (double)r * (double)r;
            }
        }
        if (i + R - 1 < N) {
            stv<ST>(reinterpret_cast<vR *>(out + i), o);
        } else {
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (i + k < N) out[i + k] = o[k];
        }
    }
    if (done) return;
    if (DOT != 0) {
        __shared__ double lds[BS / 64];
        const double u0 = block_sum<BS>(s0, lds);
        if (DOT == 2) {
            const double u1 = block_sum<BS>(s1, lds);
            if (t == 0) part[gridDim.x + lb] = u1;
        }
        if (t == 0) part[lb] = u0;
    }
}

} // namespace clowns
