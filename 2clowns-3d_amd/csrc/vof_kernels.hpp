// vof_kernels.hpp -- gfx950 kernels of the VOF update cal_vof
// (src2LOWNS/1sub-vof.F90:10-38) on the box layout, without its closing
// set_nflag (that is the classification in classify_kernels.hpp):
//
//   k_vof_flux       cal_quvwf + QFF (1sub-vof.F90:40-116) with the surface
//                    stage fused: quvwf_kaidan (:157-183) or the caller's
//                    PLIC face fluxes in place of quvwf_normal (:119-154)
//   k_vof_mod_eval   quvwf_modify (:186-213): one round of the serial walk
//   k_vof_mod_apply  quvwf_modify's flux corrections, in the serial order
//   k_vof_newf       cal_new_f (:215-269), one pass of its dt retry loop
//   k_vof_slide      simple_slide(0) + cal_fslide_m0 (:302-414), one thread
//                    per (i, j) column walking k downwards
//
// Layout: box index c = i + X*(j + Y*k); un, a, qf are [3][ncell] and hold
// the low face of c in each direction; dx is [3][stride].  A solid cell
// (nf = -1) is the reference's numbering sentinel mn = 0: read as a
// neighbour it gives a = 0 and a face flux of 0.
//
// quvwf_modify walks the surface list in order (ascending c, the k, j, i
// scan of set_nflag) and a correction changes the flux that later cells
// read.  A correction by cell r lands on a face of r; the only later cell
// that reads that face is t = r + e_l, when r points along -e_l (nfb =
// -(l+1)).  So a surface cell's evaluation depends only on its at most
// three "predecessors" r = c - e_l with nfb(r) = -(l+1) that are surface
// cells: rounds evaluate every cell whose predecessors are decided (most
// cells in the first round), and the corrections are applied afterwards per
// face, predecessor first -- the serial result, bit for bit.
//
// No fused multiply-add (-ffp-contract=off): every expression rounds as the
// reference's does.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace clowns {

constexpr double VOF_TINY = 1e-15;          // TINY, 0mod-variables.F90:39
constexpr double VOF_FLIM = 1.0 + 1e-5;     // F_lim, 0mod-variables.F90:40
constexpr double VOF_DTLIM = 1e-6;          // DT_lim, 0mod-variables.F90:41

struct VofDev {
    int nx, ny, nz, stride;
    long ncell;
    const int8_t *nf, *nb;
    const double *F, *Fp, *fb, *a, *un, *dx;
    double *qf, *Fn;
    double *D;  // df_vof of every open cell after quvwf_modify (k_vof_newf -> k_vof_slide)
};

// Launches of k_vof_flux / k_vof_newf / k_vof_slide have a multiple of 8
// blocks; the hardware deals blocks to the 8 XCDs round robin, so block b
// takes the logical index (b mod 8) * G/8 + b/8: each XCD streams one
// contiguous range, and the +-y neighbours (one block away) sit in its own L2.
__device__ __forceinline__ int vof_block() {
    const int b = blockIdx.x;
    return (b & 7) * (gridDim.x >> 3) + (b >> 3);
}

// counters: [0] retry (cal_new_f's icon = 30), [1] stop (F > F_lim on a
// surface cell), [2] correction aimed at a solid cell, [3] pending cells of
// the last modify round, [4] corrected cells, [6] invalid flags, [8..] pending
// cells of the first rounds, [16..] slid cells, in VC_SLOTS counters 64 bytes
// apart (two to a cache line): atomics on one address take their turns, some 50
// ns each, which cost k_vof_slide 8 us (a wavefront's count each)
enum { VC_RETRY = 0, VC_STOP = 1, VC_SOLID = 2, VC_PENDING = 3, VC_MODIFIED = 4, VC_BAD = 6, VC_ROUND = 8,
       VC_SLID = 16, VC_SLOTS = 64, VC_LINE = 16, VC_N = VC_SLID + VC_SLOTS * VC_LINE };
constexpr int VOF_ROUNDS = 2;  // modify rounds queued before the host looks

// The kernels of an update are queued together; each goes ahead only if what
// came before it did not end the update: valid flags, then (from the
// corrections on) no pending cell, then (simple_slide) no retry and no stop.
__device__ __forceinline__ bool vof_valid(const int *cnt) { return cnt[VC_BAD] == 0; }
__device__ __forceinline__ bool vof_settled(const int *cnt) { return (cnt[VC_BAD] | cnt[VC_PENDING]) == 0; }

// Box index of a cell (they fit 32 bits: every field of a larger box would
// outgrow the memory), in 32-bit divisions.
__device__ __forceinline__ void vof_pos(const VofDev &v, long c, int p[3]) {
    const unsigned X = v.nx + 2, Y = v.ny + 2, u = (unsigned)c, r = u / X;
    p[0] = (int)(u - r * X);
    p[2] = (int)(r / Y);
    p[1] = (int)(r - (unsigned)p[2] * Y);
}

// df_vof(nn) = fp - dt*renzoku_fv(...) (1sub-vof.F90:271-300,
// lib/src/math_func.F90:51-54); the low faces of c may carry a pending
// correction of a predecessor (sub[l], applied as qf - sub).  The loads do not
// wait for the flags: a solid neighbour's values are loaded and not used.
struct VofCell {
    double q[3], a[3], qh[3], ah[3], Fp, fb;
    bool solid[3];  // the high neighbours
};
__device__ __forceinline__ void vof_load(const VofDev &v, long c, VofCell &w) {
    const long st[3] = {1, (long)(v.nx + 2), (long)(v.nx + 2) * (v.ny + 2)};
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        const long h = min(c + st[l], v.ncell - 1);  // a ring cell's may lie past the box
        const size_t oc = (size_t)l * v.ncell + c, oh = (size_t)l * v.ncell + h;
        w.solid[l] = v.nf[h] == -1;
        w.q[l] = v.qf[oc];
        w.a[l] = v.a[oc];
        w.qh[l] = v.qf[oh];
        w.ah[l] = v.a[oh];
    }
    w.Fp = v.Fp[c];
    w.fb = v.fb[c];
}
__device__ __forceinline__ double vof_df(const VofDev &v, const VofCell &w, const int p[3], double dt) {
    double qp[3], ap[3];
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        qp[l] = w.solid[l] ? 0.0 : w.qh[l];
        ap[l] = w.solid[l] ? 0.0 : w.ah[l];
    }
    const double r = ((qp[0] * ap[0] - w.q[0] * w.a[0]) / v.dx[p[0]] +
                      (qp[1] * ap[1] - w.q[1] * w.a[1]) / v.dx[(size_t)v.stride + p[1]] +
                      (qp[2] * ap[2] - w.q[2] * w.a[2]) / v.dx[2 * (size_t)v.stride + p[2]]) / w.fb;
    return w.Fp - dt * r;
}
__device__ __forceinline__ double vof_df(const VofDev &v, long c, const int p[3], double dt, const double sub[3],
                                         const bool has_sub[3]) {
    VofCell w;
    vof_load(v, c, w);
#pragma unroll
    for (int l = 0; l < 3; ++l)
        if (has_sub[l]) w.q[l] = w.q[l] - sub[l];
    return vof_df(v, w, p, dt);
}
__device__ __forceinline__ double vof_df(const VofDev &v, long c, const int p[3], double dt) {
    VofCell w;
    vof_load(v, c, w);
    return vof_df(v, w, p, dt);
}

__device__ inline double vof_sign(double a, double b) { return signbit(b) ? -fabs(a) : fabs(a); }

// MODE 0: caller's PLIC face fluxes where qmask != 0 (qs/qmask may be null);
// MODE 1: quvwf_kaidan.  Every load but those of surface donors and partly
// open faces is issued before the first is used (each waited for the flags
// it depends on before: 84 us at 4.4M cells, now 58; the fields alone
// take 51 at a large copy's rate).
template <int MODE>
__global__ void __launch_bounds__(256)
k_vof_flux(VofDev v, double dt, const double *__restrict__ qs, const int8_t *__restrict__ qmask,
           const int *__restrict__ cnt) {
    const long c = (long)vof_block() * blockDim.x + threadIdx.x;
    if (c >= v.ncell) return;
    const long st[3] = {1, (long)(v.nx + 2), (long)(v.nx + 2) * (v.ny + 2)};
    const size_t n = (size_t)v.ncell;
    const int fc = v.nf[c], bc = v.nb[c];
    const double Fc = v.F[c];
    int fm[3], bm[3];
    double Fm[3], ul[3], al[3];
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        const long m = max(c - st[l], 0l);  // a ring cell's may lie before the box
        fm[l] = v.nf[m];
        bm[l] = v.nb[m];
        Fm[l] = v.F[m];
        ul[l] = v.un[l * n + c];
        al[l] = MODE == 1 && l < 2 ? v.a[l * n + c] : 0.0;
    }
    if (!vof_valid(cnt)) return;
    if (fc == -1) {
#pragma unroll
        for (int l = 0; l < 3; ++l) v.qf[l * n + c] = 0.0;
        return;
    }
    int p[3];
    vof_pos(v, c, p);
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        const size_t o = l * n + c;
        const double u = ul[l];
        const long m = c - st[l];
        // QFF: the donor is the upwind cell (c - e_l for u > 0, c for u < 0)
        const bool neg = signbit(u);
        double q = 0.0;
        if (u != 0.0 && fm[l] != -1) {
            const int fd = neg ? fc : fm[l], bd = neg ? bc : bm[l];
            const double Fd = neg ? Fc : Fm[l];
            if (fd == 2 && (bd < 0 ? -bd : bd) == l + 1) {
                const double dxx = v.dx[(size_t)l * v.stride + (neg ? p[l] : p[l] - 1)];
                if ((double)bd * u < 0.0) {
                    const double t = fabs(u) - (1.0 - Fd) * dxx / dt;
                    q = vof_sign(1.0, u) * (t > 0.0 ? t : 0.0);
                } else {
                    const double t = Fd * dxx / dt, au = fabs(u);
                    q = vof_sign(1.0, u) * (au < t ? au : t);
                }
            } else {
                q = u * Fd;
            }
        }
        if (MODE == 1) {
            if (l < 2) {
                const double av = al[l];
                if (av > 0.0 && av < 1.0) {
                    if (u < 0.0 && fc == 2 && av != v.fb[c]) {
                        const double t = av - v.fb[c] + Fc * v.fb[c];
                        q = u * (t > 0.0 ? t : 0.0) / av;
                    } else if (u > 0.0 && fm[l] == 2 && av != v.fb[m]) {
                        const double t = av - v.fb[m] + Fm[l] * v.fb[m];
                        q = u * (t > 0.0 ? t : 0.0) / av;
                    }
                }
            }
        } else {
            if (qmask && qmask[o]) q = qs[o];
        }
        v.qf[o] = q;
    }
}

// quvwf_normal (1sub-vof.F90:119-154) on the listed surface cells, with
// cal_idou2's flux (1sub-normal.F90:29-99) from the caller's PLIC segment
// volumes vol[6 m + 2 l + ll] (face l, ll = 0 low / 1 high of cells[m]):
// on each face the cell drains through (un (1 - 2 ll) < 0, a != 0),
// qf = sign(u) V / area / dt / a, 0 for |u| dt < SMALL or V = 0.  Runs after
// k_vof_flux<0>.  Two listed cells never write one face: the shared face's
// velocity drains only one of them.
__global__ void __launch_bounds__(256)
k_vof_plic(VofDev v, double dt, int n, const int *__restrict__ cells, const double *__restrict__ vol,
           const int *__restrict__ cnt) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n || !vof_valid(cnt)) return;
    const long c = cells[m];
    const long st[3] = {1, (long)(v.nx + 2), (long)(v.nx + 2) * (v.ny + 2)};
    int p[3];
    vof_pos(v, c, p);
    const size_t S = (size_t)v.stride, nc = (size_t)v.ncell;
    const double dxx = v.dx[p[0]], dyy = v.dx[S + p[1]], dzz = v.dx[2 * S + p[2]];
    for (int l = 0; l < 3; ++l)
        for (int ll = 0; ll < 2; ++ll) {
            const long nn = c + ll * st[l];
            const bool solid = v.nf[nn] == -1;
            const double u = solid ? 0.0 : v.un[l * nc + nn];
            const double a = solid ? 0.0 : v.a[l * nc + nn];
            const double lsn = 1.0 - 2.0 * ll;
            if (u * lsn >= 0.0 || a == 0.0) continue;
            double idou = 0.0;
            if (!(fabs(u) * dt < 1e-9)) {  // SMALL, 0mod-variables.F90:39
                const double area = l == 2 ? dxx * dyy : (l == 1 ? dxx * dzz : dzz * dyy);
                const double vs = vol[6 * (size_t)m + 2 * l + ll];
                idou = vs == 0.0 ? 0.0 : vof_sign(1.0, u) * vs / area / dt;
            }
            v.qf[l * nc + nn] = idou / a;
        }
}

// Each listed PLIC cell must be a flow cell (interior: its neighbour reads
// stay in the box, the ring being solid).
__global__ void __launch_bounds__(256)
k_vof_check_plic(VofDev v, int n, const int *__restrict__ cells, int *__restrict__ cnt) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    const long c = cells[m];
    if (c < 0 || c >= v.ncell || v.nf[c] == -1) atomicOr(&cnt[VC_BAD], 1);
}

// The flags every other kernel relies on for its neighbour reads: the box
// ring is solid (nf = -1), nf is -1..2, and a surface cell has 1 <= |nb| <= 3.
// Lists the surface cells, a segment of the list a workgroup, and sets them
// pending.  Sixteen cells
// a thread, one load a field where they are aligned (one cell a thread, and a
// pass that cleared the state of every cell: 14 + 7 us at 4.4M cells; now
// 13).
constexpr int VOF_CELLS = 16, VOF_SEG = 64 * VOF_CELLS;  // cells a thread and a list segment
__global__ void __launch_bounds__(64)
k_vof_check(VofDev v, int *__restrict__ cnt, int *__restrict__ state, unsigned *__restrict__ list,
            int *__restrict__ nlist) {
    const long c0 = VOF_CELLS * ((long)blockIdx.x * blockDim.x + threadIdx.x);
    int8_t f[VOF_CELLS], b[VOF_CELLS];
    if (c0 + VOF_CELLS <= v.ncell && (((uintptr_t)v.nf | (uintptr_t)v.nb) & 15) == 0) {
        *reinterpret_cast<uint4 *>(f) = *reinterpret_cast<const uint4 *>(v.nf + c0);
        *reinterpret_cast<uint4 *>(b) = *reinterpret_cast<const uint4 *>(v.nb + c0);
    } else {
#pragma unroll
        for (int k = 0; k < VOF_CELLS; ++k) {
            f[k] = c0 + k < v.ncell ? v.nf[c0 + k] : (int8_t)-1;
            b[k] = c0 + k < v.ncell ? v.nb[c0 + k] : (int8_t)0;
        }
    }
    int p[3];
    vof_pos(v, c0, p);
    bool bad = false;
    int ns = 0;
#pragma unroll
    for (int k = 0; k < VOF_CELLS; ++k) {
        if (c0 + k < v.ncell) {
            const bool ring = p[0] == 0 || p[0] == v.nx + 1 || p[1] == 0 || p[1] == v.ny + 1 || p[2] == 0 ||
                              p[2] == v.nz + 1;
            // object cells of the case (flag -1 with a nonzero object code) are not
            // covered: QFF's object branches (1sub-vof.F90:77-97) are not restated
            bad = bad || (ring && f[k] != -1) || f[k] < -1 || f[k] > 2 ||
                  (f[k] == 2 && (b[k] == 0 || b[k] < -3 || b[k] > 3)) || (f[k] == -1 && b[k] != 0);
            if (f[k] == 2) {
                state[c0 + k] = 0;
                ++ns;
            }
        }
        if (++p[0] == v.nx + 2) {
            p[0] = 0;
            if (++p[1] == v.ny + 2) {
                p[1] = 0;
                ++p[2];
            }
        }
    }
    if (bad) atomicOr(&cnt[VC_BAD], 1);
    const int l = threadIdx.x;
    int at = ns;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(at, d, 64);
        if (l >= d) at += o;
    }
    if (l == 63) nlist[blockIdx.x] = at;
    unsigned *mine = list + (size_t)blockIdx.x * VOF_SEG + at - ns;
#pragma unroll
    for (int k = 0; k < VOF_CELLS; ++k)
        if (c0 + k < v.ncell && f[k] == 2) *mine++ = (unsigned)(c0 + k);
}

// state: 0 pending, else 2*round + (1 if the cell's correction term is set).
// A cell counts a predecessor as decided only if it was decided in an
// earlier round (earlier launch), so the term it reads is complete.
__device__ inline bool vof_decided(int s, int round) { return s != 0 && (s >> 1) < round; }

__device__ __forceinline__ void vof_mod_cell(const VofDev &v, double dt, int round, int *state, double *term, long c,
                                             int *cnt, int slot) {
    if (state[c] != 0) return;
    const long st[3] = {1, (long)(v.nx + 2), (long)(v.nx + 2) * (v.ny + 2)};
    double sub[3] = {0.0, 0.0, 0.0};
    bool has[3] = {false, false, false};
    for (int l = 0; l < 3; ++l) {
        const long r = c - st[l];
        if (v.nf[r] == 2 && v.nb[r] == -(l + 1)) {
            const int s = state[r];
            if (!vof_decided(s, round)) {
                atomicAdd(&cnt[slot], 1);
                return;
            }
            if (s & 1) {
                sub[l] = term[r];
                has[l] = true;
            }
        }
    }
    int p[3];
    vof_pos(v, c, p);
    const double d = vof_df(v, c, p, dt, sub, has);
    if (d < VOF_FLIM) {
        state[c] = 2 * round;
        return;
    }
    const int b = v.nb[c], l = (b < 0 ? -b : b) - 1;
    const long n1 = b > 0 ? c : c + st[l];
    if (v.nf[n1] == -1) atomicOr(&cnt[VC_SOLID], 1);
    const double s = b > 0 ? 1.0 : -1.0;
    term[c] = v.dx[(size_t)l * v.stride + p[l]] * (d - 1.0) / dt * v.fb[c] / v.a[(size_t)l * v.ncell + n1] * s;
    state[c] = 2 * round + 1;
    atomicAdd(&cnt[VC_MODIFIED], 1);
}

// One round over the listed cells (a workgroup a segment), pending cells
// counted at cnt[slot]; not run where the round before (counted at prev, < 0:
// none) left none.
__global__ void __launch_bounds__(256)
k_vof_mod_eval(VofDev v, double dt, int round, int *__restrict__ state, double *__restrict__ term,
               const unsigned *__restrict__ list, const int *__restrict__ nlist, int *cnt, int prev, int slot) {
    if (!vof_valid(cnt) || (prev >= 0 && cnt[prev] == 0)) return;
    const int n = nlist[blockIdx.x];
    const unsigned *mine = list + (size_t)blockIdx.x * VOF_SEG;
    for (int q = threadIdx.x; q < n; q += 256) vof_mod_cell(v, dt, round, state, term, (long)mine[q], cnt, slot);
}

__device__ __forceinline__ void vof_apply_cell(const VofDev &v, const int *state, const double *term, long c) {
    if (!(state[c] & 1)) return;
    const long st[3] = {1, (long)(v.nx + 2), (long)(v.nx + 2) * (v.ny + 2)};
    const int b = v.nb[c], l = (b < 0 ? -b : b) - 1;
    const size_t n = (size_t)v.ncell;
    if (b > 0) {
        // own low face: a predecessor's correction first, then this one
        double q = v.qf[l * n + c];
        const long r = c - st[l];
        if (v.nf[r] == 2 && v.nb[r] == -(l + 1) && (state[r] & 1)) q = q - term[r];
        v.qf[l * n + c] = q - term[c];
    } else {
        const long t = c + st[l];
        if (v.nf[t] == -1) return;  // reported through VC_SOLID
        if (v.nf[t] == 2 && v.nb[t] == l + 1 && (state[t] & 1)) return;  // t applies both
        v.qf[l * n + t] = v.qf[l * n + t] - term[c];
    }
}
// Runs once no cell is pending; the last queued round's count becomes
// VC_PENDING's.
__global__ void __launch_bounds__(256)
k_vof_mod_apply(VofDev v, const int *__restrict__ state, const double *__restrict__ term,
                const unsigned *__restrict__ list, const int *__restrict__ nlist, const int *cnt) {
    if (!vof_settled(cnt)) return;
    const int n = nlist[blockIdx.x];
    const unsigned *mine = list + (size_t)blockIdx.x * VOF_SEG;
    for (int q = threadIdx.x; q < n; q += 256) vof_apply_cell(v, state, term, (long)mine[q]);
}

// What bounds it is HBM: 80 bytes a cell (waiting for the flags before the
// faces: 78 us at 4.4M cells; now 75, 57 at a large copy's rate).
__global__ void __launch_bounds__(256) k_vof_newf(VofDev v, double dt, int *cnt) {
    const long c = (long)vof_block() * blockDim.x + threadIdx.x;
    if (c >= v.ncell) return;
    const int f = v.nf[c];
    VofCell w;
    vof_load(v, c, w);
    if (!vof_settled(cnt)) return;
    if (f == -1) {
        v.Fn[c] = v.F[c];
        return;
    }
    int p[3];
    vof_pos(v, c, p);
    double d = vof_df(v, w, p, dt);
    v.D[c] = d;
    if (-d * dt * w.fb > 0.4) {
        atomicOr(&cnt[VC_RETRY], 1);
    } else if (fabs(d * dt) < VOF_TINY && d != 0.0) {
        d = 0.0;
    }
    if (d > VOF_FLIM && f == 2) atomicOr(&cnt[VC_STOP], 1);
    v.Fn[c] = d;
}

// simple_slide(0): one thread per column, k downwards.  cal_fslide_m0
// recomputes df_vof of the cell and of the one below before using them;
// those equal D (k_vof_newf's values on the same fluxes) unless a move in
// this column changed a face since: the cell's high face is changed by a
// move one level up (then its df_vof is the value that move left for the
// cell below), the lower cell's faces only by moves not yet made.
//
// A column is a serial walk of nz levels and there are only nx ny of them, so
// what bounds this is the chain of loads.  The flags of VOF_LEVELS levels are
// loaded at once, ahead of the walk, and where one of them may slide so are
// their D and fb; a move takes one trip more.  At 256 x 256 columns of 64 of
// which 25 levels slide, 76 us (one load after the other, and one counter for
// all moves: 144).  Everything a move needs loaded ahead: 72 to 77, and more
// where nothing slides; columns in 8 x 8 or 16 x 4 tiles: 80 to 88; 32 columns a
// wavefront: 96.
constexpr int VOF_LEVELS = 8;
__global__ void __launch_bounds__(64) k_vof_slide(VofDev v, double dt, int *cnt) {
    const int col = vof_block() * blockDim.x + threadIdx.x;
    if (col >= v.nx * v.ny) return;
    if (!vof_settled(cnt) || (cnt[VC_RETRY] | cnt[VC_STOP]) != 0) return;
    const int i = 1 + col % v.nx, j = 1 + col / v.nx;
    const long X = v.nx + 2, Y = v.ny + 2, sz = X * Y;
    const size_t S = (size_t)v.stride;
    const double dx0 = v.dx[i], dx1 = v.dx[S + j];
    int moved = 0;
    bool changed_above = false;  // qf(2, c + e_z) moved by the previous level
    double carried = 0.0;        // df_vof(c) after that move
    const long c0 = i + X * j;
    bool open = true;            // no solid cell met
    int nf[VOF_LEVELS + 1];      // of levels k0 .. k0 - VOF_LEVELS (level 0, solid, below them)
#pragma unroll
    for (int u = 0; u <= VOF_LEVELS; ++u) nf[u] = v.nf[c0 + sz * max(v.nz - u, 0)];
    for (int k0 = v.nz; k0 >= 1 && open; k0 -= VOF_LEVELS) {
        int nx[VOF_LEVELS + 1];  // the next levels'
#pragma unroll
        for (int u = 0; u <= VOF_LEVELS; ++u) nx[u] = v.nf[c0 + sz * max(k0 - VOF_LEVELS - u, 0)];
        bool any = false;
#pragma unroll
        for (int u = 0; u < VOF_LEVELS; ++u) any = any || (nf[u] != 1 && nf[u] != -1);
        double fb[VOF_LEVELS + 1], D[VOF_LEVELS + 1], dz[VOF_LEVELS + 1];
        if (any) {
#pragma unroll
            for (int u = 0; u <= VOF_LEVELS; ++u) {
                const int k = max(k0 - u, 0);
                fb[u] = v.fb[c0 + sz * k];
                D[u] = v.D[c0 + sz * k];  // of a solid cell: not used
                dz[u] = v.dx[2 * S + k];
            }
        }
#pragma unroll
        for (int u = 0; u < VOF_LEVELS; ++u) {
            const int k = k0 - u;
            if (!open || k < 1) continue;
            const long c = c0 + sz * k, m = c - sz;
            if (nf[u] == -1) {
                open = false;
                continue;
            }
            const bool above = changed_above;
            changed_above = false;
            if (nf[u] == 1 || nf[u + 1] == -1) continue;
            const double vmesh = dx0 * dx1 * dz[u];
            const double dvc = vmesh * fb[u];
            const double dvm = dx0 * dx1 * dz[u + 1] * fb[u + 1];
            if (dvc * dvm == 0.0) continue;
            const double fc = above ? carried : D[u];
            const double fm = D[u + 1];
            v.Fn[c] = fc;
            v.Fn[m] = fm;
            const double t1 = dvm * (1.0 - fm), t2 = dvc * fc;
            const double f2 = t1 < t2 ? t1 : t2;
            if (fabs(f2) == 0.0) continue;
            // both cells' fields before the move, in one trip; the moved face is
            // the one's low and the other's high
            VofCell wc, wm;
            vof_load(v, c, wc);
            vof_load(v, m, wm);
            const double q = wc.q[2] + -1.0 * f2 / vmesh / dt * dz[u] / wc.a[2];
            v.qf[2 * (size_t)v.ncell + c] = q;
            wc.q[2] = wm.qh[2] = q;
            const int pc[3] = {i, j, k}, pm[3] = {i, j, k - 1};
            const double ft = vof_df(v, wc, pc, dt);
            v.Fn[c] = fabs(ft) < VOF_TINY ? 0.0 : ft;
            carried = vof_df(v, wm, pm, dt);
            v.Fn[m] = carried;
            changed_above = true;
            ++moved;
        }
#pragma unroll
        for (int u = 0; u <= VOF_LEVELS; ++u) nf[u] = nx[u];
    }
    if (moved) atomicAdd(&cnt[VC_SLID + VC_LINE * (blockIdx.x % VC_SLOTS)], moved);
}

} // namespace clowns
