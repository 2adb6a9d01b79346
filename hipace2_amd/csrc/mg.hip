// Geometric multigrid for the explicit Bx/By system on gfx950 (hpmg type I):
//   -acf * sol + Lap(sol) = rhs, homogeneous Dirichlet, two components sharing acf.
//
// Semantics are those of the reference's CPU build of hpmg::MultiGrid
// (src/mg_solver/HpMultiGrid.cpp): node-centred levels for odd n, cell-centred with the
// 4/3 boundary stencil for even n (ctor :1043-1163); V-cycle :1430-1512 with four
// red-black Gauss-Seidel sweeps (+ residual) per level, full-weighting restriction and
// bilinear (node) / piecewise-constant (cell) prolongation; bottom solve of
// max(16, box length) sweeps on the coarsest level (:1583-1593); convergence on the max
// norm of the residual (:1330-1416). Every point update uses the reference's operation
// order, so the iterates equal the CPU build's for equal inputs. The diagonal inverse
// 1/c0 of a point depends only on acf and the point's position, so it is computed once
// per solve, in the first pass over a level, and kept.
//
// Mapping to the GPU: the sweeps (+ residual) of one level are one launch of an LDS-tiled
// kernel: each workgroup loads its tile of one component plus a halo of NSW to NSW + 2
// points, runs the NSW colour sweeps in LDS (points NSW or more away from the frozen outer
// ring see exactly the values a global sweep gives them) and writes back the interior; the
// residual, its restriction to the next level and its max norm come out of the same launch.
// Prolongation is fused into the load of the up-sweep. On level 0 the up-sweep and the
// final smoothing of the cycle are one launch of eight sweeps that leaves every
// workgroup's residual max norm; a one-workgroup launch after it reduces them, evaluates
// convergence and publishes the result to pinned host memory, which the host polls
// instead of synchronising the stream. Levels from the first one that fits (65x65 points
// and the like) down run as one workgroup per component that does the coarse part of the
// V-cycle with barriers between sweeps, its arrays in LDS; the levels of at most 64 points
// of a colour run in its first wavefront alone, without workgroup barriers. For odd n the
// level-0 arrays are the caller's planes themselves (the node-centred level-0 box with
// its ghost ring has the slice store's guarded shape).
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>

#include "barrier.hpp"
#include "internal.hpp"

namespace hpq {

namespace {

constexpr int NT = 512;                        // threads per workgroup

__host__ __device__ __forceinline__ long at(const MGLevel& L, int i, int j) {
    return long(j - L.jlo + 1) * L.ldx + (i - L.ilo + 1);
}

// Tile of this workgroup. Workgroups go to the eight XCDs in turn (linear id mod 8), and
// each XCD has its own L2: the tiles are renumbered so that XCD k takes the k-th eighth of
// the tiles in row-major order, a band of whole tile rows, and the halos that neighbouring
// tiles read twice are mostly read from that XCD's L2 (ids beyond the last multiple of
// eight keep their tile).
__device__ __forceinline__ void xcd_tile(int& bx, int& by) {
    const int gx = int(gridDim.x), n = gx * int(gridDim.y);
    const int id = int(blockIdx.x) + int(blockIdx.y) * gx;
    const int m = n & ~7;
    const int t = id < m ? (id & 7) * (m >> 3) + (id >> 3) : id;
    by = t / gx;
    bx = t - by * gx;
}
template <class LV>
__device__ __forceinline__ bool in_valid(const LV& L, int i, int j) {
    return i >= L.vilo && i <= L.vihi && j >= L.vjlo && j <= L.vjhi;
}
__host__ __device__ __forceinline__ int cdiv2(int v) { return v >= 0 ? v / 2 : -((-v + 1) / 2); }

// 1/c0 of gs1<is_cell_centered> (HpMultiGrid.cpp:267-292)
template <bool CC, class LV>
__device__ __forceinline__ double c0_inverse(const LV& L, int i, int j, double acf, double facx, double facy) {
    double c0 = -(acf + 2. * (facx + facy));
    if (CC && (i == L.ilo || i == L.ihi)) c0 -= 2. * facx;
    if (CC && (j == L.jlo || j == L.jhi)) c0 -= 2. * facy;
    return 1. / c0;
}

// the update of gs1<is_cell_centered> (HpMultiGrid.cpp:267-292); P(a, b) reads phi at
// offset (a, b)
template <bool CC, class LV, class PF>
__device__ __forceinline__ double gs_point(const LV& L, int i, int j, PF P, double rhs, double c0_inv, double facx,
                                           double facy) {
    double l;
    if (CC && i == L.ilo) l = facx * (4. / 3.) * P(1, 0);
    else if (CC && i == L.ihi) l = facx * (4. / 3.) * P(-1, 0);
    else l = facx * (P(-1, 0) + P(1, 0));
    if (CC && j == L.jlo) l += facy * (4. / 3.) * P(0, 1);
    else if (CC && j == L.jhi) l += facy * (4. / 3.) * P(0, -1);
    else l += facy * (P(0, -1) + P(0, 1));
    return (rhs - l) * c0_inv;
}

// the same on a cell-centred level, with the one-sided stencil chosen by selects
template <class LV>
__device__ __forceinline__ double gs_edge(const LV& L, int i, int j, double w, double e, double b, double t, double rhs,
                                          double c0_inv) {
    const bool x0 = i == L.ilo, x1 = i == L.ihi, y0 = j == L.jlo, y1 = j == L.jhi;
    double l = (x0 || x1 ? L.facx * (4. / 3.) : L.facx) * (x0 ? e : x1 ? w : w + e);
    l += (y0 || y1 ? L.facy * (4. / 3.) : L.facy) * (y0 ? t : y1 ? b : b + t);
    return (rhs - l) * c0_inv;
}

// laplacian + residual1 (HpMultiGrid.cpp:163-190). The box-edge branches only fire on
// cell-centred levels: on node-centred ones the edge nodes are not valid points.
template <bool CC, class LV, class PF>
__device__ __forceinline__ double residual1(const LV& L, int i, int j, PF P, double rhs, double acf, double facx,
                                            double facy) {
    double r = -2. * (facx + facy) * P(0, 0);
    if (CC && i == L.ilo) r += facx * (4. / 3. * P(1, 0) - 2. * P(0, 0));
    else if (CC && i == L.ihi) r += facx * (4. / 3. * P(-1, 0) - 2. * P(0, 0));
    else r += facx * (P(-1, 0) + P(1, 0));
    if (CC && j == L.jlo) r += facy * (4. / 3. * P(0, 1) - 2. * P(0, 0));
    else if (CC && j == L.jhi) r += facy * (4. / 3. * P(0, -1) - 2. * P(0, 0));
    else r += facy * (P(0, -1) + P(0, 1));
    return rhs + acf * P(0, 0) - r;
}

// fine_in + I(crse) at fine point (i, j) (interpcpy_cc / interpcpy_nd, :88-121) from the
// coarse values c00 .. c11 at (ic, jc), (ic + 1, jc), (ic, jc + 1), (ic + 1, jc + 1), ic = i / 2;
// no branch: the sum and its factor (a power of two) are chosen by selects
template <bool CC>
__device__ __forceinline__ double interp_sum(int i, int j, double fine_in, double c00, double c10, double c01,
                                             double c11) {
    if (CC) return fine_in + c00;
    const bool io = (i & 1) != 0, jo = (j & 1) != 0;
    double t = c00;
    t = io ? t + c10 : t;
    t = jo ? t + c01 : t;
    t = io && jo ? t + c11 : t;
    return fine_in + t * (io && jo ? 0.25 : io || jo ? 0.5 : 1.0);
}

// restrict_cc / restrict_nd (:31-52) at coarse point (i, j); f(a, b) reads the fine array
template <bool CC, class FA>
__device__ __forceinline__ double restrict_from(FA f, int i, int j) {
    if (CC) return 0.25 * (f(2 * i, 2 * j) + f(2 * i + 1, 2 * j) + f(2 * i, 2 * j + 1) + f(2 * i + 1, 2 * j + 1));
    return (1. / 16.) * (f(2 * i - 1, 2 * j - 1) + 2. * f(2 * i, 2 * j - 1) + f(2 * i + 1, 2 * j - 1) +
                         2. * f(2 * i - 1, 2 * j) + 4. * f(2 * i, 2 * j) + 2. * f(2 * i + 1, 2 * j) +
                         f(2 * i - 1, 2 * j + 1) + 2. * f(2 * i, 2 * j + 1) + f(2 * i + 1, 2 * j + 1));
}


__device__ void clear_ctl(MGCtl* c) {
    c->done = 0; c->iters = 0; c->status = 0;
    c->max_norm = 0; c->res_target = 0;
}

// one relaxed 64-bit store: the host sees the whole word or none of it
__device__ void publish(const MGCtl* c, MGMirror* m, int seq) {
    const unsigned long long w = (unsigned long long)(unsigned)seq | ((unsigned long long)(c->iters & 0xffffff) << 32) |
                                 ((unsigned long long)(c->status & 0x7f) << 56) |
                                 ((unsigned long long)(c->done ? 1 : 0) << 63);
    __hip_atomic_store(&m->word, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// end of one V-cycle (solve_doit :1371-1417), run by k_check with the max norm of the
// cycle's residual
__device__ void end_cycle(MGCtl* ctl, MGCtl* other, MGMirror* mirror, int seq, int maxiter, double norminf) {
    ctl->iters += 1;
    if (norminf <= ctl->res_target) {
        ctl->done = 1;
    } else if (norminf > 1.e20 * ctl->max_norm) {
        ctl->done = 1;
        ctl->status = HPQ_E_MG_DIVERGED;
    } else if (ctl->iters >= maxiter) {
        ctl->done = 1;
        ctl->status = HPQ_E_MG_NOT_CONVERGED;
    }
    if (ctl->done) clear_ctl(other);
    publish(ctl, mirror, seq);
}

// convergence target after the initial residual (solve_doit :1330-1366)
__device__ void end_initial(MGCtl* ctl, MGCtl* other, double tol_rel, double tol_abs, double resnorm0,
                            double rhsnorm0) {
    const double max_norm = (rhsnorm0 >= resnorm0) ? rhsnorm0 : resnorm0;
    ctl->max_norm = max_norm;
    ctl->res_target = fmax(tol_abs, fmax(tol_rel, 1.e-16) * max_norm);
    if (resnorm0 <= ctl->res_target) {
        ctl->done = 1;
        clear_ctl(other);
    }
}

// Arguments of the convergence bookkeeping after a level-0 launch.
struct Check {
    MGCtl* ctl;
    MGCtl* other;
    MGMirror* mirror;
    const double* norms;   // max |residual|, max |rhs| of every workgroup of the launch
    int nblk, seq, maxiter;
    double tol_rel, tol_abs;
};

// max over the workgroups' entries norms[2 b + k], one workgroup of NT threads
__device__ double max_norms(const double* norms, int nblk, int k, double* red) {
    double m = 0.0;
    for (int b = threadIdx.x; b < nblk; b += NT) m = fmax(m, norms[2 * b + k]);
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    double mm = red[0];
    for (int w = 1; w < NT / 64; ++w) mm = fmax(mm, red[w]);
    return mm;
}

// end of one V-cycle; a cycle enqueued after convergence only reports that it drained
__global__ __launch_bounds__(NT) void k_check(Check chk) {
    __shared__ double red[NT / 64];
    if (chk.ctl->done) {
        if (threadIdx.x == 0) publish(chk.ctl, chk.mirror, chk.seq);
        return;
    }
    const double norminf = max_norms(chk.norms, chk.nblk, 0, red);
    if (threadIdx.x == 0) end_cycle(chk.ctl, chk.other, chk.mirror, chk.seq, chk.maxiter, norminf);
}

// the convergence target; with seq != 0 the result (done after zero V-cycles or not) is
// published to the host as well
__global__ __launch_bounds__(NT) void k_target(Check chk) {
    __shared__ double red[NT / 64];
    const double resnorm0 = max_norms(chk.norms, chk.nblk, 0, red);
    const double rhsnorm0 = max_norms(chk.norms, chk.nblk, 1, red);
    if (threadIdx.x == 0) {
        end_initial(chk.ctl, chk.other, chk.tol_rel, chk.tol_abs, resnorm0, rhsnorm0);
        if (chk.seq) publish(chk.ctl, chk.mirror, chk.seq);
    }
}

// Convergence bookkeeping carried by the first launch of a V-cycle instead of a launch of
// its own. TARGET (before cycle 0): the convergence target from the initial residual and
// rhs norms, as k_target sets it. CHECK (before cycle m >= 1): the end of cycle m - 1, as
// k_check evaluates it, with m cycles done. Every workgroup of the launch reduces the
// level-0 norms and reaches the same decision; workgroup 0 records it in the control block.
struct Fold {
    enum : int { NONE = 0, TARGET = 1, CHECK = 2 };
    int mode = NONE;
    int m = 0, maxiter = 0, nblk = 0;
    double tol_rel = 0.0, tol_abs = 0.0;
    const double* norms = nullptr;
    MGCtl* ctl = nullptr;
    MGCtl* other = nullptr;
};

// the folded decision: whether the solve is finished before this launch's work
__device__ bool fold_decide(const Fold& f, const MGCtl* gate, double* red) {
    if (f.mode == Fold::NONE) return gate ? gate->done != 0 : false;
    const bool lead = blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0;
    if (f.mode == Fold::TARGET) {
        const double resnorm0 = max_norms(f.norms, f.nblk, 0, red);
        const double rhsnorm0 = max_norms(f.norms, f.nblk, 1, red);
        const double max_norm = (rhsnorm0 >= resnorm0) ? rhsnorm0 : resnorm0;
        const double target = fmax(f.tol_abs, fmax(f.tol_rel, 1.e-16) * max_norm);
        const bool done = resnorm0 <= target;
        if (lead) {
            f.ctl->max_norm = max_norm;
            f.ctl->res_target = target;
            if (done) {
                f.ctl->done = 1;
                clear_ctl(f.other);
            }
        }
        return done;
    }
    // CHECK: the control block's done flag is set by this solve's earlier launches, or by
    // workgroup 0 of this one with the decision every workgroup reaches here; one thread
    // reads it for the whole workgroup (after the barriers of the reduction), so all of its
    // threads take the same branch
    __shared__ int done_before;
    const double norminf = max_norms(f.norms, f.nblk, 0, red);
    if (threadIdx.x == 0) done_before = f.ctl->done;
    __syncthreads();
    if (done_before) return true;
    int status = 0;
    bool done = false;
    if (norminf <= f.ctl->res_target) {
        done = true;
    } else if (norminf > 1.e20 * f.ctl->max_norm) {
        done = true;
        status = HPQ_E_MG_DIVERGED;
    } else if (f.m >= f.maxiter) {
        done = true;
        status = HPQ_E_MG_NOT_CONVERGED;
    }
    if (lead) {
        f.ctl->iters = f.m;
        if (done) {
            f.ctl->status = status;
            f.ctl->done = 1;
            clear_ctl(f.other);
        }
    }
    return done;
}

// Tile of a k_smooth launch. A wavefront holds two swept rows of 32 points of one colour each,
// a thread KP points of each colour NT / 32 rows apart, so the swept region is 64 x (16 KP)
// points and the tile what is left inside it: after NSW sweeps a point is exact if
// it lies NSW or more points inside the frozen ring, the residual needs one neighbour more and
// the full weighting of node-centred levels the residual of one ring around the tile.
template <int NSW, bool CC, bool RES, int KP>
struct Tile {
    static constexpr int HALO = NSW + (RES ? (CC ? 1 : 2) : 0);
    static constexpr int SW = 64, SH = NT / 32 * KP;
    static constexpr int LX = SW + 2, LY = SH + 2;
    static constexpr int TX = LX - 2 * HALO, TY = LY - 2 * HALO;
    static_assert(TX > 0 && TY > 0 && TX % 2 == 0 && TY % 2 == 0, "the tile holds whole coarse points");
};

// NSW red-black sweeps (colours 0,1,2,3,0,1,...) of one level, LDS-tiled, optionally
// followed by the residual and its restriction to the coarse points this tile owns (res_c).
// Start: zero (ZERO), phi_in + I(cor_c) (INTERP) or phi_in. Result -> phi_out.
// NORMS: the workgroup's max |residual| over its tile and (RHSMAX) max |rhs| over its
// points go to norms[2 b], norms[2 b + 1] for the convergence check that follows.
// FIRST, a solve's first pass over the level: 1/c0 of the tile's points is computed from acf
// and kept for the later passes, and acf is restricted to the coarse points the tile owns
// (average_down_acoef, :1641-1661), which prepares the next level's coefficient.
// Every launch returns at once when the control block says the solve is finished (the
// data loads are issued before that flag is tested, so its latency is hidden).
//
// The two components are independent systems with the same acf: each has workgroups of its
// own. A thread owns KP points of each parity of (i + j) and keeps their rhs and 1/c0 in
// registers. A sweep of one colour touches one parity class
// only; the thread reads all neighbours of its points first, then updates, then writes
// (points of one colour never neighbour each other, so this is the order a global sweep has).
// Bound by latency on the small levels and by issue on the large ones: a sweep is one LDS
// round trip, a chain of seven FP64 operations and a barrier. All points of a thread share
// their LDS addresses up to a constant, the parity of i and that of j, so the sweeps and the
// prolongation have no index arithmetic. Nothing is read under a condition: global indices
// are clamped to the box and only the store of a swept point is predicated; a fence after
// each group of reads keeps the compiler from waiting for them one by one. Measured, and before
// with tiles of 32 x 16 points, both components in 256 threads and conditional reads: four sweeps
// of a small level 4.6 us (8.7; an empty launch takes 2), eight sweeps of 255 x 255 points 7.8 us
// (15.6), of 511 x 511 14.4 us (19.3), of 1023 x 1023 39 us (58; with KP = 4, 38).
template <int NSW, bool CC, bool ZERO, bool RES, bool INTERP, bool RHSMAX, bool NORMS, bool FIRST, int KP>
__global__ __launch_bounds__(NT, 4) void k_smooth(MGLevel L, MGLevel C, double* __restrict__ phi_out,
                                               const double* __restrict__ rhs, long rcs,
                                               const double* __restrict__ acf, const double* __restrict__ phi_in,
                                               const double* __restrict__ cor_c, double* __restrict__ res_c,
                                               const MGCtl* __restrict__ gate, double* __restrict__ norms,
                                               Fold fold) {
    static_assert(NSW % 2 == 0, "sweeps come in red-black pairs");
    static_assert(!NORMS || RES, "the norms come from the residual");
    static_assert(!FIRST || RES, "acf is restricted with the residual");
    using T = Tile<NSW, CC, RES, KP>;
    constexpr int HALO = T::HALO, TX = T::TX, TY = T::TY, LX = T::LX, LY = T::LY;
    constexpr int RS = NT / 32;                    // rows between a thread's points
    // rows of the residual (the tile and, node-centred, one ring) among a thread's KP points
    constexpr int RING = CC ? 0 : 1;
    constexpr int QA = RES ? (HALO - RING - 1) / RS : (HALO - 1) / RS;
    constexpr int QB = RES ? (HALO + TY + RING - 2) / RS + 1 : (HALO + TY - 2) / RS + 1;
    // LDS holds the two colours of the tile apart: point (lx, ly) lives in
    // s[(i + j) & 1][ly][lx >> 1], so a colour sweep and its neighbour reads walk consecutive
    // doubles across the lanes
    constexpr int LXH = LX / 2, PL = LY * LXH;
    constexpr int CLX = INTERP ? LX / 2 + 2 : 1, CLY = INTERP ? LY / 2 + 2 : 1;
    constexpr int NCL = (CLX * CLY + NT - 1) / NT;
    __shared__ double s[2 * PL];
    __shared__ double cc[CLX * CLY];               // the coarse correction under the tile
    __shared__ double red[2][NT / 64];
    const int gate_done = (fold.mode == Fold::NONE) ? (gate ? gate->done : 0) : 0;
    int bx, by;
    xcd_tile(bx, by);
    const int comp = bx & 1, tid = int(threadIdx.x);
    bx >>= 1;
    const int ti0 = L.vilo + bx * TX - HALO;
    const int tj0 = L.vjlo + by * TY - HALO;
    const double facx = L.facx, facy = L.facy;
    // global offsets count from the first valid point of the region, clamped to the valid box
    const int oi = max(ti0, L.vilo), oj = max(tj0, L.vjlo);
    const long ko = at(L, oi, oj);
    const double* const rhs_o = rhs + (comp ? rcs : 0) + ko;
    const double* const phi_o = ZERO ? nullptr : phi_in + (comp ? L.cs : 0) + ko;
    const double* const acf_o = acf + ko;
    double* const out_o = phi_out + (comp ? L.cs : 0) + ko;
    double* const c0i_o = L.c0i + ko;
    const int omax = (L.vjhi - oj) * L.ldx;
    auto ld = [](const double* b, int k) {
        return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(b) + unsigned(k) * 8u);
    };
    // owned points: column lx[par], rows ly + RS q; ks is the index of q = 0 in its colour's
    // plane, kw that of its west neighbour in the other one
    const int ly = 1 + (tid >> 5);
    const int row0 = __mul24(tj0 + ly - oj, L.ldx), rstep = RS * L.ldx;
    int lx[2], ks[2], kw[2], col[2];
    bool vi[2], vj[KP];
#pragma unroll
    for (int par = 0; par < 2; ++par) {
        lx[par] = 1 + 2 * (tid & 31) + ((par + ti0 + tj0 + ly + 1) & 1);
        ks[par] = ly * LXH + (lx[par] >> 1);
        kw[par] = ly * LXH + ((lx[par] - 1) >> 1);
        const int i = ti0 + lx[par];
        col[par] = min(max(i, oi), L.vihi) - oi;
        vi[par] = i >= L.vilo && i <= L.vihi;
    }
    double r0[2][KP], ci[2][KP], v[2][KP];
#pragma unroll
    for (int q = 0; q < KP; ++q) {
        const int j = tj0 + ly + RS * q;
        vj[q] = j >= L.vjlo && j <= L.vjhi;
        const int row = min(max(row0 + q * rstep, 0), omax);
#pragma unroll
        for (int par = 0; par < 2; ++par) {
            const int k = row + col[par];
            r0[par][q] = ld(rhs_o, k);
            ci[par][q] = FIRST ? ld(acf_o, k) : ld(c0i_o, k);
            v[par][q] = ZERO ? 0.0 : ld(phi_o, k);
        }
    }
    // the frozen ring without its corners: threads [0, 64) its first row, [64, 128) the last,
    // the next LY - 2 the first column, the next the last
    constexpr int NRING = 2 * T::SW + 2 * (LY - 2), KRING = (NRING + NT - 1) / NT;
    double vr[KRING];
    auto ring = [&](int q, int& x, int& y) {
        const int e = tid + q * NT;
        const int f = e - 2 * T::SW;
        x = e < 2 * T::SW ? 1 + (e & 63) : f < LY - 2 ? 0 : LX - 1;
        y = e < T::SW ? 0 : e < 2 * T::SW ? LY - 1 : 1 + (f < LY - 2 ? f : min(f - (LY - 2), LY - 3));
    };
#pragma unroll
    for (int q = 0; q < KRING; ++q) {
        int x, y;
        ring(q, x, y);
        vr[q] = ZERO ? 0.0
                     : ld(phi_o, min(max(__mul24(tj0 + y - oj, L.ldx), 0), omax) +
                                     (min(max(ti0 + x, oi), L.vihi) - oi));
    }
    const int ic0 = cdiv2(ti0), jc0 = cdiv2(tj0);
    double cv[NCL];
    if (INTERP) {
        const double* const cor_k = cor_c + (comp ? C.cs : 0);
#pragma unroll
        for (int it = 0; it < NCL; ++it) {
            const int e = min(tid + it * NT, CLX * CLY - 1);
            const int cy = e / CLX, cx = e - cy * CLX;
            cv[it] = cor_k[at(C, min(max(ic0 + cx, C.ilo - 1), C.ihi + 1), min(max(jc0 + cy, C.jlo - 1), C.jhi + 1))];
        }
    }
    if (gate_done) return;
    // a folded convergence decision: its norm loads are issued after the tile's own
    if (fold.mode != Fold::NONE && fold_decide(fold, nullptr, &red[0][0])) return;
    if (INTERP) {
#pragma unroll
        for (int it = 0; it < NCL; ++it) cc[min(tid + it * NT, CLX * CLY - 1)] = cv[it];
        lds_barrier();
#pragma unroll
        for (int q = 0; q < KRING; ++q) {
            int x, y;
            ring(q, x, y);
            const int i = ti0 + x, j = tj0 + y;
            const double* const p = cc + (cdiv2(j) - jc0) * CLX + (cdiv2(i) - ic0);
            const double c00 = p[0], c10 = CC ? 0.0 : p[1], c01 = CC ? 0.0 : p[CLX], c11 = CC ? 0.0 : p[CLX + 1];
            vr[q] = interp_sum<CC>(i, j, vr[q], c00, c10, c01, c11);
        }
    }
    double rmax = 0.0;
#pragma unroll
    for (int par = 0; par < 2; ++par) {
        if (INTERP) {
            const int i = ti0 + lx[par], j = tj0 + ly;
            const double* const p = cc + (cdiv2(j) - jc0) * CLX + (cdiv2(i) - ic0);
            // node-centred: i and j are both even or both odd for colour 0 (the coarse point
            // or four of them), one of them is odd for colour 1 (two along that direction)
            const bool jo = (j & 1) != 0;
            const int p1 = par == 0 || !jo ? 1 : CLX;
            double c[4][KP];
#pragma unroll
            for (int q = 0; q < KP; ++q) {
                const double* const pq = p + q * (RS / 2) * CLX;
                c[0][q] = pq[0];
                if (!CC) c[1][q] = pq[p1];
                if (!CC && par == 0) {
                    c[2][q] = pq[CLX];
                    c[3][q] = pq[CLX + 1];
                }
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int q = 0; q < KP; ++q) {
                if (CC) v[par][q] += c[0][q];
                else if (par == 1) v[par][q] += (c[0][q] + c[1][q]) * 0.5;
                else {
                    const double four = (c[0][q] + c[1][q] + c[2][q] + c[3][q]) * 0.25;
                    v[par][q] += jo ? four : c[0][q];
                }
            }
        }
#pragma unroll
        for (int q = 0; q < KP; ++q) {
            s[par * PL + ks[par] + q * RS * LXH] = vi[par] && vj[q] ? v[par][q] : 0.0;
            if (RHSMAX) rmax = fmax(rmax, fabs(r0[par][q]));
            if (FIRST) {
                ci[par][q] = c0_inverse<CC>(L, ti0 + lx[par], tj0 + ly + RS * q, ci[par][q], facx, facy);
                const int y = ly + RS * q;
                const bool out = lx[par] >= HALO && lx[par] < HALO + TX && y >= HALO && y < HALO + TY;
                if (comp == 0 && out && vi[par] && vj[q]) c0i_o[row0 + q * rstep + col[par]] = ci[par][q];
            }
        }
        asm volatile("" ::: "memory");   // one colour at a time, for the registers
    }
#pragma unroll
    for (int q = 0; q < KRING; ++q) {
        int x, y;
        ring(q, x, y);
        if (tid + q * NT < NRING)
            s[((ti0 + tj0 + x + y) & 1) * PL + y * LXH + (x >> 1)] = in_valid(L, ti0 + x, tj0 + y) ? vr[q] : 0.0;
    }
    lds_barrier();
    // cell-centred tiles at the edge of the box have points with a one-sided stencil
    const bool edge = CC && (ti0 + 1 <= L.ilo || ti0 + T::SW >= L.ihi || tj0 + 1 <= L.jlo || tj0 + T::SH >= L.jhi);
    // one colour: reads, then updates, then writes
    auto sweep = [&](auto PARC) {
        constexpr int par = decltype(PARC)::value;
        // a point of colour par has (i + j) & 1 == par; its neighbours the other one
        const double* const sn = s + (1 - par) * PL;
        double w[KP], e[KP], b[KP], t[KP], u[KP];
#pragma unroll
        for (int q = 0; q < KP; ++q) {
            w[q] = sn[kw[par] + q * RS * LXH];
            e[q] = sn[kw[par] + q * RS * LXH + 1];
            b[q] = sn[ks[par] + (q * RS - 1) * LXH];
            t[q] = sn[ks[par] + (q * RS + 1) * LXH];
        }
        asm volatile("" ::: "memory");
        if (CC && edge) {
#pragma unroll
            for (int q = 0; q < KP; ++q)
                u[q] = gs_edge(L, ti0 + lx[par], tj0 + ly + RS * q, w[q], e[q], b[q], t[q], r0[par][q], ci[par][q]);
        } else {
#pragma unroll
            for (int q = 0; q < KP; ++q) {
                double l = facx * (w[q] + e[q]);
                l += facy * (b[q] + t[q]);
                u[q] = (r0[par][q] - l) * ci[par][q];
            }
        }
        // all updates before the first predicated store, or each would be moved under its own
#pragma unroll
        for (int q = 0; q < KP; ++q) asm volatile("" : "+v"(u[q]));
#pragma unroll
        for (int q = 0; q < KP; ++q)
            if (vi[par] && vj[q]) s[par * PL + ks[par] + q * RS * LXH] = u[q];
        lds_barrier();
    };
    // colour c updates the points with (i + j + c) even, i.e. parity c & 1
#pragma unroll 1
    for (int c2 = 0; c2 < NSW - 2; c2 += 2) {
        sweep(std::integral_constant<int, 0>{});
        sweep(std::integral_constant<int, 1>{});
    }
    // acf of the residual's points, in flight during the last two sweeps
    double ar[2][RES ? QB - QA : 1];
    if (RES) {
#pragma unroll
        for (int q = QA; q < QB; ++q) {
            const int row = min(max(row0 + q * rstep, 0), omax);
            ar[0][q - QA] = ld(acf_o, row + col[0]);
            ar[1][q - QA] = ld(acf_o, row + col[1]);
        }
    }
    sweep(std::integral_constant<int, 0>{});
    sweep(std::integral_constant<int, 1>{});
    double m = 0.0;
    double z[2][QB - QA], g[2][RES ? QB - QA : 1];
#pragma unroll
    for (int par = 0; par < 2; ++par) {
        const double* const sn = s + (1 - par) * PL;
        double w[QB - QA], e[QB - QA], b[QB - QA], t[QB - QA];
#pragma unroll
        for (int q = QA; q < QB; ++q) {
            z[par][q - QA] = s[par * PL + ks[par] + q * RS * LXH];
            if (RES) {
                w[q - QA] = sn[kw[par] + q * RS * LXH];
                e[q - QA] = sn[kw[par] + q * RS * LXH + 1];
                b[q - QA] = sn[ks[par] + (q * RS - 1) * LXH];
                t[q - QA] = sn[ks[par] + (q * RS + 1) * LXH];
            }
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int q = QA; q < QB; ++q) asm volatile("" : "+v"(z[par][q - QA]));
#pragma unroll
        for (int q = QA; q < QB; ++q) {
            const int n = q - QA, y = ly + RS * q;
            const bool val = vi[par] && vj[q];
            const bool out = val && lx[par] >= HALO && lx[par] < HALO + TX && y >= HALO && y < HALO + TY;
            if (out) out_o[row0 + q * rstep + col[par]] = z[par][n];
            if (RES) {
                auto P = [&](int di, int dj) {
                    return di < 0 ? w[n] : di > 0 ? e[n] : dj < 0 ? b[n] : dj > 0 ? t[n] : z[par][n];
                };
                const double x = CC && edge
                                     ? residual1<CC>(L, ti0 + lx[par], tj0 + y, P, r0[par][q], ar[par][n], facx, facy)
                                     : residual1<false>(L, 0, 0, P, r0[par][q], ar[par][n], facx, facy);
                if (out) m = fmax(m, fabs(x));
                // points outside the valid box hold zero residual
                g[par][n] = val ? x : 0.0;
            }
        }
    }
    if (RES) {
        // the residual takes the place of the iterate
        lds_barrier();
#pragma unroll
        for (int par = 0; par < 2; ++par)
#pragma unroll
            for (int q = QA; q < QB; ++q) s[par * PL + ks[par] + q * RS * LXH] = g[par][q - QA];
        lds_barrier();
        // coarse points whose centre fine point 2*ic lies in this tile: TX/2 x TY/2 of them
        static_assert(TX / 2 <= 32, "one lane per coarse point of a row");
        const int ic = cdiv2(ti0 + HALO + 1) + (tid & 31);
        auto restricted = [&](int jc) {
            // the four diagonal neighbours have the centre's parity, 0, the others parity 1
            const int cx = 2 * ic - ti0, cy = 2 * jc - tj0;
            const double* const p0 = s + cy * LXH;
            const double* const p1 = p0 + PL;
            const int xw = (cx - 1) >> 1, xc = cx >> 1, xe = (cx + 1) >> 1;
            double f[9];
            f[4] = p0[xc];
            f[5] = p1[xe];
            f[7] = p1[LXH + xc];
            f[8] = p0[LXH + xe];
            if (!CC) {
                f[0] = p0[xw - LXH];
                f[1] = p1[xc - LXH];
                f[2] = p0[xe - LXH];
                f[3] = p1[xw];
                f[6] = p0[xw + LXH];
            }
            asm volatile("" ::: "memory");
            auto F = [&](int a, int b) { return f[(b - 2 * jc + 1) * 3 + (a - 2 * ic) + 1]; };
            return restrict_from<CC>(F, ic, jc);
        };
        const int jc_0 = cdiv2(tj0 + HALO + 1) + (tid >> 5);
        const bool own = (tid & 31) < TX / 2 && ic >= C.vilo && ic <= C.vihi;
#pragma unroll
        for (int q = 0; q < TY / 2; q += RS) {
            const int jc = jc_0 + q;
            if (own && q + (tid >> 5) < TY / 2 && jc >= C.vjlo && jc <= C.vjhi)
                res_c[at(C, ic, jc) + (comp ? C.cs : 0)] = restricted(jc);
        }
        if (FIRST) {
            lds_barrier();
            if (comp == 0) {
                // then acf that of the residual
#pragma unroll
                for (int par = 0; par < 2; ++par)
#pragma unroll
                    for (int q = QA; q < QB; ++q)
                        s[par * PL + ks[par] + q * RS * LXH] = vi[par] && vj[q] ? ar[par][q - QA] : 0.0;
            }
            lds_barrier();
            if (comp == 0) {
#pragma unroll
                for (int q = 0; q < TY / 2; q += RS) {
                    const int jc = jc_0 + q;
                    if (own && q + (tid >> 5) < TY / 2 && jc >= C.vjlo && jc <= C.vjhi)
                        C.acf[at(C, ic, jc)] = restricted(jc);
                }
            }
        }
    }
    if (NORMS) {
        for (int o = 32; o > 0; o >>= 1) {
            m = fmax(m, __shfl_xor(m, o));
            if (RHSMAX) rmax = fmax(rmax, __shfl_xor(rmax, o));
        }
        if ((threadIdx.x & 63) == 0) {
            red[0][threadIdx.x >> 6] = m;
            red[1][threadIdx.x >> 6] = rmax;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double mm = red[0][0], rm = red[1][0];
            for (int w = 1; w < NT / 64; ++w) {
                mm = fmax(mm, red[0][w]);
                rm = fmax(rm, red[1][w]);
            }
            const unsigned b = by * gridDim.x + 2 * bx + comp;
            norms[2 * b] = mm;
            norms[2 * b + 1] = rm;
        }
    }
}

// ---------------------------------------------------------------------------------
// coarse levels in one workgroup
// ---------------------------------------------------------------------------------
// The coarse part of the V-cycle is a chain of some fifty dependent steps, bound by the length
// of each: an LDS round trip, seven FP64 operations and a barrier. So a thread owns at most two
// points of each colour of a level and knows their LDS addresses; its neighbours' reads are in
// flight together; rhs and 1/c0 sit in registers during a level's sweeps; and the levels of at
// most 64 points of a colour run on wavefront 0 alone, without barriers (LDS operations of one
// wavefront execute in order, so a fence for the compiler is enough).
// LDS of a level: phi and sc (acf, from the residual on the residual) with the colours apart,
// [(i + j) & 1][y][x >> 1] over the box and one ghost ring; ci and r (1/c0, rhs) by owner,
// [colour][thread]. The top level's ci, r and acf stay in registers. Below it, sc and ci depend
// only on acf: a solve's first V-cycle averages acf down and leaves a copy of these arrays
// (blob) in global memory for the later ones, which load it during the top level's sweeps. The
// levels' geometry is computed, not read: loads from the argument block would be one more
// round trip per level.
constexpr int FT = 1024;                        // threads of the kernel
constexpr int FKP = 2;                          // points of a colour per thread, top level
constexpr int FNB = 4;                          // blob values per thread in flight
constexpr size_t FLDS_MAX = 150 * 1024;

// A level's box starts at point 0; its valid points at V = 0 (cell-centred) or 1.
template <bool CC>
struct FLev {
    static constexpr int V = CC ? 0 : 1;
    int nvx, nvy;            // valid points
    int hw, np;              // points of one colour: hw per row, np in all
    int nt;                  // threads that own points (whole wavefronts)
    int pitch, plane;        // doubles per row and per colour
    int sc, ci, bend;        // LDS offsets: the part kept in the blob, from 0
    int phi, r, pend;        // the rest, from the blob's size
    double facx, facy;
    // the level below arrays that end at b and p (the top level has phi alone)
    __host__ __device__ __forceinline__ FLev(int nvx_, int nvy_, double fx, double fy, int b, int p, bool top)
        : nvx(nvx_), nvy(nvy_), facx(fx), facy(fy) {
        hw = (nvx + 1) / 2;
        np = hw * nvy;
        nt = np >= FT ? FT : (np + 63) & ~63;
        pitch = (nvx + 2 * V + 3) / 2;
        plane = pitch * (nvy + 2 * V + 2);
        sc = b;
        ci = sc + 2 * plane;
        bend = top ? b : ci + 2 * nt;
        phi = p;
        r = phi + 2 * plane;
        pend = top ? r : r + 2 * nt;
    }
    // the next coarser level, and the next finer one; spacings double exactly
    __host__ __device__ __forceinline__ FLev coarser() const {
        return FLev(CC ? nvx / 2 : (nvx - 1) / 2, CC ? nvy / 2 : (nvy - 1) / 2, 0.25 * facx, 0.25 * facy, bend, pend,
                    false);
    }
    __device__ __forceinline__ FLev finer() const {
        FLev f(CC ? 2 * nvx : 2 * nvx + 1, CC ? 2 * nvy : 2 * nvy + 1, 4.0 * facx, 4.0 * facy, 0, 0, false);
        const int b = sc - f.bend, p = phi - f.pend;
        f.sc += b; f.ci += b; f.bend += b;
        f.phi += p; f.r += p; f.pend += p;
        return f;
    }
};
struct FArgs {
    int nlev, nblock;    // levels [0, nblock) run on the whole workgroup
    int bottom_sweeps;
    int first;           // a solve's first V-cycle
    int nblob;           // doubles of the blob
    int tsc;             // LDS offset of the top level's sc
    int gcs, ldx;        // level cb in global memory
    int nvx, nvy;
    double facx, facy;
    const double *acf, *res;
    double *c0i, *cor, *gblob;
};

// the points of a level that a thread owns: valid point (2 h + b, row) has colour
// (b + row) & 1, so b = row & 1 for colour 0. at = (box row + 1) pitch + h addresses the
// colour planes: node-centred, both colours' points lie at at + 1 and their west neighbours at
// at + b; cell-centred, the points at at + b and the west neighbours at at.
template <bool CC, int KP>
struct Own {
    static constexpr int V = CC ? 0 : 1;
    int h[KP], row[KP], at[KP];
    bool v[2][KP];
    bool any;   // this wavefront owns points
    __device__ __forceinline__ Own(const FLev<CC>& L) {
        any = __builtin_amdgcn_readfirstlane(int(threadIdx.x)) < L.nt;
        const float rhw = __frcp_rn(float(L.hw));   // e / hw for e < FKP * FT: see row
#pragma unroll
        for (int q = 0; q < KP; ++q) {
            const int e0 = int(threadIdx.x) + q * L.nt, e = min(e0, L.np - 1);
            // (e + 1/2) / hw is 1 / (2 hw) or more from an integer, its error below 1e-3 / hw
            row[q] = int((float(e) + 0.5f) * rhw);
            h[q] = e - row[q] * L.hw;
            at[q] = (row[q] + 1 + V) * L.pitch + h[q];
            v[0][q] = e0 < L.np && 2 * h[q] + (row[q] & 1) < L.nvx;
            v[1][q] = e0 < L.np && 2 * h[q] + 1 - (row[q] & 1) < L.nvx;
        }
    }
    __device__ __forceinline__ int b(int par, int q) const { return (par + row[q]) & 1; }
    __device__ __forceinline__ int ks(int par, int q) const { return CC ? at[q] + b(par, q) : at[q] + 1; }
    __device__ __forceinline__ int kw(int par, int q) const { return CC ? at[q] : at[q] + b(par, q); }
    // coordinates, inside the box also for a point that is not valid
    __device__ __forceinline__ int i(const FLev<CC>& L, int par, int q) const {
        return V + min(2 * h[q] + b(par, q), L.nvx - 1);
    }
    __device__ __forceinline__ int j(int q) const { return V + row[q]; }
};

// the cell-centred box for the functions that look at its edges
template <bool CC>
struct FBox {
    int ilo, ihi, jlo, jhi;
    double facx, facy;
    __device__ __forceinline__ FBox(const FLev<CC>& L)
        : ilo(0), ihi(L.nvx - 1), jlo(0), jhi(L.nvy - 1), facx(L.facx), facy(L.facy) {}
};

template <bool WAVE>
__device__ __forceinline__ void f_sync() {
    if (WAVE) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    } else {
        lds_barrier();
    }
}

// one sweep of colour PAR
template <bool CC, int KP, bool WAVE, int PAR>
__device__ __forceinline__ void f_sweep(double* phi, const FLev<CC>& L, const Own<CC, KP>& o, const double (&r)[2][KP],
                                        const double (&ci)[2][KP]) {
    if (o.any) {
        double w[KP], e[KP], b[KP], t[KP], u[KP];
        const double* const pn = phi + (1 - PAR) * L.plane;
#pragma unroll
        for (int q = 0; q < KP; ++q) {
            const int ks = o.ks(PAR, q), kw = o.kw(PAR, q);
            w[q] = pn[kw];
            e[q] = pn[kw + 1];
            b[q] = pn[ks - L.pitch];
            t[q] = pn[ks + L.pitch];
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int q = 0; q < KP; ++q) {
            if (CC) {
                u[q] = gs_edge(FBox<CC>(L), o.i(L, PAR, q), o.j(q), w[q], e[q], b[q], t[q], r[PAR][q], ci[PAR][q]);
            } else {
                double l = L.facx * (w[q] + e[q]);
                l += L.facy * (b[q] + t[q]);
                u[q] = (r[PAR][q] - l) * ci[PAR][q];
            }
            asm volatile("" : "+v"(u[q]));
        }
#pragma unroll
        for (int q = 0; q < KP; ++q)
            if (o.v[PAR][q]) phi[PAR * L.plane + o.ks(PAR, q)] = u[q];
    }
    f_sync<WAVE>();
}

// n sweeps, n even; ZERO: from phi = 0, whose neighbour sums are zero. The loop has one copy
// of each colour's sweep: the kernel runs through its code once, and fetching it counts.
template <bool CC, int KP, bool WAVE, bool ZERO>
__device__ __forceinline__ void f_sweeps(double* w, const FLev<CC>& L, const Own<CC, KP>& o, const double (&r)[2][KP],
                                         const double (&ci)[2][KP], int n) {
    double* const phi = w + L.phi;
    if (ZERO) {
#pragma unroll
        for (int q = 0; q < KP; ++q)
            if (o.v[0][q]) phi[o.ks(0, q)] = r[0][q] * ci[0][q];
        f_sync<WAVE>();
    } else {
        f_sweep<CC, KP, WAVE, 0>(phi, L, o, r, ci);
    }
#pragma unroll 1
    for (;;) {
        f_sweep<CC, KP, WAVE, 1>(phi, L, o, r, ci);
        if ((n -= 2) <= 0) break;
        f_sweep<CC, KP, WAVE, 0>(phi, L, o, r, ci);
    }
}

// sc = residual; acf comes from sc, or from registers (REG)
template <bool CC, int KP, bool WAVE, bool REG>
__device__ __forceinline__ void f_residual(double* w, const FLev<CC>& L, int sc, const Own<CC, KP>& o,
                                           const double (&r)[2][KP], double (&a)[2][KP]) {
    if (o.any) {
        double z[2][KP], x0[2][KP], x1[2][KP], y0[2][KP], y1[2][KP], g[2][KP];
#pragma unroll
        for (int par = 0; par < 2; ++par) {
            const double* const p = w + L.phi + par * L.plane;
            const double* const pn = w + L.phi + (1 - par) * L.plane;
#pragma unroll
            for (int q = 0; q < KP; ++q) {
                const int ks = o.ks(par, q), kw = o.kw(par, q);
                z[par][q] = p[ks];
                x0[par][q] = pn[kw];
                x1[par][q] = pn[kw + 1];
                y0[par][q] = pn[ks - L.pitch];
                y1[par][q] = pn[ks + L.pitch];
                if (!REG) a[par][q] = w[sc + par * L.plane + ks];
            }
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int par = 0; par < 2; ++par)
#pragma unroll
            for (int q = 0; q < KP; ++q) {
                auto P = [&](int di, int dj) {
                    return di < 0   ? x0[par][q]
                           : di > 0 ? x1[par][q]
                           : dj < 0 ? y0[par][q]
                           : dj > 0 ? y1[par][q]
                                    : z[par][q];
                };
                g[par][q] =
                    residual1<CC>(FBox<CC>(L), o.i(L, par, q), o.j(q), P, r[par][q], a[par][q], L.facx, L.facy);
                asm volatile("" : "+v"(g[par][q]));
            }
#pragma unroll
        for (int par = 0; par < 2; ++par)
#pragma unroll
            for (int q = 0; q < KP; ++q)
                if (o.v[par][q]) w[sc + par * L.plane + o.ks(par, q)] = g[par][q];
    }
    f_sync<WAVE>();
}

// sc of level F restricted to point (i, j) of the next level: the fine centre (2 i, 2 j) and
// its diagonal neighbours have colour 0, the others colour 1
template <bool CC>
__device__ __forceinline__ double f_restrict(const double* w, const FLev<CC>& F, int sc, int i, int j) {
    const int P = F.pitch;
    const double* const p0 = w + sc + (2 * j + 1) * P + i;
    const double* const p1 = p0 + F.plane;
    double f[9] = {};
    f[4] = p0[0];
    f[5] = p1[1];
    f[7] = p1[P];
    f[8] = p0[P + 1];
    if (!CC) {
        f[0] = p0[-P];
        f[1] = p1[-P];
        f[2] = p0[1 - P];
        f[3] = p1[0];
        f[6] = p0[P];
    }
    asm volatile("" ::: "memory");
    auto A = [&](int a, int b) { return f[(b - 2 * j + 1) * 3 + (a - 2 * i) + 1]; };
    return restrict_from<CC>(A, i, j);
}

// phi of level L += I(phi of level C)
template <bool CC, int KP, bool WAVE>
__device__ __forceinline__ void f_interp(double* w, const FLev<CC>& L, const FLev<CC>& C, const Own<CC, KP>& o) {
    if (o.any) {
#pragma unroll
        for (int par = 0; par < 2; ++par) {
            double c[4][KP], x[KP];
#pragma unroll
            for (int q = 0; q < KP; ++q) {
                // node-centred: point (1 + 2 h + b, 1 + row) lies at or right after coarse (h + b,
                // (row + 1) / 2); both odd or both even (colour 0), or odd along one direction
                const int ic = CC ? o.h[q] : o.h[q] + o.b(par, q), jc = CC ? o.row[q] >> 1 : (o.row[q] + 1) >> 1;
                const int pc = ((ic + jc) & 1) * C.plane, pd = C.plane - pc;
                const double* const p = w + C.phi + (jc + 1) * C.pitch + ((ic + 1) >> 1);
                const int e = 1 - (ic & 1);   // to the east neighbour's place in its row
                c[0][q] = p[pc];
                if (!CC && par == 0) {
                    c[1][q] = p[pd + e];
                    c[2][q] = p[pd + C.pitch];
                    c[3][q] = p[pc + C.pitch + e];
                }
                if (!CC && par == 1) c[1][q] = p[pd + ((o.row[q] & 1) ? e : C.pitch)];
                x[q] = w[L.phi + par * L.plane + o.ks(par, q)];
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int q = 0; q < KP; ++q) {
                if (CC) {
                    x[q] += c[0][q];
                } else if (par == 1) {
                    x[q] += (c[0][q] + c[1][q]) * 0.5;
                } else {
                    const double four = (c[0][q] + c[1][q] + c[2][q] + c[3][q]) * 0.25;
                    x[q] += (o.row[q] & 1) ? c[0][q] : four;
                }
                asm volatile("" : "+v"(x[q]));
            }
#pragma unroll
            for (int q = 0; q < KP; ++q)
                if (o.v[par][q]) w[L.phi + par * L.plane + o.ks(par, q)] = x[q];
        }
    }
    f_sync<WAVE>();
}

// level L below the top, fine level F with its residual at sc: rhs from that, sweeps from
// zero; then, on all but the bottom level, the residual
template <bool CC, bool WAVE>
__device__ __forceinline__ void f_down(double* w, const FLev<CC>& F, int sc, const FLev<CC>& L, int sweeps,
                                       bool bottom) {
    const Own<CC, 1> o(L);
    double r[2][1] = {}, ci[2][1] = {}, a[2][1];
    if (o.any) {
#pragma unroll
        for (int par = 0; par < 2; ++par) {
            const int slot = par * L.nt + int(threadIdx.x);
            ci[par][0] = w[L.ci + slot];
            r[par][0] = f_restrict<CC>(w, F, sc, o.i(L, par, 0), o.j(0));
            w[L.r + slot] = r[par][0];
        }
    }
    f_sweeps<CC, 1, WAVE, true>(w, L, o, r, ci, sweeps);
    if (!bottom) f_residual<CC, 1, WAVE, false>(w, L, L.sc, o, r, a);
}

template <bool CC, bool WAVE>
__device__ __forceinline__ void f_up(double* w, const FLev<CC>& L, const FLev<CC>& C) {
    const Own<CC, 1> o(L);
    double r[2][1] = {}, ci[2][1] = {};
    if (o.any) {
#pragma unroll
        for (int par = 0; par < 2; ++par) {
            const int slot = par * L.nt + int(threadIdx.x);
            ci[par][0] = w[L.ci + slot];
            r[par][0] = w[L.r + slot];
        }
    }
    f_interp<CC, 1, WAVE>(w, L, C, o);
    f_sweeps<CC, 1, WAVE, false>(w, L, o, r, ci, 4);
}

// x of the lane OFF lanes away within a row of 16 lanes, zero beyond it
template <int OFF>
__device__ __forceinline__ double row_lane(double x) {
    constexpr int ctrl = OFF < 0 ? 0x110 - OFF : 0x100 + OFF;   // row_shr, row_shl
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), ctrl, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), ctrl, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// The bottom level of at most 3 x 3 valid points (all grids of 2^k - 1 points), node-centred, in
// registers: point (col, row) on lane 4 row + col, whose neighbours are 1 and 4 lanes away and
// whose border lanes hold zero. A sweep is 8 lane moves and 7 FP64 operations, 90 cycles instead
// of 290 through LDS.
__device__ __forceinline__ void f_bottom3(double* w, const FLev<false>& F, int sc, const FLev<false>& L, int sweeps) {
    const int lane = int(threadIdx.x), col = lane & 3, row = lane >> 2;
    const bool own = col < L.nvx && row < L.nvy;
    const int par = (col + row) & 1, c = min(col, L.nvx - 1), d = min(row, L.nvy - 1);
    const double ci = w[L.ci + ((c + d) & 1) * L.nt + d * L.hw + (c >> 1)];
    const double r = f_restrict<false>(w, F, sc, 1 + c, 1 + d);
    double x = 0.0;
#pragma unroll 1
    for (int k = 0; k < sweeps; ++k) {
        double l = L.facx * (row_lane<-1>(x) + row_lane<1>(x));
        l += L.facy * (row_lane<-4>(x) + row_lane<4>(x));
        const double u = (r - l) * ci;
        x = own && par == (k & 1) ? u : x;
    }
    if (own) w[L.phi + par * L.plane + (row + 2) * L.pitch + (col >> 1) + 1] = x;
    f_sync<true>();
}

// acf of level L from level F, whose acf is at sc, and its 1/c0 (average_down_acoef, :1641-1661)
template <bool CC>
__device__ __forceinline__ void f_average(double* w, const FLev<CC>& F, int sc, const FLev<CC>& L) {
    const Own<CC, 1> o(L);
    if (o.any) {
#pragma unroll
        for (int par = 0; par < 2; ++par) {
            const int i = o.i(L, par, 0);
            const double a = f_restrict<CC>(w, F, sc, i, o.j(0));
            w[L.ci + par * L.nt + int(threadIdx.x)] = c0_inverse<CC>(FBox<CC>(L), i, o.j(0), a, L.facx, L.facy);
            if (o.v[par][0]) w[L.sc + par * L.plane + o.ks(par, 0)] = a;
        }
    }
    __syncthreads();
}

// Levels [cb, maxl] of one V-cycle for component blockIdx.x: down-sweep with residual
// restriction, bottom solve (CPU branch of MultiGrid::bottomsolve, :1583-1593), up-sweep.
// KP: points of one colour per thread on level cb. acf and rhs of level cb come from global
// memory, its correction goes back there.
// Measured: 17.5 us from 65 x 65 points down (node-centred), 21.5 us from 64 x 64 (cell-centred).
// Before, with the arrays in LDS alone and 512 threads, 23.5 us from 33 x 33 and 36 us from
// 32 x 32 points, and two more launches of 8.7 us for the level above. Loading its 150 KB takes
// 3 us; a level's step costs 300 cycles a sweep on the small levels and 780, the LDS bandwidth,
// on the top one.
template <bool CC, int KP>
__global__ __launch_bounds__(FT) void k_coarse_lds(const FArgs A, const MGCtl* __restrict__ ctl) {
    extern __shared__ double w[];
    const int comp = blockIdx.x, nl = A.nlev, nb = A.nblock;
    const FLev<CC> T(A.nvx, A.nvy, A.facx, A.facy, 0, A.nblob, true);
    const int done = ctl->done;
    const Own<CC, KP> o(T);
    double r[2][KP], ci[2][KP], a[2][KP], bl[FNB];
    int k[2][KP];
    const double* const gres = A.res + long(comp) * A.gcs;
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
        for (int q = 0; q < KP; ++q) {
            k[par][q] = (o.j(q) + 1) * A.ldx + o.i(T, par, q) + 1;
            r[par][q] = gres[k[par][q]];
            ci[par][q] = A.first ? A.acf[k[par][q]] : A.c0i[k[par][q]];
        }
    // what the sweeps do not need comes in during them
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
        for (int q = 0; q < KP; ++q) a[par][q] = A.acf[k[par][q]];
    if (!A.first && nl > 1) {
#pragma unroll
        for (int q = 0; q < FNB; ++q) bl[q] = A.gblob[min(q * FT + int(threadIdx.x), A.nblob - 1)];
    }
    if (done) return;
    for (int t = 2 * int(threadIdx.x); t < A.tsc - A.nblob; t += 2 * FT)
        *reinterpret_cast<double2*>(w + A.nblob + t) = make_double2(0.0, 0.0);
    if (A.first) {
#pragma unroll
        for (int par = 0; par < 2; ++par)
#pragma unroll
            for (int q = 0; q < KP; ++q) {
                ci[par][q] = c0_inverse<CC>(FBox<CC>(T), o.i(T, par, q), o.j(q), ci[par][q], T.facx, T.facy);
                if (comp == 0 && o.v[par][q]) A.c0i[k[par][q]] = ci[par][q];
                if (o.v[par][q]) w[A.tsc + par * T.plane + o.ks(par, q)] = a[par][q];
            }
        for (int t = threadIdx.x; t < A.nblob; t += FT) w[t] = 0.0;
        __syncthreads();
        FLev<CC> F = T;
        for (int l = 1, sc = A.tsc; l < nl; ++l) {
            const FLev<CC> L = F.coarser();
            f_average<CC>(w, F, sc, L);
            F = L;
            sc = L.sc;
        }
        if (comp == 0)
            for (int t = threadIdx.x; t < A.nblob; t += FT) A.gblob[t] = w[t];
    }
    lds_barrier();
    f_sweeps<CC, KP, false, true>(w, T, o, r, ci, nl == 1 ? A.bottom_sweeps : 4);
    if (nl > 1) {
        if (!A.first) {
#pragma unroll
            for (int q = 0; q < FNB; ++q) w[min(q * FT + int(threadIdx.x), A.nblob - 1)] = bl[q];
            for (int t = FNB * FT + int(threadIdx.x); t < A.nblob; t += FT) w[t] = A.gblob[t];
        }
        f_residual<CC, KP, false, true>(w, T, A.tsc, o, r, a);
        FLev<CC> F = T;
        int sc = A.tsc;
        for (int l = 1; l < nb; ++l) {
            const FLev<CC> L = F.coarser();
            f_down<CC, false>(w, F, sc, L, l == nl - 1 ? A.bottom_sweeps : 4, l == nl - 1);
            F = L;
            sc = L.sc;
        }
        if (__builtin_amdgcn_readfirstlane(int(threadIdx.x)) < 64) {
            for (int l = nb; l < nl; ++l) {
                const FLev<CC> L = F.coarser();
                const bool bottom = l == nl - 1;
                if constexpr (!CC) {
                    if (bottom && L.nvx <= 3 && L.nvy <= 3) {
                        f_bottom3(w, F, sc, L, A.bottom_sweeps);
                        F = L;
                        break;
                    }
                }
                f_down<CC, true>(w, F, sc, L, bottom ? A.bottom_sweeps : 4, bottom);
                F = L;
                sc = L.sc;
            }
            for (int l = nl - 2; l >= nb; --l) {
                const FLev<CC> L = F.finer();
                f_up<CC, true>(w, L, F);
                F = L;
            }
        } else if (nb < nl) {
            F = F.coarser();
        }
        lds_barrier();
        for (int l = min(nb, nl - 1) - 1; l >= 1; --l) {
            const FLev<CC> L = F.finer();
            f_up<CC, false>(w, L, F);
            F = L;
        }
        f_interp<CC, KP, false>(w, T, F, o);
        f_sweeps<CC, KP, false, false>(w, T, o, r, ci, 4);
    }
    double* const gcor = A.cor + long(comp) * A.gcs;
#pragma unroll
    for (int par = 0; par < 2; ++par)
#pragma unroll
        for (int q = 0; q < KP; ++q)
            if (o.v[par][q]) gcor[k[par][q]] = w[T.phi + par * T.plane + o.ks(par, q)];
}

// Bottom solve of a bottom level that is too large for k_coarse_lds (a grid that hardly
// coarsens): the same sweeps on the level's global arrays, one workgroup per component.
template <bool CC>
__global__ __launch_bounds__(FT) void k_bottom(MGLevel L, int sweeps, const MGCtl* __restrict__ ctl) {
    if (ctl->done) return;
    const long ck = blockIdx.x ? L.cs : 0;
    double* const phi = L.cor + ck;
    const int hw = (L.vihi - L.vilo + 2) / 2, np = hw * (L.vjhi - L.vjlo + 1);
    for (int sw = 0; sw < sweeps; ++sw) {
        for (int e = threadIdx.x; e < np; e += FT) {
            const int j = L.vjlo + e / hw, i = L.vilo + 2 * (e % hw) + ((sw + L.vilo + j) & 1);
            if (i > L.vihi) continue;
            const long k = at(L, i, j);
            const double ci = c0_inverse<CC>(L, i, j, L.acf[k], L.facx, L.facy);
            const double rhs = L.res[k + ck];
            auto P = [&](int a, int b) { return sw == 0 ? 0.0 : phi[k + b * L.ldx + a]; };
            phi[k] = gs_point<CC>(L, i, j, P, rhs, ci, L.facx, L.facy);
        }
        // the other colour starts from zero as well
        if (sw == 0)
            for (int e = threadIdx.x; e < np; e += FT) {
                const int j = L.vjlo + e / hw, i = L.vilo + 2 * (e % hw) + ((1 + L.vilo + j) & 1);
                if (i <= L.vihi) phi[at(L, i, j)] = 0.0;
            }
        __syncthreads();
    }
}

// level-0 load (copy path): acf, sol and rhs (2 comps) over the whole box
__global__ void k_mg_load(MGLevel L, int sh, Geom g, const double* __restrict__ sol, const double* __restrict__ rhs,
                          const double* __restrict__ acf, long cstride, double* __restrict__ acf0,
                          double* __restrict__ msol, double* __restrict__ mrhs) {
    const int nbx = L.ihi - L.ilo + 1, nby = L.jhi - L.jlo + 1;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nbx * nby) return;
    const int j = L.jlo + t / nbx, i = L.ilo + t % nbx;
    const long gk = g.idx(i - sh, j - sh);
    const long k = at(L, i, j);
    acf0[k] = acf[gk];
    msol[k] = sol[gk];
    msol[k + L.cs] = sol[gk + cstride];
    mrhs[k] = rhs[gk];
    mrhs[k + L.cs] = rhs[gk + cstride];
}

// sol (valid points) = src, the level-0 iterate
__global__ void k_mg_store(MGLevel L, int sh, Geom g, double* __restrict__ sol, long cstride,
                           const double* __restrict__ src) {
    const int nvx = L.vihi - L.vilo + 1, nvy = L.vjhi - L.vjlo + 1;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nvx * nvy) return;
    const int j = L.vjlo + t / nvx, i = L.vilo + t % nvx;
    const long gk = g.idx(i - sh, j - sh);
    const long k = at(L, i, j);
    sol[gk] = src[k];
    sol[gk + cstride] = src[k + L.cs];
}

// initial guess of the next solve: b = 2 b - h and h = old b (EXTRAP), or h = b (record only)
template <bool EXTRAP>
__global__ void k_guess_linear(double* __restrict__ b, double* __restrict__ h, long n) {
    const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const double b1 = b[t];
    if (EXTRAP) b[t] = 2.0 * b1 - h[t];
    h[t] = b1;
}

bool coarsenable(bool cc, int lo, int hi, int min_width) {
    const int size = hi - lo + 1;
    if (size < 2 * min_width) return false;
    if (cc) return (cdiv2(lo) * 2 == lo) && (cdiv2(hi) * 2 + 1 == hi);
    return (cdiv2(lo) * 2 == lo) && (cdiv2(hi) * 2 == hi);
}

int bottom_sweeps(const MGLevel& B) {
    const int len = std::max(B.ihi - B.ilo + 1, B.jhi - B.jlo + 1);
    return std::max(16, (len + 1) / 2 * 2);
}

// the description of levels cb..max_level for k_coarse_lds, or false where they do not fit: a
// thread would own more than FKP points of a colour, or the arrays exceed the LDS
template <bool CC>
bool coarse_lds_args(MultiGrid& M, int cb) {
    const MGLevel& G = M.lev[cb];
    FArgs A{};
    A.nlev = M.max_level - cb + 1;
    A.nvx = G.vihi - G.vilo + 1;
    A.nvy = G.vjhi - G.vjlo + 1;
    if (A.nvx > 2 * FKP * FT || A.nvy > FKP * FT) return false;
    A.facx = G.facx;
    A.facy = G.facy;
    const FLev<CC> T(A.nvx, A.nvy, G.facx, G.facy, 0, 0, true);
    FLev<CC> L = T;
    for (int l = 0; l < A.nlev; ++l) {
        if (l) L = L.coarser();
        if (L.np > L.nt * (l == 0 ? FKP : 1)) return false;
        if (l == 0 || L.nt > 64) A.nblock = l + 1;
    }
    A.nblob = (L.bend + 1) & ~1;
    A.tsc = (A.nblob + L.pend + 1) & ~1;
    M.coarse_lds_bytes = sizeof(double) * size_t(A.tsc + 2 * T.plane);
    if (M.coarse_lds_bytes > FLDS_MAX) return false;
    M.coarse_kp = T.np <= FT ? 1 : 2;
    A.bottom_sweeps = bottom_sweeps(M.lev[M.max_level]);
    A.gcs = int(G.cs);
    A.ldx = G.ldx;
    A.acf = G.acf;
    A.res = G.res;
    A.c0i = G.c0i;
    A.cor = G.cor;
    std::memcpy(M.coarse_args, &A, sizeof(A));
    return true;
}

}  // namespace

void mg_init(hpq_ctx* c) {
    static_assert(sizeof(FArgs) <= sizeof(MultiGrid::coarse_args), "coarse argument block too small");
    MultiGrid& M = c->mg;
    const int nx = c->g.nx, ny = c->g.ny;
    if (nx % 2 != ny % 2) throw HpqError(HPQ_E_UNSUPPORTED, "hpmg: nx and ny must have the same parity");
    M.cc = (nx % 2 == 0);
    M.dx = c->g.dx;
    M.dy = c->g.dy;
    MGLevel l0;
    l0.cc = M.cc;
    l0.ilo = 0; l0.jlo = 0;
    l0.ihi = M.cc ? nx - 1 : nx + 1;
    l0.jhi = M.cc ? ny - 1 : ny + 1;
    M.lev.clear();
    M.lev.push_back(l0);
    const int mw = M.cc ? 2 : 4;
    for (int i = 0; i < 30; ++i) {
        const MGLevel& b = M.lev.back();
        if (coarsenable(M.cc, b.ilo, b.ihi, mw) && coarsenable(M.cc, b.jlo, b.jhi, mw)) {
            MGLevel n;
            n.cc = M.cc;
            n.ilo = b.ilo / 2; n.jlo = b.jlo / 2; n.ihi = b.ihi / 2; n.jhi = b.jhi / 2;
            M.lev.push_back(n);
        } else {
            break;
        }
    }
    M.max_level = int(M.lev.size()) - 1;
    if (M.max_level < 1)
        throw HpqError(HPQ_E_UNSUPPORTED, "hpmg: the slice cannot be coarsened at least once");
    for (int l = 0; l <= M.max_level; ++l) {
        MGLevel& L = M.lev[l];
        if (M.cc) { L.vilo = L.ilo; L.vihi = L.ihi; L.vjlo = L.jlo; L.vjhi = L.jhi; }
        else { L.vilo = L.ilo + 1; L.vihi = L.ihi - 1; L.vjlo = L.jlo + 1; L.vjhi = L.jhi - 1; }
        L.ldx = (L.ihi - L.ilo + 1) + 2;
        L.ldy = (L.jhi - L.jlo + 1) + 2;
        L.cs = long(L.ldx) * L.ldy;
        L.dx = M.dx * double(1 << l);
        L.dy = M.dy * double(1 << l);
        L.facx = 1. / (L.dx * L.dx);
        L.facy = 1. / (L.dy * L.dy);
        const size_t b1 = sizeof(double) * L.cs;
        HPQ_HIP(hipMalloc(&L.acf, b1));
        HPQ_HIP(hipMalloc(&L.c0i, b1));
        HPQ_HIP(hipMalloc(&L.res, 2 * b1));
        HPQ_HIP(hipMalloc(&L.cor, 2 * b1));
        HPQ_HIP(hipMalloc(&L.rescor, 2 * b1));
        HPQ_HIP(hipMemset(L.acf, 0, b1));
        HPQ_HIP(hipMemset(L.res, 0, 2 * b1));
        HPQ_HIP(hipMemset(L.cor, 0, 2 * b1));
        HPQ_HIP(hipMemset(L.rescor, 0, 2 * b1));
    }
    // from the first level that k_coarse_lds can take, or the bottom level alone from global memory
    M.coarse_begin = M.max_level;
    M.coarse_in_lds = false;
    for (int l = 1; l <= M.max_level && !M.coarse_in_lds; ++l) {
        M.coarse_in_lds = M.cc ? coarse_lds_args<true>(M, l) : coarse_lds_args<false>(M, l);
        if (M.coarse_in_lds) M.coarse_begin = l;
    }
    if (M.coarse_in_lds) {
        FArgs& A = *reinterpret_cast<FArgs*>(M.coarse_args);
        HPQ_HIP(hipMalloc(&M.coarse_work, sizeof(double) * size_t(std::max(1, A.nblob))));
        A.gblob = M.coarse_work;
    }
    const size_t b0 = sizeof(double) * 2 * M.lev[0].cs;
    HPQ_HIP(hipMalloc(&M.msol, b0));
    HPQ_HIP(hipMalloc(&M.mrhs, b0));
    HPQ_HIP(hipMemset(M.msol, 0, b0));
    HPQ_HIP(hipMemset(M.mrhs, 0, b0));
    HPQ_HIP(hipMalloc(&M.d_ctl, 2 * sizeof(MGCtl)));
    HPQ_HIP(hipMemset(M.d_ctl, 0, 2 * sizeof(MGCtl)));
    {
        const MGLevel& L0 = M.lev[0];
        // the tiles of level-0 launches have 8 x 4 points or more, for each component
        const long nblk = 2 * long((L0.vihi - L0.vilo + 8) / 8) * ((L0.vjhi - L0.vjlo + 4) / 4);
        HPQ_HIP(hipMalloc(&M.d_norms, sizeof(double) * 2 * nblk));
    }
    HPQ_HIP(hipHostMalloc(&M.h_mirror, sizeof(MGMirror), hipHostMallocMapped | hipHostMallocCoherent));
    M.h_mirror->word = 0;
    HPQ_HIP(hipHostGetDevicePointer((void**)&M.d_mirror, M.h_mirror, 0));
    if (M.coarse_in_lds) {
        const void* fs[2][2] = {{(const void*)k_coarse_lds<false, 1>, (const void*)k_coarse_lds<false, 2>},
                                {(const void*)k_coarse_lds<true, 1>, (const void*)k_coarse_lds<true, 2>}};
        HPQ_HIP(hipFuncSetAttribute(fs[M.cc][M.coarse_kp - 1], hipFuncAttributeMaxDynamicSharedMemorySize,
                                    int(M.coarse_lds_bytes)));
    }
}

void mg_guess_linear(hpq_ctx* c, double* bxby, int islice) {
    MultiGrid& M = c->mg;
    const long n = 2 * c->g.plane;
    if (!M.hist) HPQ_HIP(hipMalloc(&M.hist, sizeof(double) * n));
    const dim3 grid(unsigned((n + 255) / 256));
    if (M.hist_slice == islice + 2)
        hipLaunchKernelGGL(k_guess_linear<true>, grid, dim3(256), 0, c->stream, bxby, M.hist, n);
    else
        hipLaunchKernelGGL(k_guess_linear<false>, grid, dim3(256), 0, c->stream, bxby, M.hist, n);
    HPQ_HIP(hipGetLastError());
    M.hist_slice = islice + 1;
}

void mg_free(hpq_ctx* c) {
    MultiGrid& M = c->mg;
    if (M.hist) (void)hipFree(M.hist);
    for (auto& L : M.lev)
        for (void* p : {(void*)L.acf, (void*)L.c0i, (void*)L.res, (void*)L.cor, (void*)L.rescor})
            if (p) (void)hipFree(p);
    if (M.coarse_work) (void)hipFree(M.coarse_work);
    if (M.msol) (void)hipFree(M.msol);
    if (M.mrhs) (void)hipFree(M.mrhs);
    if (M.d_ctl) (void)hipFree(M.d_ctl);
    if (M.d_norms) (void)hipFree(M.d_norms);
    if (M.h_mirror) (void)hipHostFree(M.h_mirror);
    M = MultiGrid{};
}

namespace {

// the caller's view of one solve: level-0 rhs, acf and the two iterate buffers
struct Solve {
    const double* rhs0;   // comp stride rcs
    long rcs;
    MGLevel L0;           // level 0 with acf pointing at the level-0 acf
    double* buf[2];       // iterate after an even / odd number of V-cycles
    MGCtl* ctl;
    MGCtl* other;
    double tol_rel, tol_abs;
    int nblk;             // workgroups of the last level-0 launch (entries of d_norms)
};

template <int NSW, bool CC, bool RES, int KP>
dim3 smooth_grid(const MGLevel& L) {
    using T = Tile<NSW, CC, RES, KP>;
    return dim3(2 * ((L.vihi - L.vilo + T::TX) / T::TX), (L.vjhi - L.vjlo + T::TY) / T::TY);
}

// Returns the number of workgroups (entries of norms).
template <int NSW, bool ZERO, bool RES, bool INTERP, bool RHSMAX = false, bool NORMS = false, bool FIRST = false>
int smooth(hpq_ctx* c, const MGLevel& L, const MGLevel& C, double* phi_out, const double* rhs, long rcs,
           const double* acf, const double* phi_in, const double* cor_c, double* res_c, const MGCtl* gate,
           double* norms = nullptr, const Fold& fold = Fold{}) {
    TraceScope ts(c, HPQ_TRACE_MG_SMOOTH);
    auto launch = [&](auto CCC, auto KPC) {
        constexpr bool CC = decltype(CCC)::value;
        constexpr int KP = decltype(KPC)::value;
        const dim3 grid = smooth_grid<NSW, CC, RES, KP>(L);
        hipLaunchKernelGGL((k_smooth<NSW, CC, ZERO, RES, INTERP, RHSMAX, NORMS, FIRST, KP>), grid, dim3(NT), 0,
                           c->stream, L, C, phi_out, rhs, rcs, acf, phi_in, cor_c, res_c, gate, norms, fold);
        return int(grid.x * grid.y);
    };
    // The smaller tile while all its workgroups are resident (four to a CU at one point of a
    // colour per thread, two at two): 4.6 against 5.6 us for four sweeps of 127 x 127 points (78
    // or 30 workgroups), 7.8 against 9.5 us for eight of 255 x 255 (228 or 108). Beyond that the
    // larger one, which recomputes less of its surroundings: 9.0 against 16.0 us for four sweeps
    // of 511 x 511 (480 or 1720 workgroups), 14.4 against 18.7 us for eight (432 or 888).
    constexpr int KP = NSW == 8 ? 2 : 1;
    constexpr unsigned resident = 256 * (NSW == 8 ? 2 : 4);
    auto pick = [&](auto CCC) {
        const dim3 g = smooth_grid<NSW, decltype(CCC)::value, RES, KP>(L);
        return g.x * g.y <= resident ? launch(CCC, std::integral_constant<int, KP>{})
                                     : launch(CCC, std::integral_constant<int, KP + 1>{});
    };
    return L.cc ? pick(std::true_type{}) : pick(std::false_type{});
}

// MultiGrid::vcycle (:1430-1512), V-cycle number m of the solve. Level 0's residual and
// its restriction to level 1 come from the end of the previous cycle (or the initial
// residual); every kernel returns at once when the control block says the solve is
// finished. Cycle m runs only if cycles 0..m-1 ran, so the host knows that it starts from
// buf[m & 1] and ends in buf[(m + 1) & 1]. fold: the convergence target (m = 0) or the end
// of cycle m - 1 is evaluated by the cycle's first launch (level 1 down); check: the cycle
// ends with a k_check launch that publishes its result to the host.
void vcycle(hpq_ctx* c, Solve& S, int m, int maxiter, bool fold, bool check) {
    MultiGrid& M = c->mg;
    MGCtl* ctl = S.ctl;
    const int cb = M.coarse_begin;
    for (int l = 1; l < cb; ++l) {
        MGLevel& L = M.lev[l];
        MGLevel& C = M.lev[l + 1];
        Fold f;
        if (fold && l == 1) {
            f.mode = m == 0 ? Fold::TARGET : Fold::CHECK;
            f.m = m;
            f.maxiter = maxiter;
            f.nblk = S.nblk;
            f.tol_rel = S.tol_rel;
            f.tol_abs = S.tol_abs;
            f.norms = M.d_norms;
            f.ctl = ctl;
            f.other = S.other;
        }
        if (m == 0)
            smooth<4, true, true, false, false, false, true>(c, L, C, L.cor, L.res, L.cs, L.acf, nullptr, nullptr,
                                                             C.res, ctl, nullptr, f);
        else
            smooth<4, true, true, false>(c, L, C, L.cor, L.res, L.cs, L.acf, nullptr, nullptr, C.res, ctl, nullptr, f);
    }
    {
        TraceScope ts(c, HPQ_TRACE_MG_COARSE);
        if (M.coarse_in_lds) {
            FArgs& A = *reinterpret_cast<FArgs*>(M.coarse_args);
            A.first = m == 0;
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(2), dim3(FT), M.coarse_lds_bytes, c->stream, A, ctl);
            };
            if (M.cc) M.coarse_kp == 1 ? launch(k_coarse_lds<true, 1>) : launch(k_coarse_lds<true, 2>);
            else M.coarse_kp == 1 ? launch(k_coarse_lds<false, 1>) : launch(k_coarse_lds<false, 2>);
        } else {
            const MGLevel& B = M.lev[cb];
            hipLaunchKernelGGL(M.cc ? k_bottom<true> : k_bottom<false>, dim3(2), dim3(FT), 0, c->stream, B,
                               bottom_sweeps(B), ctl);
        }
    }
    // Up-sweep: the result of level l >= 1 goes to rescor[l] (dead after the restriction),
    // so the kernel never overwrites cor[l], which neighbouring tiles read as their halo.
    // The coarse kernel leaves its top level in cor[cb].
    for (int l = cb - 1; l >= 1; --l) {
        MGLevel& L = M.lev[l];
        MGLevel& C = M.lev[l + 1];
        const double* corc = (l + 1 == cb) ? C.cor : C.rescor;
        smooth<4, false, false, true>(c, L, C, L.rescor, L.res, L.cs, L.acf, L.cor, corc, nullptr, ctl);
    }
    // Level 0: the up-sweep's four sweeps and the cycle's final four sweeps + residual are
    // eight consecutive sweeps from x + I(cor_1), where x is the current iterate; the
    // intermediate after four sweeps is not needed.
    MGLevel& L1 = M.lev[1];
    const double* corc = (cb == 1) ? L1.cor : L1.rescor;
    S.nblk = smooth<8, false, true, true, false, true>(c, S.L0, L1, S.buf[(m + 1) & 1], S.rhs0, S.rcs, S.L0.acf,
                                                       S.buf[m & 1], corc, L1.res, ctl, M.d_norms);
    if (check) {
        const Check chk{ctl, S.other, M.d_mirror, M.d_norms, S.nblk, ++M.seq, maxiter, 0.0, 0.0};
        hipLaunchKernelGGL(k_check, dim3(1), dim3(NT), 0, c->stream, chk);
    }
}

struct Published {
    int seq, iters, status;
    bool done;
};

Published decode(unsigned long long w) {
    return {int(unsigned(w & 0xffffffffull)), int((w >> 32) & 0xffffff), int((w >> 56) & 0x7f), (w >> 63) != 0};
}

// waits until the device has published sequence number seq
Published wait_mirror(hpq_ctx* c, int seq) {
    MultiGrid& M = c->mg;
    unsigned long long* word = &M.h_mirror->word;
    const auto t0 = std::chrono::steady_clock::now();
    for (long spin = 0;; ++spin) {
        const Published p = decode(__atomic_load_n(word, __ATOMIC_ACQUIRE));
        if (p.seq == seq) return p;
        if ((spin & 1023) == 1023 && std::chrono::steady_clock::now() - t0 > std::chrono::seconds(30)) break;
    }
    // the device has not reported: let the stream drain, then look once more
    HPQ_HIP(hipStreamSynchronize(c->stream));
    const Published p = decode(__atomic_load_n(word, __ATOMIC_ACQUIRE));
    if (p.seq != seq) throw HpqError(HPQ_E_HIP, "hpmg: the device did not report convergence");
    return p;
}

}  // namespace

// MultiGrid::solve1 + solve_doit (HpMultiGrid.cpp:1170-1190, 1308-1427)
int mg_solve1(hpq_ctx* c, double* sol, const double* rhs, const double* acf, long cstride, double tol_rel,
              double tol_abs, int maxiter, int* iters) {
    MultiGrid& M = c->mg;
    MGLevel& L1 = M.lev[1];
    if (M.ctl_dirty) {
        HPQ_HIP(hipMemsetAsync(M.d_ctl, 0, 2 * sizeof(MGCtl), c->stream));
        M.ctl_dirty = false;
    }
    Solve S;
    S.ctl = M.d_ctl + M.ctl_pick;
    S.other = M.d_ctl + (M.ctl_pick ^ 1);
    S.L0 = M.lev[0];
    const int sh = M.cc ? 0 : 1;
    // node-centred level 0 (odd n) has the guarded plane's shape: work on the caller's
    // planes directly when the two components are one plane apart
    const bool alias = !M.cc && cstride == S.L0.cs;
    if (alias) {
        S.rhs0 = rhs;
        S.rcs = cstride;
        S.L0.acf = const_cast<double*>(acf);
        S.buf[0] = S.L0.cor;
        S.buf[1] = sol;
    } else {
        const int n = (S.L0.ihi - S.L0.ilo + 1) * (S.L0.jhi - S.L0.jlo + 1);
        hipLaunchKernelGGL(k_mg_load, grid1d(n, 256), dim3(256), 0, c->stream, S.L0, sh, c->g, sol, rhs, acf, cstride,
                           M.lev[0].acf, M.msol, M.mrhs);
        S.rhs0 = M.mrhs;
        S.rcs = S.L0.cs;
        S.buf[0] = S.L0.cor;
        S.buf[1] = M.msol;
    }
    M.ctl_dirty = true;   // until the solve ends normally
    // average_down_acoef (:1641-1661): level 1 in the initial smoothing, levels 2..cb in the
    // first V-cycle's down-sweep, the coarse ones inside k_coarse_lds
    // initial smoothing from the guess (buf[1]) into buf[0], the iterate after zero cycles;
    // k_target then sets the convergence target from its residual and rhs max norms
    S.nblk = smooth<4, false, true, false, true, true, true>(c, S.L0, L1, S.buf[0], S.rhs0, S.rcs, S.L0.acf, S.buf[1],
                                                             nullptr, L1.res, nullptr, M.d_norms);
    S.tol_rel = tol_rel;
    S.tol_abs = tol_abs;
    // the convergence bookkeeping rides on the first launch of the next V-cycle when there
    // is a tiled level 1 to carry it; the last cycle of every batch publishes with k_check.
    // After a solve that needed no V-cycle (an initial guess within the tolerance), the
    // target is evaluated and published first, so that no cycle is enqueued speculatively.
    const bool can_fold = M.coarse_begin > 1 && maxiter > 0;
    const bool probe = M.last_zero && maxiter > 0;
    if (!can_fold || probe) {
        const int seq = probe ? ++M.seq : 0;
        const Check chk0{S.ctl, S.other, M.d_mirror, M.d_norms, S.nblk, seq, maxiter, tol_rel, tol_abs};
        hipLaunchKernelGGL(k_target, dim3(1), dim3(NT), 0, c->stream, chk0);
    }
    HPQ_HIP(hipGetLastError());
    int batch = std::max(1, std::min(M.last_iters, maxiter));
    int issued = 0;
    bool checked = !can_fold || probe;   // the previous cycle's end (or the target) has been evaluated
    Published pub{};
    const bool done0 = probe && (pub = wait_mirror(c, M.seq)).done;
    while (!done0) {
        for (int b = 0; b < batch && issued < maxiter; ++b, ++issued) {
            const bool last = b + 1 == batch || issued + 1 == maxiter;
            vcycle(c, S, issued, maxiter, !checked, last || !can_fold);
            checked = last || !can_fold;
        }
        HPQ_HIP(hipGetLastError());
        if (issued == 0) break;   // maxiter == 0

        pub = wait_mirror(c, M.seq);
        if (pub.done || issued >= maxiter) break;
        batch = 1;
    }
    int it = 0, status = 0;
    if (issued || done0) {
        it = pub.iters;
        status = pub.status;
    } else {
        // no V-cycle allowed: converged only if the initial residual met the target
        MGCtl h;
        HPQ_HIP(hipMemcpyAsync(&h, S.ctl, sizeof(MGCtl), hipMemcpyDeviceToHost, c->stream));
        HPQ_HIP(hipStreamSynchronize(c->stream));
        status = h.done ? HPQ_OK : HPQ_E_MG_NOT_CONVERGED;
    }
    M.last_iters = std::max(1, it);
    M.last_zero = (issued || done0) && it == 0 && status == HPQ_OK;
    if (iters) *iters = it;
    // the result is buf[it & 1]; in the aliased layout buf[1] is sol itself
    if (!(alias && (it & 1))) {
        const int n = (S.L0.vihi - S.L0.vilo + 1) * (S.L0.vjhi - S.L0.vjlo + 1);
        hipLaunchKernelGGL(k_mg_store, grid1d(n, 256), dim3(256), 0, c->stream, S.L0, sh, c->g, sol, cstride,
                           S.buf[it & 1]);
    }
    HPQ_HIP(hipGetLastError());
    if (issued || done0) {
        M.ctl_pick ^= 1;
        M.ctl_dirty = false;
    }
    return status;
}

}  // namespace hpq
