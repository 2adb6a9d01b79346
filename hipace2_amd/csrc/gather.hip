// Beam deposition in the reference CPU build's summation order, on gfx950, without atomics on
// the planes.
//
// The CPU build deposits with SharedMemoryDeposition's tiled loop
// (src/particles/deposition/DepositionUtil.H:204-253; tiling on, 32-cell tiles under OpenMP,
// src/Hipace.H:235-240): particles are binned by the tile of their lowest deposited cell
// (start cell), the tiles are visited in four colours (even/odd tile index in x, then in y),
// and inside a tile the particles go in index order. Tiles of one colour never share a cell,
// so every cell receives its contributions in one fixed sequence: the up to four tiles that
// reach it in colour order, and inside each tile the particles by index. (The plasma's
// depositions in this order are in ordered.hip: its indices follow its cells, a beam's do
// not.)
//
// The particles that reach a cell are those whose start cell lies in the S x S window below it
// (S = stencil width); they are found through per-start-cell lists:
//   keys    the start cell of every particle and its slot in that cell's list (one atomic per
//           distinct cell of a wavefront, slots in lane order);
//   count   particles per start cell, exclusive scan -> list offsets;
//   scatter particles into their lists (atomic slots, any order);
//   order   each list sorted by particle index (rank by counting inside the list); at its
//           list position the particle's record is written;
//   pairs   every (particle, stencil offset) pair writes its contribution at its place in its
//           cell's sequence;
//   sum     each cell adds its sequence in order to the plane's value. The sequences hold jx, jy
//           and jz and depend on the beam alone: the predictor-corrector loop, which deposits
//           the same slice's beam in every iteration, builds them once, and the slice after it
//           uses them again.
#include <climits>
#include <cmath>

#include "internal.hpp"
#include "ordered.hpp"
#include "shape.hpp"

namespace hpq {

namespace {

// lists of one particle set keyed by base cell: base cells [blo, blo + w) in each direction;
// tiles of the deposition order: T cells (hipace.tile_size), ntx x nty over the guarded box
struct CLView {
    int bxlo, bylo, wx, wy;
    int T, ntx, nty;
    const int32_t* __restrict__ off;    // wx * wy + 1 list offsets
    const int32_t* __restrict__ perm;   // particle indices, list by list, increasing in a list
};

// The colours (0..3, the CPU build's tile loop order) of the lists of the window of cell
// (i, j): a window of S <= T cells spans at most two tiles per direction, split at column xs
// and row ys; bit k of mask[c] is set when list k = ky * S + kx has colour c (S <= 6).
template <int S>
struct WindowColours {
    unsigned long long mask[4];   // S * S <= 36 lists
    __device__ __forceinline__ WindowColours(const Geom& g, const CLView& cl, int i, int j) {
        const int x0 = i - S + 1, y0 = j - S + 1;
        const int txa = dep_tile(x0, g.ng, cl.T, cl.ntx), txb = dep_tile(i, g.ng, cl.T, cl.ntx);
        const int tya = dep_tile(y0, g.ng, cl.T, cl.nty), tyb = dep_tile(j, g.ng, cl.T, cl.nty);
        const int xs = txa == txb ? i + 1 : txb * cl.T - g.ng;
        const int ys = tya == tyb ? j + 1 : tyb * cl.T - g.ng;
#pragma unroll
        for (int c = 0; c < 4; ++c) mask[c] = 0ull;
#pragma unroll
        for (int k = 0; k < S * S; ++k) {
            const int kx = k % S, ky = k / S;
            const int tx = x0 + kx < xs ? txa : txb, ty = y0 + ky < ys ? tya : tyb;
            const int c = ((tx & 1) << 1) | (ty & 1);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (c == q) mask[q] |= 1ull << k;
        }
    }
};

// ---- list construction --------------------------------------------------------------------

// The beam deposit's per-particle values (BeamDepositCurrent.cpp:133-193): [0] wq vx,
// [1] wq vy, [2] wq vz, then the shape factors of its O + 1 stencil columns and of its O + 1
// stencil rows (a beam's dense core makes every cell merge long lists: the factors are taken
// once per particle here instead of once per cell there).
constexpr int BEAM_NREC = 3 + 2 * 4;

// slot of a particle in the list of start cell k (k < 0: none): one atomic per distinct k
// among the active lanes of the wavefront, and consecutive slots for its lanes in lane order
__device__ __forceinline__ int list_slot(int k, int32_t* __restrict__ count) {
    const int lane = threadIdx.x & 63;
    const unsigned long long lt = lane ? (~0ull >> (64 - lane)) : 0ull;
    unsigned long long todo = __ballot(k >= 0);
    unsigned long long peers = 0;
    while (todo) {
        const int l = __ffsll((long long)todo) - 1;
        const int kk = __shfl(k, l);
        const unsigned long long m = __ballot(k == kk);
        if (k == kk) peers = m;
        todo &= ~m;
    }
    const int leader = peers ? __ffsll((long long)peers) - 1 : lane;
    int base = 0;
    if (k >= 0 && lane == leader) base = atomicAdd(&count[k], __popcll(peers));
    base = __shfl(base, leader);
    return base + __popcll(peers & lt);
}

// Beam keys (BeamDepositCurrent.cpp:109-160): particles first .. first + count - 1 of the
// beam, numbered from 0.
template <int O>
__global__ __launch_bounds__(256) void k_keys_beam(Geom g, hpq_beam b, long first, long count_p, CLView cl,
                                                   const int32_t* __restrict__ select, int select_value,
                                                   int32_t* __restrict__ key, int32_t* __restrict__ slot,
                                                   int32_t* __restrict__ count) {
    const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= count_p) return;
    const long ip = first + t;
    int k = -1;
    if (b.valid[ip] && !(select && select[ip] != select_value)) {
        const double xmid = (b.x[ip] - g.xoff) * g.dxi;
        const double ymid = (b.y[ip] - g.yoff) * g.dyi;
        const int bx = shape<O>(xmid, 0).cell - shape_delta<O>() - cl.bxlo;
        const int by = shape<O>(ymid, 0).cell - shape_delta<O>() - cl.bylo;
        if (bx >= 0 && bx < cl.wx && by >= 0 && by < cl.wy) k = by * cl.wx + bx;
    }
    key[t] = k;
    const int sl = list_slot(k, count);
    if (k >= 0) slot[t] = sl;
}

// a fresh set of lists: the per-start-cell counts off[0, n) and the count of long sequences
__global__ __launch_bounds__(256) void k_lists_clear(int32_t* __restrict__ off, long n, int32_t* __restrict__ longc) {
    const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < n) off[t] = 0;
    if (t == 0) longc[0] = 0;
}

// particle t into its list at its atomic slot
__global__ __launch_bounds__(256) void k_lists_scatter(long n, const int32_t* __restrict__ key,
                                                       const int32_t* __restrict__ slot,
                                                       const int32_t* __restrict__ off, int32_t* __restrict__ unsorted) {
    const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n || key[t] < 0) return;
    unsorted[off[key[t]] + slot[t]] = int32_t(t);
}

// the rank of particle t by index inside its list: its list position
__device__ __forceinline__ int list_position(long t, const int32_t* __restrict__ key, const int32_t* __restrict__ off,
                                             const int32_t* __restrict__ unsorted) {
    const int a = off[key[t]], b = off[key[t] + 1];
    int r = 0;
    int u = a;
    // eight loads in flight at a time: a beam core's lists hold hundreds of particles
    for (; u + 8 <= b; u += 8) {
        int32_t q[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) q[k] = unsorted[u + k];
#pragma unroll
        for (int k = 0; k < 8; ++k) r += q[k] < int32_t(t) ? 1 : 0;
    }
    for (; u < b; ++u) r += unsorted[u] < int32_t(t) ? 1 : 0;
    return a + r;
}

// beam particle first + t to its list position, with its record (BEAM_NREC arrays, list order)
template <int O>
__global__ __launch_bounds__(256) void k_lists_order_beam(Geom g, hpq_beam b, long first, long count_p,
                                                          const int32_t* __restrict__ key,
                                                          const int32_t* __restrict__ off,
                                                          const int32_t* __restrict__ unsorted,
                                                          int32_t* __restrict__ perm, double* __restrict__ rec) {
    const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= count_p || key[t] < 0) return;
    const int pos = list_position(t, key, off, unsorted);
    perm[pos] = int32_t(t);
    const long ip = first + t;
    const double clightsq = 1.0 / (1.0 * 1.0);
    const double ux = b.ux[ip], uy = b.uy[ip], uz = b.uz[ip];
    const double gaminv = 1.0 / sqrt(1.0 + ux * ux * clightsq + uy * uy * clightsq + uz * uz * clightsq);
    const double wq = b.charge * b.w[ip] * 1.0;
    rec[pos] = wq * (ux * gaminv);
    rec[count_p + pos] = wq * (uy * gaminv);
    rec[2 * count_p + pos] = wq * (uz * gaminv);
    const double xmid = (b.x[ip] - g.xoff) * g.dxi;
    const double ymid = (b.y[ip] - g.yoff) * g.dyi;
#pragma unroll
    for (int k = 0; k <= O; ++k) {
        rec[(3 + k) * count_p + pos] = shape<O>(xmid, k).s;
        rec[(3 + O + 1 + k) * count_p + pos] = shape<O>(ymid, k).s;
    }
}

// ---- beam: per-cell contribution sequences -----------------------------------------------
// A beam's core puts hundreds of particles in a cell, in random index order, so merging a
// cell's window lists one element at a time would leave one thread per cell walking thousands
// of entries. Instead every (particle, stencil offset) pair finds its own place in its target
// cell's sequence at once: the sequence is the window's lists colour by colour, each colour
// merged by particle index, so a pair's place is the length of the lists of earlier colours
// plus, for every list of its own colour, the number of its entries with a smaller index (a
// binary search; the pair's own list gives its list rank). The pair writes its contribution
// there; then each cell adds its sequence in order to the plane's value, one thread per cell,
// or one wavefront per cell where the sequence is long.
constexpr int BEAM_LONG = 32;   // longer sequences: a wavefront per cell

// sequence length of every plane cell: the entries of its window lists (thread per cell);
// cells with long sequences are listed in longc (count at longc[0])
template <int O>
__global__ __launch_bounds__(256) void k_beam_seg_count(Geom g, CLView cl, int32_t* __restrict__ seg,
                                                        int32_t* __restrict__ longc) {
    constexpr int S = O + 1, DELTA = shape_delta<O>();
    const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t > g.plane) return;
    if (t == g.plane) {
        seg[t] = 0;
        return;
    }
    const int i = int(t % g.ldx) - g.ng, j = int(t / g.ldx) - g.ng;
    const int col0 = i - S + 1 - DELTA - cl.bxlo, row0 = j - S + 1 - DELTA - cl.bylo;
    int len = 0;
#pragma unroll
    for (int ky = 0; ky < S; ++ky) {
        const long r = long(row0 + ky) * cl.wx;
        len += cl.off[r + col0 + S] - cl.off[r + col0];
    }
    seg[t] = len;
    if (len > BEAM_LONG) longc[1 + atomicAdd(&longc[0], 1)] = int32_t(t);
}

// entries of perm[a, b) (increasing) below v
__device__ __forceinline__ int count_below(const int32_t* __restrict__ perm, int a, int b, int v) {
    int lo = a, hi = b;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (perm[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo - a;
}

// pair (list entry pos, stencil offset q): its place in the target cell's sequence and its
// contribution (BeamDepositCurrent.cpp:160-193: wq v times the two shape factors)
template <int O>
__global__ __launch_bounds__(256) void k_beam_pairs(Geom g, CLView cl, const int32_t* __restrict__ key,
                                                    const double* __restrict__ rec, long n,
                                                    const int32_t* __restrict__ seg, double* __restrict__ contrib,
                                                    long m) {
    constexpr int S = O + 1, DELTA = shape_delta<O>();
    const long tid = long(blockIdx.x) * blockDim.x + threadIdx.x;
    const long pl = tid / (S * S);
    const int q = int(tid - pl * (S * S));
    if (pl >= cl.off[long(cl.wx) * cl.wy]) return;
    const int pos = int(pl);
    const int p = cl.perm[pos];
    const int list = key[p];
    const int ix = q % S, iy = q / S;
    const int i = list % cl.wx + cl.bxlo + DELTA + ix, j = list / cl.wx + cl.bylo + DELTA + iy;
    if (i < -g.ng || i > g.nx - 1 + g.ng || j < -g.ng || j > g.ny - 1 + g.ng) return;
    const WindowColours<S> wc(g, cl, i, j);
    const int kp = (S - 1 - iy) * S + (S - 1 - ix);
    int cp = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if ((wc.mask[c] >> kp) & 1ull) cp = c;
    const int col0 = i - S + 1 - DELTA - cl.bxlo, row0 = j - S + 1 - DELTA - cl.bylo;
    int rank = pos - cl.off[list];
#pragma unroll
    for (int k = 0; k < S * S; ++k) {
        if (k == kp) continue;
        int c = 0;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc)
            if ((wc.mask[cc] >> k) & 1ull) c = cc;
        if (c > cp) continue;
        const long L = long(row0 + k / S) * cl.wx + col0 + k % S;
        const int a = cl.off[L], e = cl.off[L + 1];
        rank += c < cp ? e - a : count_below(cl.perm, a, e, p);
    }
    const long out = long(seg[g.idx(i, j)]) + rank;
    const double sx = rec[(3 + ix) * n + pos], sy = rec[(3 + O + 1 + iy) * n + pos];
    contrib[out] = sx * sy * rec[pos];
    contrib[m + out] = sx * sy * rec[n + pos];
    contrib[2 * m + out] = sx * sy * rec[2 * n + pos];
}

// Every cell's sum, added to the plane's value in sequence order; jx and jy go together, as in
// the deposit functor. The first workgroups take a wavefront per cell of longc: chunks of 64
// contributions per component are read by the whole wavefront into LDS (LCH chunks in flight), and
// lanes 0-2 add the jx, jy and jz chunks. The last nshort take a thread per cell with a short
// sequence. One launch for both: the predictor-corrector loop runs it in every iteration, where a
// launch more costs 4 us of some 60. Bound by the chain of adds of the longest sequences, so these
// start first, and the wavefronts of a workgroup take cells far apart in the list, whose neighbours
// are neighbours in the beam's core. Measured for the densest slice of a beam of two million particles
// at 255 x 255 (the longest sequences hold some 300000) 2.00 ms, of four million at
// 511 x 511, order 3, 205 us; with two launches, the long ones in workgroups of one wavefront,
// 2.13 ms and 221 us; with neighbours in one workgroup, after the short ones, 2.52 ms and 289 us.
__global__ __launch_bounds__(256) void k_beam_sum(Geom g, const int32_t* __restrict__ seg,
                                                  const double* __restrict__ contrib, long m,
                                                  double* __restrict__ store, int cjx, int cjy, int cjz,
                                                  const int32_t* __restrict__ longc, int nshort) {
    const long ps = g.plane;
    const int nlong = int(gridDim.x) - nshort;
    if (int(blockIdx.x) >= nlong) {
        const long t = long(int(blockIdx.x) - nlong) * blockDim.x + threadIdx.x;
        if (t >= g.plane) return;
        const int a = seg[t], e = seg[t + 1];
        if (a == e || e - a > BEAM_LONG) return;
        if (cjx >= 0) {
            double ajx = store[cjx * ps + t], ajy = store[cjy * ps + t];
            for (int h = a; h < e; ++h) {
                ajx += contrib[h];
                ajy += contrib[m + h];
            }
            store[cjx * ps + t] = ajx;
            store[cjy * ps + t] = ajy;
        }
        if (cjz >= 0) {
            double ajz = store[cjz * ps + t];
            for (int h = a; h < e; ++h) ajz += contrib[2 * m + h];
            store[cjz * ps + t] = ajz;
        }
        return;
    }
    constexpr int LCH = 4;
    __shared__ double buf_[4][3][64];
    const int lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
    double(*buf)[64] = buf_[wave];
    // a wavefront uses its own part of the LDS, whose operations execute in order
    auto fence = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    };
    const int comp = lane == 0 ? cjx : lane == 1 ? (cjx >= 0 ? cjy : -1) : lane == 2 ? cjz : -1;
    const int nl = longc[0];
    for (int w = wave * nlong + int(blockIdx.x); w < nl; w += 4 * nlong) {
        const long t = longc[1 + w];
        const int a = seg[t], e = seg[t + 1];
        double acc = comp >= 0 ? store[comp * ps + t] : 0.0;
        double v[LCH][3];
#pragma unroll
        for (int d = 0; d < LCH; ++d) {
            const int h = a + 64 * d + lane;
            v[d][0] = v[d][1] = v[d][2] = 0.0;
            if (h < e) {
                v[d][0] = contrib[h];
                v[d][1] = contrib[m + h];
                v[d][2] = contrib[2 * m + h];
            }
        }
        for (int h0 = a; h0 < e; h0 += 64 * LCH) {
#pragma unroll
            for (int d = 0; d < LCH; ++d) {
                const int hc = h0 + 64 * d;
                if (hc >= e) break;
                fence();
                buf[0][lane] = v[d][0];
                buf[1][lane] = v[d][1];
                buf[2][lane] = v[d][2];
                fence();
                const int hn = hc + 64 * LCH + lane;
                if (hn < e) {
                    v[d][0] = contrib[hn];
                    v[d][1] = contrib[m + hn];
                    v[d][2] = contrib[2 * m + hn];
                }
                if (comp >= 0) {
                    // in sequence order; eight LDS reads in flight while the eight before are added
                    const int cnt = min(64, e - hc);
                    const double* row = buf[lane];
                    if (cnt == 64) {
                        double q[2][8];
#pragma unroll
                        for (int k = 0; k < 8; ++k) q[0][k] = row[k];
#pragma unroll
                        for (int u = 8; u <= 64; u += 8) {
#pragma unroll
                            for (int k = 0; k < 8; ++k)
                                if (u < 64) q[(u / 8) & 1][k] = row[u + k];
                            asm volatile("" ::: "memory");
#pragma unroll
                            for (int k = 0; k < 8; ++k) acc += q[(u / 8 + 1) & 1][k];
                        }
                    } else {
                        int u = 0;
                        for (; u + 8 <= cnt; u += 8) {
                            double q[8];
#pragma unroll
                            for (int k = 0; k < 8; ++k) q[k] = row[u + k];
                            asm volatile("" ::: "memory");
#pragma unroll
                            for (int k = 0; k < 8; ++k) acc += q[k];
                        }
                        for (; u < cnt; ++u) acc += row[u];
                    }
                }
            }
        }
        if (comp >= 0) store[comp * ps + t] = acc;
    }
}

// base-cell grid of a context: every start cell whose stencil (at most 6 wide, start at most 2
// below the base cell) reaches the guarded plane; the deposition tiles
void lists_geometry(const hpq_ctx* c, CellLists& L) {
    const Geom& g = c->g;
    L.bxlo = -g.ng - 6;
    L.bylo = -g.ng - 6;
    L.wx = g.nx + 2 * g.ng + 9;
    L.wy = g.ny + 2 * g.ng + 9;
    L.T = c->p.tile_size > 0 ? c->p.tile_size : 32;
    L.ntx = (g.ldx + L.T - 1) / L.T;
    L.nty = (g.ldy + L.T - 1) / L.T;
}

CLView view(const CellLists& L) {
    return CLView{L.bxlo, L.bylo, L.wx, L.wy, L.T, L.ntx, L.nty, L.off, L.perm};
}

void lists_reserve(CellLists& L, long n, int nrec) {
    const long ns = long(L.wx) * L.wy;
    grow(L.off, L.off_cap, ns + 1);
    grow(L.tmp, L.tmp_cap, scan_tmp_size(ns + 1));
    grow(L.key, L.key_cap, n);
    grow(L.slot, L.slot_cap, n);
    grow(L.unsorted, L.unsorted_cap, n);
    grow(L.perm, L.perm_cap, n);
    grow(L.rec, L.rec_cap, long(nrec) * n);
}

// count (already in L.off) -> offsets -> unsorted lists; the caller's order kernel then
// sorts every list and writes the records
void lists_scatter(hipStream_t s, CellLists& L, long n) {
    const long ns = long(L.wx) * L.wy;
    scan_exclusive(s, L.off, ns + 1, L.tmp);
    hipLaunchKernelGGL(k_lists_scatter, grid1d(n, 256), dim3(256), 0, s, n, L.key, L.slot, L.off, L.unsorted);
    HPQ_HIP(hipGetLastError());
}

void lists_clear(hipStream_t s, CellLists& L) {
    const long ns = long(L.wx) * L.wy;
    hipLaunchKernelGGL(k_lists_clear, grid1d(ns + 1, 256), dim3(256), 0, s, L.off, ns + 1, L.longc);
}

}  // namespace

void cell_lists_free(CellLists& L) {
    for (void* q : {(void*)L.off, (void*)L.tmp, (void*)L.key, (void*)L.slot, (void*)L.unsorted, (void*)L.perm,
                    (void*)L.rec, (void*)L.seg, (void*)L.segtmp, (void*)L.longc, (void*)L.contrib})
        if (q) (void)hipFree(q);
    L = CellLists{};
}

// The contribution sequences of ::DepositCurrentSlice in the CPU build's order (particles of
// `slice` whose select entry equals select_value; select NULL: all), for beam_sequences_add.
// The slice has particles. Two slices' sequences are held: a slice deposits its own jz and the
// next one's jx and jy, so each slice's beam is deposited in two slices in a row, and the
// sequences that the first built serve the second. They are forgotten when the particles may have
// changed: at every call from outside, and where the slice is pushed or its weights change.
const CellLists& beam_sequences(hpq_ctx* c, const hpq_beam* b, int slice, const int32_t* select, int select_value) {
    const Geom& g = c->g;
    for (const CellLists& L : c->cl_beam)
        if (!select && L.slice == slice) return L;
    // in the place of none or of the slice that is done with: slices go downwards
    auto age = [](const CellLists& L) { return L.slice < 0 ? INT_MAX : L.slice; };
    CellLists& L = c->cl_beam[age(c->cl_beam[1]) > age(c->cl_beam[0]) ? 1 : 0];
    L.slice = -1;
    const long first = b->off[slice];
    const long count = b->off[slice + 1] - first;
    const int S = c->p.depos_order + 1;
    if (count > INT32_MAX / (S * S)) throw HpqError(HPQ_E_INVALID, "ordered beam deposition: too many particles in a slice");
    lists_geometry(c, L);
    lists_reserve(L, count, BEAM_NREC);
    grow(L.seg, L.seg_cap, g.plane + 1);
    grow(L.segtmp, L.segtmp_cap, scan_tmp_size(g.plane + 1));
    grow(L.longc, L.longc_cap, g.plane + 1);
    const long m = long(S) * S * count;
    grow(L.contrib, L.contrib_cap, 3 * m);
    L.m = m;
    TraceScope ts(c, HPQ_TRACE_BEAM_DEPOSIT);
    lists_clear(c->stream, L);
    dispatch_order(c->p.depos_order, [&](auto O) {
        constexpr int o = decltype(O)::value;
        hipLaunchKernelGGL(k_keys_beam<o>, grid1d(count, 256), dim3(256), 0, c->stream, g, *b, first, count, view(L),
                           select, select_value, L.key, L.slot, L.off);
        HPQ_HIP(hipGetLastError());
        lists_scatter(c->stream, L, count);
        hipLaunchKernelGGL(k_lists_order_beam<o>, grid1d(count, 256), dim3(256), 0, c->stream, g, *b, first, count,
                           L.key, L.off, L.unsorted, L.perm, L.rec);
        hipLaunchKernelGGL(k_beam_seg_count<o>, grid1d(g.plane + 1, 256), dim3(256), 0, c->stream, g, view(L), L.seg,
                           L.longc);
        scan_exclusive(c->stream, L.seg, g.plane + 1, L.segtmp);
        hipLaunchKernelGGL(k_beam_pairs<o>, grid1d(m, 256), dim3(256), 0, c->stream, g, view(L), L.key, L.rec, count,
                           L.seg, L.contrib, m);
    });
    HPQ_HIP(hipGetLastError());
    if (!select) L.slice = slice;
    return L;
}

void beam_sequences_forget(hpq_ctx* c, int slice) {
    for (CellLists& L : c->cl_beam)
        if (slice < 0 || L.slice == slice) L.slice = -1;
}

// the sequences added to the planes comps (jx, jy, jz; -1: none)
void beam_sequences_add(hpq_ctx* c, const CellLists& L, double* store, const int32_t* comps) {
    const Geom& g = c->g;
    TraceScope ts(c, HPQ_TRACE_BEAM_DEPOSIT);
    const int nshort = int((g.plane + 255) / 256);
    hipLaunchKernelGGL(k_beam_sum, dim3(nshort + 512), dim3(256), 0, c->stream, g, L.seg, L.contrib, L.m, store,
                       comps[0], comps[1], comps[2], L.longc, nshort);
    HPQ_HIP(hipGetLastError());
}

}  // namespace hpq
