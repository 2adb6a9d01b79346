// Plasma deposition in the reference CPU build's summation order, on gfx950, without atomics
// on the planes.
//
// The CPU build deposits with SharedMemoryDeposition's tiled loop
// (src/particles/deposition/DepositionUtil.H:204-253; tiling on, 32-cell tiles under OpenMP,
// src/Hipace.H:235-240): particles are binned by the tile of their lowest deposited cell
// (start cell), the tiles are visited in four colours (even/odd tile index in x, then in y),
// and inside a tile the particles go in index order (amrex::DenseBins is a stable counting
// sort). Tiles of one colour never share a cell, so every cell receives its contributions in
// one fixed sequence: the up to four tiles that reach it in colour order, and inside each
// tile the particles by index.
//
// Here a wavefront owns a block of cells and takes the particles that reach it in that order,
// one after the other, so the planes come out bit for bit as the CPU build's loop leaves them,
// and no two wavefronts write one cell. Nothing is sorted: the particle arrays are in index
// order already, and
//   records  one pass over the particles writes each one's deposit values as one 64-byte
//            record, its cell as one word, and the bounding boxes of the cells of every RUN
//            and every SUPER consecutive particles (the QSA removal of the deposit functor
//            happens here); every run is listed at the blocks whose window (the cells a particle
//            reaching the block can start in) its box meets, or, where these are many, its
//            particles are linked into lists by cell;
//   deposit  a wavefront sorts its list, takes the window's particles from the listed runs by
//            index and the linked ones with them, sequences them by colour, and adds them to its
//            block's sums in LDS.
// What a window's particles cost to add does not depend on the order of the arrays; what they cost
// to find does. Measured at 511 x 511, 2 x 2 particles per cell, order 2, in us of kernels, with
// per-cell lists (built by counting, scanning and scattering; walked cell by cell, block by block
// in raster order where the plasma is near its lattice and merged by index elsewhere) and now:
//                                        lists / records   current      explicit
//   linear wake (near the lattice)          51 -> 36      123 -> 111   229 -> 191
//   nonlinear wake (crossing)               57 -> 39      402 -> 131  1313 -> 249
//   arrays in random order (linked)        222 -> 58      342 -> 231  1034 -> 319
//
// A particle's cell is the floor of the cell-scaled position the shape functions take theirs
// from (floor(xmid) or floor(xmid + 1/2)); a stencil's start cell is that floor plus a
// constant, so the explicit Sx/Sy deposition of the default derivative type reuses the
// records the current deposition made of the same particles.
#include <algorithm>
#include <climits>
#include <cmath>

#include "internal.hpp"
#include "ordered.hpp"
#include "shape.hpp"

namespace hpq {

namespace {

constexpr int RUN = 64;          // particles per box of the first level
constexpr int SUPER = 256;       // particles per box of the second level
constexpr int RUNS_PER_SUPER = SUPER / RUN;
constexpr uint32_t NO_CELL = 0xffffffffu;
constexpr int REC = 8;           // doubles per record
constexpr int LIST = 128;        // runs listed per block
constexpr int NEXT = 0, MADE = 16, PASS_WORDS = 32;   // words of OrdView::pass, on lines of their own
constexpr int BIN = 2;           // log2 of the width and height of a bin of linked particles
constexpr int HEADS = 8;         // linked lists per bin

// Records, cells and boxes of one plasma state. Cells count from (bxlo, bylo): x in the low
// `shift` bits of the word, y above them. A box is (xmin, xmax, ymin, ymax), empty when
// xmin > xmax.
struct OrdView {
    int bxlo, bylo, shift;
    int T, ntx, nty;   // deposition tiles: T cells (hipace.tile_size), ntx x nty over the guarded box
    int nrun, nsuper;
    int lw, lh;        // log2 of a block's width and height
    int nbx, nby;      // blocks
    int mlo, mhi;      // cells a block's window reaches below and above it
    int narrow;        // blocks that a listed run meets, at most
    long n;
    const double* __restrict__ rec;
    const uint32_t* __restrict__ cell;
    const int4* __restrict__ rbox;
    const int4* __restrict__ sbox;
    // Runs listed per block (may exceed LIST), then whether particles are linked: two sets, those of
    // even and of odd passes, each cleared by the pass before.
    const int32_t* __restrict__ count;
    const int32_t* __restrict__ list;    // LIST runs per block, in any order
    // Kept beside these arrays, and found from them by the few that need it, since a kernel argument
    // takes a register all along:
    // Passes are numbered on the device. A records pass takes the number in pass()[NEXT] and notes it
    // in pass()[MADE], the deposition that reads it sets pass()[NEXT] to the one after. Nothing that a
    // pass depends on is kept by the host, so that a recorded pass may be replayed any number of times.
    __host__ __device__ const int32_t* pass() const { return count - PASS_WORDS; }
    // The particles of runs that meet too many blocks, linked by the bin of their cell in HEADS
    // lists each: the pass that made the list in the high word, particle + 1 in the low one, and the
    // next of a particle's list + 1 (0: none) in link().
    __host__ __device__ const unsigned long long* head() const {
        return reinterpret_cast<const unsigned long long*>(count + 2 * (nbx * nby + 1));
    }
    __host__ __device__ const uint32_t* link() const { return cell + n; }
    __host__ __device__ static int bins(int cells, int ng) { return (cells_found(cells, ng) + (1 << BIN) - 1) >> BIN; }
    // cells counted in one direction: every start cell whose stencil (at most 6 wide, start at most 2
    // below the cell) reaches the guarded plane has its cell among them
    __host__ __device__ static int cells_found(int cells, int ng) { return cells + 2 * ng + 9; }
};

// The deposit functor's per-particle values of the current and explicit deposition
// (PlasmaDepositCurrent.cpp:182-243, ExplicitDeposition.cpp:174-205; the two evaluate them
// with the same operations): q w invvol, vx/c = ux/psi, vy/c, gamma/psi, 1/psi, and the
// cell-scaled position.
struct PlasmaVals {
    double q_invvol, vx_c, vy_c, gamma_psi, psi_inv, xmid, ymid;
};
__device__ __forceinline__ PlasmaVals plasma_vals(const Geom& g, const hpq_plasma& p, long ip, double charge_invvol) {
    const double clightinv = 1.0 / 1.0;
    PlasmaVals v;
    v.psi_inv = 1.0 / p.psi[ip];
    v.vx_c = p.ux[ip] * v.psi_inv;
    v.vy_c = p.uy[ip] * v.psi_inv;
    v.q_invvol = charge_invvol * p.w[ip];
    v.xmid = (p.x[ip] - g.xoff) * g.dxi;
    v.ymid = (p.y[ip] - g.yoff) * g.dyi;
    const double Aabssqp = 0.0;
    v.gamma_psi = 0.5 * ((1.0 + 0.5 * Aabssqp) * v.psi_inv * v.psi_inv + v.vx_c * v.vx_c * clightinv * clightinv +
                         v.vy_c * v.vy_c * clightinv * clightinv + 1.0);
    return v;
}

// Records of SUPER consecutive particles per workgroup, RUN of them per wavefront. QSA: the
// removal of the current deposit functor (PlasmaDepositCurrent.cpp:182-198).
// wx, wy: particles whose cell lies outside [0, wx) x [0, wy) reach no cell of the plane.
// Bound by HBM: 52 bytes read and 68 written per particle. Where all particles are linked (random
// order), by one atomic exchange for each, 22 us more at a million particles.
constexpr int REC_T = SUPER;
template <int BASE, bool QSA>
__global__ __launch_bounds__(REC_T) void k_records(Geom g, hpq_plasma p, OrdView v, int wx, int wy,
                                                   double charge_invvol, double max_qsa, double* __restrict__ rec,
                                                   uint32_t* __restrict__ cell, int4* __restrict__ rbox,
                                                   int4* __restrict__ sbox, int32_t* __restrict__ counts,
                                                   int32_t* __restrict__ list, unsigned long long* __restrict__ head,
                                                   uint32_t* __restrict__ link, int32_t* __restrict__ made,
                                                   int* __restrict__ qsa_count) {
    __shared__ int box[4];
    const int nblk = v.nbx * v.nby;
    const unsigned pass = unsigned(v.pass()[NEXT]);
    int32_t* const count = counts + long(pass & 1) * (nblk + 1);
    if (threadIdx.x < 4) box[threadIdx.x] = (threadIdx.x & 1) ? -1 : INT_MAX;
    __syncthreads();
    const long ip = long(blockIdx.x) * SUPER + threadIdx.x;
    int bx = -1, by = -1;
    if (ip < p.n) {
        uint32_t w = NO_CELL;
        if (p.valid[ip]) {
            const PlasmaVals u = plasma_vals(g, p, ip, charge_invvol);
            if (QSA && (u.gamma_psi < 0.0 || u.gamma_psi > max_qsa || u.psi_inv < 0.0)) {
                atomicAdd(qsa_count, 1);
                p.w[ip] = 0.0;
                p.valid[ip] = 0;
            } else {
                const int cx = int(BASE ? floor(u.xmid + 0.5) : floor(u.xmid)) - v.bxlo;
                const int cy = int(BASE ? floor(u.ymid + 0.5) : floor(u.ymid)) - v.bylo;
                if (cx >= 0 && cx < wx && cy >= 0 && cy < wy) {
                    bx = cx;
                    by = cy;
                    w = (uint32_t(cy) << v.shift) | uint32_t(cx);
                    double2* r = reinterpret_cast<double2*>(rec + ip * REC);
                    r[0] = make_double2(u.q_invvol, u.vx_c);
                    r[1] = make_double2(u.vy_c, u.gamma_psi);
                    r[2] = make_double2(u.psi_inv, u.xmid);
                    r[3] = make_double2(u.ymid, __hiloint2double(0, int(w)));
                }
            }
        }
        cell[ip] = w;
    }
    // the bounding box of the cells of the wavefront's particles that `of` selects
    auto bounds = [&](bool of) -> int4 {
        int4 q = make_int4(of ? bx : INT_MAX, of ? bx : -1, of ? by : INT_MAX, of ? by : -1);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            q.x = min(q.x, __shfl_xor(q.x, o));
            q.y = max(q.y, __shfl_xor(q.y, o));
            q.z = min(q.z, __shfl_xor(q.z, o));
            q.w = max(q.w, __shfl_xor(q.w, o));
        }
        return q;
    };
    // the blocks whose window a box meets
    struct Met {
        int bx0, bx1, by0, by1, nx, n;
    };
    auto met = [&](const int4& q) -> Met {
        const int c0 = v.bxlo + g.ng, r0 = v.bylo + g.ng;   // cell 0 counted from block 0's first
        Met m;
        m.bx0 = max(q.x + c0 - v.mhi, 0) >> v.lw;
        m.bx1 = min((q.y + c0 + v.mlo) >> v.lw, v.nbx - 1);
        m.by0 = max(q.z + r0 - v.mhi, 0) >> v.lh;
        m.by1 = min((q.w + r0 + v.mlo) >> v.lh, v.nby - 1);
        m.nx = m.bx1 - m.bx0 + 1;
        m.n = m.nx > 0 && m.by1 >= m.by0 ? m.nx * (m.by1 - m.by0 + 1) : 0;
        return m;
    };
    // the run into the lists of blocks
    const int lane = int(threadIdx.x & 63);
    auto into_lists = [&](const Met& m) {
        for (int t = lane; t < m.n; t += 64) {
            const int blk = (m.by0 + t / m.nx) * v.nbx + m.bx0 + t % m.nx;
            const int at = atomicAdd(&count[blk], 1);
            if (at < LIST) list[long(blk) * LIST + at] = int(ip / RUN);
        }
    };
    int4 q = bounds(bx >= 0);
    if (q.x <= q.y) {
        const Met m = met(q);
        if (m.n <= v.narrow) {
            into_lists(m);
        } else {
            // Up to four pieces, split along the longer side: the end of one lattice row and the start
            // of the next, particles on either side of a periodic boundary, a stray one. Where these
            // meet too many blocks as well, or one block twice, the particles go by themselves.
            auto halve = [&](bool of, const int4& r, bool& low) {   // true: along x
                const bool along = r.y - r.x >= r.w - r.z;
                low = of && (along ? bx <= (r.x + r.y) >> 1 : by <= (r.z + r.w) >> 1);
                return along;
            };
            auto apart = [&](bool along, const Met& a, const Met& b) {
                return a.n == 0 || b.n == 0 || (along ? a.bx1 < b.bx0 : a.by1 < b.by0);
            };
            bool of[2], low;
            const bool along = halve(bx >= 0, q, of[0]);
            of[1] = bx >= 0 && !of[0];
            int4 half[2];
            Met m[4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                half[h] = bounds(of[h]);
                m[2 * h] = met(half[h]);
                m[2 * h + 1] = Met{};
            }
            bool pieces = apart(along, m[0], m[2]);
            if (pieces && m[0].n + m[2].n > v.narrow) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bool al = halve(of[h], half[h], low);
                    const Met a = met(bounds(low)), b = met(bounds(of[h] && !low));
                    if (apart(al, a, b)) {
                        m[2 * h] = a;
                        m[2 * h + 1] = b;
                    }
                }
                pieces = m[0].n + m[1].n + m[2].n + m[3].n <= v.narrow;
            }
            if (pieces) {
#pragma unroll
                for (int k = 0; k < 4; ++k) into_lists(m[k]);
            } else {
                if (bx >= 0) {
                    const long k = (long(by >> BIN) * OrdView::bins(g.nx, g.ng) + (bx >> BIN)) * HEADS + ip % HEADS;
                    const unsigned long long mine = (unsigned long long)pass << 32 | unsigned(ip + 1);
                    const unsigned long long old = atomicExch(&head[k], mine);
                    link[ip] = unsigned(old >> 32) == pass ? uint32_t(old) : 0u;
                }
                // read by later launches only, so that each L2 may gather the stores
                if (lane == 0) __hip_atomic_store(&count[nblk], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                q = make_int4(INT_MAX, -1, INT_MAX, -1);   // found through the bins, not the boxes
            }
        }
    }
    if (lane == 0 && ip < p.n) {
        rbox[ip / RUN] = q;
        atomicMin(&box[0], q.x);
        atomicMax(&box[1], q.y);
        atomicMin(&box[2], q.z);
        atomicMax(&box[3], q.w);
    }
    int32_t* const next_count = counts + long(~pass & 1) * (nblk + 1);
    for (int t = int(blockIdx.x) * REC_T + int(threadIdx.x); t <= nblk; t += int(gridDim.x) * REC_T) next_count[t] = 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *made = int(pass);
    __syncthreads();
    if (threadIdx.x == 0) sbox[blockIdx.x] = make_int4(box[0], box[1], box[2], box[3]);
}

// ---- deposition -----------------------------------------------------------------------------
constexpr int SUPER_BATCH = 64;     // second-level boxes tested at a time
constexpr int BATCH = 16;           // runs tested at a time

__device__ __forceinline__ int lanes_before(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi(unsigned(m >> 32), __builtin_amdgcn_mbcnt_lo(unsigned(m), 0));
}

enum { CURRENT = 0, EXPLICIT = 1 };

// EXPLICIT: the components of Bz, Ez, ExmBy, EypBx, Sy, Sx. CURRENT: those asked for (-1: none)
// and the quantity of each, 0..5 for jx, jy, jz, rho, chi, rhomjz.
struct Comps {
    int c[6];
    int q[6];
};

template <int KIND, int T, int O>
struct Stencil {
    static constexpr int S = KIND == CURRENT ? O + 1 : dshape_width<T, O>();
    static constexpr int DELTA = KIND == CURRENT ? shape_delta<O>() : dshape_delta<T, O>();
    // the centred derivative's corner offsets contribute nothing
    static constexpr bool CORNERS = KIND == EXPLICIT && T == 2;
    static constexpr int N = S * S - (CORNERS ? 4 : 0);   // offsets
    // column and row of offset k (row by row, without the corners)
    static __host__ __device__ constexpr int row(int k) {
        if (!CORNERS) return k / S;
        return k < S - 2 ? 0 : k >= N - (S - 2) ? S - 1 : 1 + (k - (S - 2)) / S;
    }
    static __host__ __device__ constexpr int col(int k) {
        if (!CORNERS) return k % S;
        return k < S - 2 ? k + 1 : k >= N - (S - 2) ? k - (N - (S - 2)) + 1 : (k - (S - 2)) % S;
    }
    // particles a wavefront takes in one step, steps whose LDS reads are in flight together,
    // and particles staged at a time
    static constexpr int PP = KIND == EXPLICIT ? 64 / N : 1;
    static constexpr int U = KIND == EXPLICIT ? (PP <= 12 ? 3 : 1) : 8;
    static constexpr int CHUNK = KIND == EXPLICIT ? (36 / (PP * U) > 0 ? 36 / (PP * U) * (PP * U) : PP * U) : 32;
    static_assert(CHUNK <= 64, "one lane stages one particle");
    // double2 words of a staged entry. EXPLICIT: the shape factors and their derivatives of the
    // S columns and of the S rows, (q w invvol, 1/psi), (vx/c, vy/c), (gamma/psi, target).
    // CURRENT: (charge density, target) of the N offsets, the two factors of every quantity.
    static constexpr int ENT = KIND == EXPLICIT ? 2 * S + 3 : N + 6;
    // Entries sequenced at a time with blocks of `cells` cells, found in the place of the staged
    // ones; where a window holds more, its colours are taken one after the other, each from all
    // runs. The largest block's current deposition has room for 2048 without losing a wavefront
    // per CU: 131 instead of 156 us for crossing orbits at 511 x 511, 2 x 2 particles per cell, the
    // same near the lattice. The explicit one has not: with 1920 entries and 27 particles staged at a
    // time it takes 233 instead of 249 us there, but 201 instead of 191 near the lattice.
    static constexpr int seq(int cells) {
        const int room = CHUNK * ENT * 8, want = KIND == CURRENT && cells == 128 ? 2048 : 1024;
        return room < want ? room : want;
    }
};

// One wavefront per block of BW x BH cells of the guarded plane. ::DepositCurrent's per-cell
// sums (PlasmaDepositCurrent.cpp:199-283) or ::ExplicitDeposition's (ExplicitDeposition.cpp:
// 186-262, no laser, with the cell's own Bz, Ez, ExmBy, EypBx).
//
// The sums live in LDS and the particles are taken in order: the lanes are the offsets of a
// particle's stencil (EXPLICIT: of PP consecutive particles at once, the adds then issued one
// particle after the other; CURRENT: times the components), so the work per particle does not
// depend on where the next one sits. A wavefront's LDS operations execute in the order of its
// instructions, so ds_add_f64 adds in particle order. Values a particle's offsets share (shape
// factors, charge densities) are computed once when it is staged, one lane per particle.
//
// What bounds it is the LDS: per step of three particles seven 16-byte reads (4.3 cycles of a
// CU's LDS each) and six ds_add_f64 (8 each, however few lanes are active), 78 cycles, next to
// 60 vector instructions (42 of them FP64) on each of four SIMDs. A 16 x 8 block keeps the
// window of an order-2 derivative stencil at 1.9 times its cells and gives 511 x 511 cells
// 2145 wavefronts; CHUNK, SEQ and BS are chosen so that nine of them fit a CU's LDS, one round
// for that grid (eight in two rounds: 211 instead of 191 us). Smaller grids have smaller blocks.
// NSUM: the sums of a cell (CURRENT: components asked for, at most NSUM).
template <int KIND, int T, int O, int NSUM, int BW, int BH>
__global__ __launch_bounds__(64) void k_deposit_ordered(Geom g, OrdView v, double* __restrict__ store, Comps cm,
                                                        double charge_mass_ratio, int32_t* __restrict__ next) {
    using St = Stencil<KIND, T, O>;
    constexpr int S = St::S, N = St::N, PP = St::PP, U = St::U, CHUNK = St::CHUNK, ENT = St::ENT, SEQ = St::seq(BW * BH);
    constexpr int NW = BW + S - 1, NH = BH + S - 1;   // window, in cells
    constexpr int BS = BW + 4;   // LDS pitch of a block row: a stencil's rows on different banks
    constexpr int CELLS = BS * BH;
    static_assert(NW <= 64 && N <= 32, "window and offset masks");
    __shared__ double2 ent[CHUNK][ENT];
    __shared__ double2 field[KIND == EXPLICIT ? 2 : 1][KIND == EXPLICIT ? CELLS : 1];
    __shared__ double sum[NSUM][CELLS];
    // entries: colour << 13 | listed run << 6 | particle of the run, first by index (found, in the
    // place of the staged entries), then by colour
    __shared__ alignas(8) uint16_t seq[SEQ];
    uint16_t* const found = reinterpret_cast<uint16_t*>(&ent[0][0]);
    // with linked particles the sequence holds particle indices, sorted in the place of the staged
    // entries (see below)
    uint32_t* const seq_ip = reinterpret_cast<uint32_t*>(seq);
    uint32_t* const key = reinterpret_cast<uint32_t*>(&ent[0][0]);
    constexpr int KEYS = sizeof(ent) >= 4096 ? 1024 : 512;
    constexpr int KEEP = KEYS / 2 < SEQ / 2 ? KEYS / 2 : SEQ / 2;
    static_assert(sizeof(ent) >= KEYS * sizeof(uint32_t) && KEYS - KEEP >= 2 * RUN, "room for the keys");
    static_assert(sizeof(ent) >= SEQ * sizeof(uint16_t), "the found entries fit");
    __shared__ int runs[LIST];
    __shared__ uint16_t supers[SUPER_BATCH];
    const int lane = int(threadIdx.x);
    const int b = xcd_block(int(blockIdx.x), int(gridDim.x));
    const int i0 = (b % v.nbx) * BW - g.ng, j0 = (b / v.nbx) * BH - g.ng;
    const int X0 = i0 - S + 1 - St::DELTA - v.bxlo, Y0 = j0 - S + 1 - St::DELTA - v.bylo;
    const uint32_t xmask = (1u << v.shift) - 1u;
    // parity of the tile of every window column and row
    const unsigned long long PX = __ballot(dep_tile(i0 - S + 1 + lane, g.ng, v.T, v.ntx) & 1);
    const unsigned long long PY = __ballot(dep_tile(j0 - S + 1 + lane, g.ng, v.T, v.nty) & 1);

    auto meets = [&](const int4& q) { return q.y >= X0 && q.x < X0 + NW && q.w >= Y0 && q.z < Y0 + NH; };

    // Runs of particles that may hold some of the window, by index. The block's own list, sorted,
    // when it holds them all; otherwise (listed == false) those whose box meets the window, found
    // through the two levels of boxes, LIST at most by one call; pos is where the next goes on.
    const int nblk = v.nbx * v.nby, pass = v.pass()[MADE];
    // both sets' loads in flight with that of the pass
    const int own2[2] = {v.count[b], v.count[nblk + 1 + b]}, any2[2] = {v.count[nblk], v.count[2 * nblk + 1]};
    const int own = pass & 1 ? own2[1] : own2[0], any_linked = pass & 1 ? any2[1] : any2[0];
    if (blockIdx.x == 0 && lane == 0) *next = pass + 1;
    const bool listed = own <= LIST;
    // the lists of the bins that the window meets, and whether they hold any particle
    const int binx = X0 >> BIN, biny = Y0 >> BIN;
    const int nbinx = OrdView::bins(g.nx, g.ng), nbinw = min((X0 + NW - 1) >> BIN, nbinx - 1) - binx + 1;
    const int nlinks = nbinw * (min((Y0 + NH - 1) >> BIN, OrdView::bins(g.ny, g.ng) - 1) - biny + 1) * HEADS;
    auto first_linked = [&](int t) -> uint32_t {
        const int bin = t / HEADS, r = bin / nbinw;
        const unsigned long long h = v.head()[(long(biny + r) * nbinx + binx + bin - r * nbinw) * HEADS + t % HEADS];
        return unsigned(h >> 32) == unsigned(pass) ? uint32_t(h) : 0u;
    };
    bool linked = false;
    if (any_linked) {
        for (int t = lane; t < nlinks; t += 64) linked |= first_linked(t) != 0u;
        linked = __ballot(linked) != 0ull;
    }
    struct Pos {
        int s0 = 0;            // next second-level box
        int first = 0;         // first box of the current batch
        int n = 0, at = 0;     // listed boxes of the batch, and those taken
        bool end = false;
    };
    Pos pos;
    auto find_runs = [&]() -> int {
        int n = 0;
        __syncthreads();
        while (n <= LIST - 64 && !pos.end) {
            if (pos.at >= pos.n) {
                if (pos.s0 >= v.nsuper) {
                    pos.end = true;
                    break;
                }
                pos.first = pos.s0;
                pos.n = pos.at = 0;
                bool hit[SUPER_BATCH / 64];
#pragma unroll
                for (int q = 0; q < SUPER_BATCH / 64; ++q) {
                    const int s = pos.s0 + q * 64 + lane;
                    hit[q] = s < v.nsuper && meets(v.sbox[s]);
                }
                __syncthreads();
#pragma unroll
                for (int q = 0; q < SUPER_BATCH / 64; ++q) {
                    const unsigned long long h = __ballot(hit[q]);
                    if (hit[q]) supers[pos.n + lanes_before(h)] = uint16_t(q * 64 + lane);
                    pos.n += __popcll(h);
                }
                pos.s0 += SUPER_BATCH;
                __syncthreads();
                continue;
            }
            // sixteen listed boxes, the four runs of each on four lanes
            const int s = pos.at + lane / RUNS_PER_SUPER;
            const int id = s < pos.n ? (pos.first + int(supers[s])) * RUNS_PER_SUPER + lane % RUNS_PER_SUPER : v.nrun;
            const bool hit = id < v.nrun && meets(v.rbox[id]);
            pos.at += 64 / RUNS_PER_SUPER;
            const unsigned long long h = __ballot(hit);
            if (hit) runs[n + lanes_before(h)] = id;
            n += __popcll(h);
        }
        __syncthreads();
        return n;
    };
    // the block's sums and fields
    const long ps = g.plane;
    for (int t = lane; t < BW * BH; t += 64) {
        const int i = i0 + t % BW, j = j0 + t / BW, c = t / BW * BS + t % BW;
        const bool in = i <= g.nx - 1 + g.ng && j <= g.ny - 1 + g.ng;
        const long k = in ? g.idx(i, j) : 0;
        if constexpr (KIND == EXPLICIT) {
            field[0][c] = make_double2(store[cm.c[0] * ps + k], store[cm.c[1] * ps + k]);
            field[1][c] = make_double2(store[cm.c[2] * ps + k], store[cm.c[3] * ps + k]);
            sum[0][c] = store[cm.c[4] * ps + k];
            sum[1][c] = store[cm.c[5] * ps + k];
        } else {
#pragma unroll
            for (int q = 0; q < NSUM; ++q)
                if (cm.c[q] >= 0) sum[q][c] = store[cm.c[q] * ps + k];
        }
    }

    int nruns = 0;
    if (listed) {
        static_assert(LIST == 128 && sizeof(ent) >= LIST * sizeof(int), "two listed runs per lane");
        int4* unsorted = reinterpret_cast<int4*>(&ent[0][0]);
        int mine[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int t = lane + 64 * q;
            mine[q] = INT_MAX;
            if (t < own) mine[q] = v.list[long(b) * LIST + t];
            reinterpret_cast<int*>(unsorted)[t] = mine[q];
        }
        nruns = own;
        __syncthreads();
        int rank[2] = {0, 0};
#pragma unroll 4
        for (int t = 0; 4 * t < own; ++t) {
            const int4 r = unsorted[t];
#pragma unroll
            for (int q = 0; q < 2; ++q)
                rank[q] += (r.x < mine[q] ? 1 : 0) + (r.y < mine[q] ? 1 : 0) + (r.z < mine[q] ? 1 : 0) +
                           (r.w < mine[q] ? 1 : 0);
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (mine[q] != INT_MAX) runs[rank[q]] = mine[q];
        __syncthreads();
        pos.end = true;
    } else if (!linked) {
        nruns = find_runs();
    }

    // cells of the block inside the plane
    const int ncol_in = min(BW, g.nx + g.ng - i0), nrow_in = min(BH, g.ny + g.ng - j0);
    // this lane's offset of the stencil, and its particle of a step (EXPLICIT) or component
    const int part = lane / N, off = lane % N;
    const int ox = St::col(off), oy = St::row(off);
    const int shift = oy * BS + ox;

    int n = 0;   // entries of the sequence
    // the record of entry e of the sequence, of this lane in a chunk
    struct Record {
        double2 d[4];
    };
    auto fetch = [&](int e) -> Record {
        Record r;
        if (lane < CHUNK && e < n) {
            long ip;
            if (linked) {
                ip = long(seq_ip[e]);
            } else {
                const int id = seq[e];
                ip = long(runs[(id >> 6) & 127]) * RUN + (id & 63);
            }
            const double2* p = reinterpret_cast<const double2*>(v.rec + ip * REC);
#pragma unroll
            for (int f = 0; f < 4; ++f) r.d[f] = p[f];
        }
        return r;
    };
    // one chunk: cnt particles, lane by lane
    auto process = [&](const Record& rec, int cnt) {
        __syncthreads();
        if (lane < cnt) {
            const double2 r0 = rec.d[0], r1 = rec.d[1], r2 = rec.d[2], r3 = rec.d[3];
            const double q_invvol = r0.x, vx = r0.y, vy = r1.x, gamma_psi = r1.y, psi_inv = r2.x;
            const double xm = r2.y, ym = r3.x;
            const uint32_t word = uint32_t(__double2loint(r3.y));
            // column and row of the stencil's first cell in the block, and its cells inside
            const int x = int(word & xmask) - X0 - (S - 1), y = int(word >> v.shift) - Y0 - (S - 1);
            const uint32_t cols = stencil_bits(-x, ncol_in - x, S), rows = stencil_bits(-y, nrow_in - y, S);
            uint32_t inside = 0u;
#pragma unroll
            for (int r = 0; r < S; ++r) {
                constexpr uint32_t MID = S > 2 ? (1u << (S - 2)) - 1u : 0u;
                const bool edge = St::CORNERS && (r == 0 || r == S - 1);
                const uint32_t m = edge ? (cols >> 1) & MID : cols;
                const int at = !St::CORNERS ? r * S : r == 0 ? 0 : r * S - 2;
                if ((rows >> r) & 1u) inside |= m << at;
            }
            const double target = __hiloint2double(y * BS + x, int(inside));
            double2* e = ent[lane];
            if constexpr (KIND == EXPLICIT) {
#pragma unroll
                for (int k = 0; k < S; ++k) {
                    const Dsf X = dshape<T, O>(xm, k), Y = dshape<T, O>(ym, k);
                    e[k] = make_double2(X.s, X.ds);
                    e[S + k] = make_double2(Y.s, Y.ds);
                }
                e[2 * S] = make_double2(q_invvol, psi_inv);
                e[2 * S + 1] = make_double2(vx, vy);
                e[2 * S + 2] = make_double2(gamma_psi, target);
            } else {
#pragma unroll
                for (int k = 0; k < N; ++k)
                    e[k] = make_double2(q_invvol * shape<O>(xm, St::col(k)).s * shape<O>(ym, St::row(k)).s, target);
                double2* f = e + N;
                const double clight = 1.0;
                f[0] = make_double2(vx, 1.0);
                f[1] = make_double2(vy, 1.0);
                f[2] = make_double2(gamma_psi - 1.0, clight);
                f[3] = make_double2(gamma_psi, 1.0);
                f[4] = make_double2(charge_mass_ratio, psi_inv);
                f[5] = make_double2(1.0, 1.0);
            }
        } else if (lane < CHUNK) {   // an empty place: no cell inside
            if constexpr (KIND == EXPLICIT) {
                ent[lane][2 * S + 2] = make_double2(0.0, 0.0);
            } else {
#pragma unroll
                for (int k = 0; k < N; ++k) ent[lane][k] = make_double2(0.0, 0.0);
            }
        }
        __syncthreads();
        if constexpr (KIND == EXPLICIT) {
            const double qmr = charge_mass_ratio, dxi = g.dxi, dyi = g.dyi;
            const uint32_t mybit = part < PP ? 1u << off : 0u;
            const int mypart = part < PP ? part : 0;
#pragma unroll 1
            for (int e0 = 0; e0 < cnt; e0 += U * PP) {
                double2 X[U], Y[U], a[U], u[U], d[U], f0[U], f1[U];
                int c[U];
                bool in[U];
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    const double2* r = ent[e0 + q * PP + mypart];
                    X[q] = r[ox];
                    Y[q] = r[S + oy];
                    a[q] = r[2 * S];
                    u[q] = r[2 * S + 1];
                    d[q] = r[2 * S + 2];
                }
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    in[q] = (uint32_t(__double2loint(d[q].y)) & mybit) != 0u;
                    c[q] = in[q] ? __double2hiint(d[q].y) + shift : 0;
                    f0[q] = field[0][c[q]];
                    f1[q] = field[1][c[q]];
                }
                double sy[U], sx[U];
#pragma unroll
                for (int q = 0; q < U; ++q) {
                    const double Bz = f0[q].x, Ez = f0[q].y, ExmBy = f1[q].x, EypBx = f1[q].y;
                    const double q_invvol = a[q].x, psi_inv = a[q].y, vx = u[q].x, vy = u[q].y, gamma_psi = d[q].x;
                    // the reference's products and sums in its order; a factor -1 moves through a
                    // product and a + (-b) is a - b without a change of the result's bits
                    const double vxvy = vx * vy;
                    const double gx = gamma_psi - vx * vx, gy = gamma_psi - vy * vy;
                    const double ss = X[q].x * Y[q].x;
                    const double dsx = X[q].y * Y[q].x * dxi, sdy = X[q].x * Y[q].y * dyi;
                    const double A = (Ez * vy - ExmBy * vxvy + EypBx * gy) - Bz * vx;
                    const double B = (Ez * vx + ExmBy * gx - EypBx * vxvy) + Bz * vy;
                    sy[q] = q_invvol * (-ss * A * qmr * psi_inv + (dsx * vxvy - sdy * (gy - 1.0)));
                    sx[q] = q_invvol * (ss * B * qmr * psi_inv + (dsx * (gx - 1.0) - sdy * vxvy));
                }
#pragma unroll
                for (int q = 0; q < U; ++q) {
#pragma unroll
                    for (int p = 0; p < PP; ++p) {
                        if (in[q] && part == p) {
                            __hip_atomic_fetch_add(&sum[0][c[q]], sy[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                            __hip_atomic_fetch_add(&sum[1][c[q]], sx[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        }
                        __builtin_amdgcn_wave_barrier();
                    }
                }
            }
        } else {
            constexpr int PER = 64 / N < NSUM ? 64 / N : NSUM;   // components of one pass
#pragma unroll
            for (int q0 = 0; q0 < NSUM; q0 += PER) {
                int comp = -1, quantity = 0;
#pragma unroll
                for (int k = 0; k < NSUM; ++k)
                    if (part < PER && k == q0 + part) {
                        comp = cm.c[k];
                        quantity = cm.q[k];
                    }
                const uint32_t mybit = comp >= 0 ? 1u << off : 0u;
                double* acc = &sum[comp >= 0 ? q0 + part : 0][0];
#pragma unroll 1
                for (int e0 = 0; e0 < cnt; e0 += U) {
                    double2 cd[U], f[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        cd[u] = ent[e0 + u][off];
                        f[u] = ent[e0 + u][N + quantity];
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const double val = cd[u].x * f[u].x * f[u].y;
                        if (uint32_t(__double2loint(cd[u].y)) & mybit)
                            __hip_atomic_fetch_add(&acc[__double2hiint(cd[u].y) + shift], val, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_WORKGROUP);
                        __builtin_amdgcn_wave_barrier();
                    }
                }
            }
        }
    };

    // The window's entries of the colours of `mask` in the listed runs from run `from` on, by
    // index, into `found` until it is full; returns the run to go on with.
    unsigned present = 0u;   // colours in the window's tiles
    {
        const unsigned long long wx = ~0ull >> (64 - NW), wy = ~0ull >> (64 - NH);
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if ((((c >> 1) ? PX : ~PX) & wx) && (((c & 1) ? PY : ~PY) & wy)) present |= 1u << c;
    }
    auto collect = [&](unsigned mask, int from) -> int {
        const bool one = (mask & (mask - 1u)) == 0u;
        uint16_t* const into = one ? seq : found;
        int ncol[3];
        n = 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) ncol[c] = 0;
        auto load = [&](int t, uint32_t (&w)[BATCH]) {
#pragma unroll
            for (int q = 0; q < BATCH; ++q) {
                const long ip = t + q < nruns ? long(runs[t + q]) * RUN + lane : v.n;
                w[q] = ip < v.n ? v.cell[ip] : NO_CELL;
            }
        };
        uint32_t w[BATCH], wn[BATCH];
        load(from, w);
        int t = from;
        bool full = false;
        for (; t < nruns && !full; t += BATCH) {
            load(t + BATCH, wn);
#pragma unroll
            for (int q = 0; q < BATCH; ++q) {
                const unsigned x = unsigned(int(w[q] & xmask) - X0), y = unsigned(int(w[q] >> v.shift) - Y0);
                int c = 4;
                if (w[q] != NO_CELL && x < unsigned(NW) && y < unsigned(NH))
                    c = int((PX >> (x & 63)) & 1ull) * 2 + int((PY >> (y & 63)) & 1ull);
                const bool hit = c < 4 && ((mask >> c) & 1u);
                const unsigned long long h = __ballot(hit);
                if (h == 0ull) continue;
                if (hit) into[n + lanes_before(h)] = uint16_t(c << 13 | (t + q) << 6 | lane);
                n += __popcll(h);
                if (!one) {
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        if ((mask >> k) & 1u) ncol[k] += __popcll(__ballot(hit && c == k));
                }
                if (n > SEQ - RUN) {
                    full = true;
                    t += q + 1 - BATCH;
                    break;
                }
            }
#pragma unroll
            for (int q = 0; q < BATCH; ++q) w[q] = wn[q];
        }
        __syncthreads();
        if (one) return t;
        // by colour into seq: a stable counting sort
        int at[4] = {0, ncol[0], ncol[0] + ncol[1], ncol[0] + ncol[1] + ncol[2]};
        for (int e0 = 0; e0 < n; e0 += 64) {
            const int e = e0 + lane;
            const int id = e < n ? int(found[e]) : -1;
            const int c = id >> 13;
            int to = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (!((mask >> k) & 1u)) continue;
                const unsigned long long h = __ballot(c == k);
                if (c == k) to = at[k] + lanes_before(h);
                at[k] += __popcll(h);
            }
            if (id >= 0) seq[to] = uint16_t(id);
        }
        __syncthreads();
        return t;
    };
    auto run_sequence = [&] {
        Record r = fetch(lane);
#pragma unroll 1
        for (int e0 = 0; e0 < n; e0 += CHUNK) {
            const Record next = fetch(e0 + CHUNK + lane);
            process(r, min(CHUNK, n - e0));
            r = next;
        }
        __syncthreads();
    };
    // With linked particles in the window: colour by colour, KEEP particles at a time. Of those from
    // index `lo` on the lowest are taken, from the linked lists, whose order is that of chance, and from
    // the runs, which go by index; sorted, they are the sequence, and the next one starts where it
    // ends (`hi`). Every round walks the lists again: a lane follows one of HEADS lists of a bin, so
    // that a walk is as long as a bin has particles / HEADS, 8 loads after one another at 2 x 2 particles
    // per cell, three times for the window's bins (of 4 lists, 16 and twice: 300 and 308 us for all of
    // the current deposition at 511 x 511, but 534 and 408 us with 2000 particles more in one spot of
    // 127 x 127). Walks, sorts and records read out of order make the current deposition of a
    // plasma in random order take 231 instead of 111 us (511 x 511, 2 x 2 particles per cell). When
    // such a plasma's runs were all tested by every block, it took 15 ms.
    auto window_colour = [&](uint32_t w) -> int {
        const unsigned x = unsigned(int(w & xmask) - X0), y = unsigned(int(w >> v.shift) - Y0);
        if (w == NO_CELL || x >= unsigned(NW) || y >= unsigned(NH)) return 4;
        return int((PX >> (x & 63)) & 1ull) * 2 + int((PY >> (y & 63)) & 1ull);
    };
    // the first cnt keys sorted (bitonic, the next power of two of them)
    auto sort_keys = [&](int cnt) {
        int P = 64;
        while (P < cnt) P <<= 1;
        for (int t = cnt + lane; t < P; t += 64) key[t] = ~0u;
        __syncthreads();
        for (int k = 2; k <= P; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
#pragma unroll 4
                for (int t = lane; t < P / 2; t += 64) {
                    const int i = 2 * (t & ~(j - 1)) | (t & (j - 1));
                    const uint32_t a = key[i], c = key[i | j];
                    const bool up = (i & k) == 0;
                    key[i] = up == (a < c) ? a : c;
                    key[i | j] = up == (a < c) ? c : a;
                }
                __syncthreads();
            }
    };
    auto collect_linked = [&](int colour, uint32_t lo) -> uint32_t {
        constexpr int AHEAD = 8;
        uint32_t hi = ~0u;
        int cnt = 0;
        // the KEEP lowest of the keys so far
        auto cut = [&] {
            sort_keys(cnt);
            hi = uint32_t(__builtin_amdgcn_readfirstlane(int(key[KEEP])));
            cnt = KEEP;
            __syncthreads();
        };
        __syncthreads();
        for (int t0 = 0;; t0 += 64) {
            const bool last = t0 >= nlinks;   // room for the runs, too
            uint32_t p = t0 + lane < nlinks ? first_linked(t0 + lane) : 0u;
            do {
                uint32_t w = NO_CELL, after = 0u;
                if (p) {
                    w = v.cell[p - 1];
                    after = v.link()[p - 1];
                }
                if (cnt > (last ? KEEP : KEYS - 64)) cut();
                const bool hit = window_colour(w) == colour && p - 1 >= lo && p - 1 < hi;
                const unsigned long long h = __ballot(hit);
                if (hit) key[cnt + lanes_before(h)] = p - 1;
                cnt += __popcll(h);
                p = after;
            } while (__ballot(p != 0u) != 0ull);
            if (last) break;
        }
        __syncthreads();
        if (!listed) {
            pos = Pos{};
            pos.s0 = int(lo / SUPER);
            nruns = 0;
        }
        for (int t = 0;; t += AHEAD) {
            if (t >= nruns) {
                if (pos.end) break;
                nruns = find_runs();
                t = 0;
            }
            uint32_t w[AHEAD];
#pragma unroll
            for (int q = 0; q < AHEAD; ++q) {
                const long ip = t + q < nruns ? long(runs[t + q]) * RUN + lane : v.n;
                w[q] = ip < v.n && ip >= long(lo) && ip < long(hi) ? v.cell[ip] : NO_CELL;
            }
            bool full = false;
#pragma unroll
            for (int q = 0; q < AHEAD; ++q) {
                if (full || t + q >= nruns) continue;
                const uint32_t first = uint32_t(__builtin_amdgcn_readfirstlane(runs[t + q])) * RUN;
                if (first >= hi || cnt > KEYS - RUN) {
                    hi = min(hi, first);
                    full = true;
                    continue;
                }
                const bool hit = window_colour(w[q]) == colour;
                const unsigned long long h = __ballot(hit);
                if (hit) key[cnt + lanes_before(h)] = first + unsigned(lane);
                cnt += __popcll(h);
            }
            if (full) break;
        }
        __syncthreads();
        sort_keys(cnt);
        // those below hi, KEEP at most
        int m = 0;
        for (int t0 = 0; t0 < cnt; t0 += 64) m += __popcll(__ballot(t0 + lane < cnt && key[t0 + lane] < hi));
        if (m > KEEP) {
            m = KEEP;
            hi = uint32_t(__builtin_amdgcn_readfirstlane(int(key[KEEP])));
        }
        for (int t = lane; t < m; t += 64) seq_ip[t] = key[t];
        n = m;
        __syncthreads();
        return hi;
    };
    // All colours at once when their entries fit, otherwise colour by colour; `all`: one list
    // holds every run of the window.
    const bool all = pos.end;
    bool together = all && !linked;   // for the first sequence
    unsigned mask = present;
    int t = 0, colour = 0;
    uint32_t lo = 0u;   // linked: where the next sequence starts, all ones after a colour's last
    while (true) {
        if (linked) {
            if (lo == ~0u) {
                ++colour;
                lo = 0u;
            }
            while (colour < 4 && !((present >> colour) & 1u)) ++colour;
            if (colour > 3) break;
            lo = collect_linked(colour, lo);
        } else {
            // the next entries of this colour
            while (!together && colour < 4) {
                mask = present & (1u << colour);
                if (mask && t < nruns) break;
                if (mask && !pos.end) {
                    nruns = find_runs();
                    t = 0;
                    continue;
                }
                ++colour;
                t = 0;
                if (!all) {
                    pos = Pos{};
                    nruns = 0;
                }
            }
            if (colour > 3) break;
            t = collect(mask, t);
            if (together && t < nruns) {   // too many: colour by colour from the first run
                together = false;
                t = 0;
                continue;
            }
        }
        run_sequence();
        if (together) break;
    }
    __syncthreads();
    for (int t = lane; t < BW * BH; t += 64) {
        const int i = i0 + t % BW, j = j0 + t / BW, c = t / BW * BS + t % BW;
        if (i > g.nx - 1 + g.ng || j > g.ny - 1 + g.ng) continue;
        const long k = g.idx(i, j);
        if constexpr (KIND == EXPLICIT) {
            store[cm.c[4] * ps + k] = sum[0][c];
            store[cm.c[5] * ps + k] = sum[1][c];
        } else {
#pragma unroll
            for (int q = 0; q < NSUM; ++q)
                if (cm.c[q] >= 0) store[cm.c[q] * ps + k] = sum[q][c];
        }
    }
}

__global__ __launch_bounds__(256) void k_clear_counts(int32_t* __restrict__ a, long n) {
    const long t = long(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < n) a[t] = 0;
}

int bits(long v) {
    int b = 0;
    while ((1L << b) <= v) ++b;
    return b;
}

// The blocks of a grid: 16 x 8 cells, 8 x 8 or 8 x 4, the largest of which there are as many as
// the CUs hold wavefronts at once, or the smallest. A larger block's window holds fewer
// particles that other blocks take as well; too few blocks leave the chip idle, and a wavefront
// takes its particles one after the other. Measured at order 2, current + explicit in us, with
// 16 x 8, 8 x 8 and 8 x 4 cells:
//   near the lattice, one particle per cell: 63 x 63 53, 39, 32; 127 x 127 62, 48, 41;
//     255 x 255 72, 64, 56; 383 x 383 87, 76, 96; 511 x 511 102, 117, 144 (2 x 2 per cell 300, 316, 347);
//   crossing orbits, 2 x 2 per cell: 255 x 255 274, 201, 176; 383 x 383 321, 272, 260;
//     511 x 511 383, 370, 387, where the next smaller blocks would be 4 % faster: the line stays
//     where the lattice, the usual state, puts it.
constexpr long FILL = 8 * 256;
void blocks(const Geom& g, OrdView& v) {
    const int sizes[3][2] = {{4, 3}, {3, 3}, {3, 2}};
    for (const auto& s : sizes) {
        v.lw = s[0];
        v.lh = s[1];
        v.nbx = (g.ldx + (1 << v.lw) - 1) >> v.lw;
        v.nby = (g.ldy + (1 << v.lh) - 1) >> v.lh;
        if (long(v.nbx) * v.nby >= FILL) break;
    }
}

// Blocks that a listed run meets, at most; a run that meets more has its particles linked. When
// all runs met LIST * blocks / runs of them, the lists would be full on average, and full lists
// make a block look for its runs among all boxes, which costs more than links do: the line lies an
// eighth below, and not below 20, for a run of a lattice meets up to 9 and one of crossing orbits
// up to 20 whatever their number. Measured with runs spread by random displacements (511 x 511,
// 2 x 2 particles per cell, current + explicit in us; listed unless they meet 512 blocks, with this
// line, with one at 16): 7 cells 540, 510, 630; 10 cells 930, 720, 790; 14 cells 1060, 1250, 720;
// 20 cells 1290, 730, 670; 40 cells 2260, 710, 700.
constexpr long NARROW = 20;

// cells are counted in [bxlo, bxlo + wx) x [bylo, bylo + wy)
OrdView view(const hpq_ctx* c, const PlasmaOrder& L, long n, int& wx, int& wy) {
    const Geom& g = c->g;
    OrdView v{};
    v.bxlo = -g.ng - 6;
    v.bylo = -g.ng - 6;
    wx = OrdView::cells_found(g.nx, g.ng);
    wy = OrdView::cells_found(g.ny, g.ng);
    v.shift = bits(wx);
    if (v.shift + bits(wy) > 31) throw HpqError(HPQ_E_UNSUPPORTED, "ordered deposition: more than 2^31 cells");
    v.T = c->p.tile_size > 0 ? c->p.tile_size : 32;
    v.ntx = (g.ldx + v.T - 1) / v.T;
    v.nty = (g.ldy + v.T - 1) / v.T;
    v.n = n;
    v.nrun = int((n + RUN - 1) / RUN);
    v.nsuper = int((n + SUPER - 1) / SUPER);
    blocks(g, v);
    // the current deposition's stencil starts at most 1 below the cell and ends at most 2 above,
    // the derivative ones' at most 2 below and 3 above
    v.mlo = 3;
    v.mhi = 2;
    v.rec = L.rec;
    v.cell = L.cell;
    v.rbox = reinterpret_cast<const int4*>(L.boxes);
    v.sbox = v.rbox + v.nrun;
    const long nblk = long(v.nbx) * v.nby;
    v.narrow = int(std::min<long>(std::max(NARROW, 7 * LIST * nblk / (8 * long(std::max(v.nrun, 1)))), INT_MAX));
    v.count = L.count + PASS_WORDS;
    v.list = L.list;
    return v;
}

// records, cells and boxes of the particles for cells floor(xmid + BASE / 2)
template <int BASE, bool QSA>
OrdView make_records(hpq_ctx* c, const hpq_plasma* p, double charge_invvol) {
    PlasmaOrder& L = c->ord_plasma;
    const Geom& g = c->g;
    const long n = p->n;
    grow(L.rec, L.rec_cap, n * REC);
    grow(L.cell, L.cell_cap, 2 * n);
    grow(L.boxes, L.boxes_cap, 4 * ((n + RUN - 1) / RUN + (n + SUPER - 1) / SUPER));
    int wx, wy;
    OrdView v = view(c, L, n, wx, wy);
    const long nblk = long(v.nbx) * v.nby;
    const long words = PASS_WORDS + 2 * (nblk + 1) + 2L * HEADS * OrdView::bins(g.nx, g.ng) * OrdView::bins(g.ny, g.ng);
    grow(L.list, L.list_cap, nblk * LIST);
    grow(L.count, L.count_cap, words);
    v = view(c, L, n, wx, wy);
    // the first pass, and the one after a pass whose deposition was not launched
    if (L.unclear) hipLaunchKernelGGL(k_clear_counts, grid1d(words, 256), dim3(256), 0, c->stream, L.count, words);
    L.unclear = true;
    hipLaunchKernelGGL((k_records<BASE, QSA>), dim3(unsigned(v.nsuper)), dim3(REC_T), 0, c->stream, g, *p, v, wx, wy,
                       charge_invvol, c->p.max_qsa, L.rec, L.cell, reinterpret_cast<int4*>(L.boxes),
                       reinterpret_cast<int4*>(L.boxes) + v.nrun, L.count + PASS_WORDS, L.list,
                       const_cast<unsigned long long*>(v.head()), L.cell + n, L.count + MADE, c->d_count);
    HPQ_HIP(hipGetLastError());
    return v;
}

template <int KIND, int T, int O, int NSUM>
void launch_deposit(hpq_ctx* c, const OrdView& v, double* store, const Comps& cm, double ratio) {
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(unsigned(v.nbx * v.nby)), dim3(64), 0, c->stream, c->g, v, store, cm, ratio,
                           c->ord_plasma.count + NEXT);
    };
    if (v.lw == 4) launch(k_deposit_ordered<KIND, T, O, NSUM, 16, 8>);
    else if (v.lh == 3) launch(k_deposit_ordered<KIND, T, O, NSUM, 8, 8>);
    else launch(k_deposit_ordered<KIND, T, O, NSUM, 8, 4>);
    HPQ_HIP(hipGetLastError());
    c->ord_plasma.unclear = false;
}

void check_count(const hpq_plasma* p) {
    if (p->n > INT32_MAX) throw HpqError(HPQ_E_INVALID, "ordered deposition: more than 2^31-1 particles");
}

}  // namespace

void plasma_order_free(PlasmaOrder& L) {
    for (void* q : {(void*)L.rec, (void*)L.cell, (void*)L.boxes, (void*)L.count, (void*)L.list})
        if (q) (void)hipFree(q);
    L = PlasmaOrder{};
}

// ::DepositCurrent in the CPU build's order; the records it makes describe the particle state
// for the explicit deposition that follows on it
void deposit_current_ordered(hpq_ctx* c, const hpq_plasma* p, double* store, const int32_t* comps, bool ions) {
    const Geom& g = c->g;
    PlasmaOrder& L = c->ord_plasma;
    L.valid = false;
    if (p->n <= 0) return;
    check_count(p);
    const double charge = ions ? -c->p.plasma_charge : c->p.plasma_charge;
    const double mu0 = 1.0;
    const double invvol = g.dx * g.dy * g.dxi * g.dyi;
    const double cmr = charge * mu0 / c->p.plasma_mass;
    Comps cm{{-1, -1, -1, -1, -1, -1}, {0, 0, 0, 0, 0, 0}};
    int nsum = 0;
    for (int q = 0; q < 6; ++q)
        if (comps[q] >= 0) {
            cm.c[nsum] = comps[q];
            cm.q[nsum++] = q;
        }
    TraceScope ts(c, HPQ_TRACE_DEPOSIT);
    dispatch_order(c->p.depos_order, [&](auto O) {
        constexpr int o = decltype(O)::value;
        const OrdView v = make_records<shape_base<o>(), true>(c, p, charge * invvol);
        // the usual four components (jx, jy, chi, rhomjz) leave room for more wavefronts per CU
        if (nsum <= 4) launch_deposit<CURRENT, 0, o, 4>(c, v, store, cm, cmr);
        else launch_deposit<CURRENT, 0, o, 6>(c, v, store, cm, cmr);
        L.base = shape_base<o>();
    });
    L.valid = !ions;
    L.x = p->x;
    L.n = p->n;
}

// ::ExplicitDeposition in the CPU build's order; reuses the records of the current deposition
// on the same particle state when the start cells share their floor
void explicit_deposition_ordered(hpq_ctx* c, const hpq_plasma* p, double* store) {
    const Geom& g = c->g;
    const Layout& Ly = c->L;
    PlasmaOrder& L = c->ord_plasma;
    if (p->n <= 0) return;
    check_count(p);
    const double mu0 = 1.0;
    const double invvol = g.dx * g.dy * g.dxi * g.dyi;
    const double qimu0 = c->p.plasma_charge * invvol * mu0;
    const double qmr = c->p.plasma_charge / c->p.plasma_mass;
    const Comps cm{{Ly.Bz, Ly.Ez, Ly.ExmBy, Ly.EypBx, Ly.Sy, Ly.Sx}, {}};
    TraceScope ts(c, HPQ_TRACE_EXPLICIT_DEPOSIT);
    dispatch_order(c->p.depos_order, [&](auto O) {
        constexpr int o = decltype(O)::value;
        auto run = [&](auto TT) {
            constexpr int t = decltype(TT)::value;
            OrdView v;
            if (L.valid && L.x == p->x && L.n == p->n && L.base == dshape_base<t, o>()) {
                int wx, wy;
                v = view(c, L, p->n, wx, wy);
            } else {
                v = make_records<dshape_base<t, o>(), false>(c, p, qimu0);
                L.valid = true;
                L.base = dshape_base<t, o>();
                L.x = p->x;
                L.n = p->n;
            }
            launch_deposit<EXPLICIT, t, o, 2>(c, v, store, cm, qmr);
        };
        const int type = c->p.derivative_type;
        if (type == 0) run(std::integral_constant<int, 0>{});
        else if (type == 1) run(std::integral_constant<int, 1>{});
        else run(std::integral_constant<int, 2>{});
    });
}

}  // namespace hpq
