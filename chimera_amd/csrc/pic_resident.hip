// pic_resident.hip -- particle kernels of device-resident simulations.
//
// Particles live in structure-of-arrays form: coordinate component c of
// particle i at coord[c*ld + i] (likewise momenta), weights[i].  Every pointer
// is device memory; calls are asynchronous on the library stream.
//
//  * chimera_soa_push_coords   leap-frog push (particle_tools.f90:58-82)
//  * chimera_soa_dep_curr/dens deposition without the ghost fold, which the
//                              forward FB transform applies when it reads
//                              row 1 (grid_deps.f90:80-85, :144-145)
//  * chimera_soa_gather_push   gather (grid_deps.f90:149-217) + analytic
//                              undulator (devices.f90:162-203) + Boris push
//                              (particle_tools.f90:18-56) in one pass, with
//                              the reference's order: field on particles is
//                              zeroed, gathered, device fields added, pushed
//                              (chimera_main.py:130-151, :91-92)
//  * chimera_soa_compact       stable removal of particles outside lims
//                              (particle_tools.f90:130-153 + the permutation
//                              gathers of species.py:385-398)
#include <climits>
#include <type_traits>

#include "common.hpp"
#include "fb_kernels.hpp"
#include "pic_device.hpp"
#include "sort.hpp"
#include "../../include/chimera_hip.h"

namespace chimera {

// NMOD = number of azimuthal modes, a template parameter so that every mode
// index is a constant and the per-particle phases stay in registers.
// R: precision of momenta, weights and fields (double, or float in mixed
// precision, where the Boris push runs in FP32); positions and the cell
// geometry are FP64.
//
// A block takes GP_T consecutive (cell-ordered) particles, one per thread,
// finds the bounding box of their cells, and copies the field nodes of that
// box (all six components and modes) into LDS with coalesced loads; each
// particle then reads its 4 x 6 x NMOD values from LDS instead of from L2 (at
// 16 particles per cell the block's 256 particles share 17 x 3 nodes).  The
// momenta load with the positions, in flight while the tile loads.  A box
// too large for GP_LDS_BYTES reads the field from global memory.  The values
// and the order of the sums are the same either way.
constexpr int GP_T = 256, GP_LDS_BYTES = 24 * 1024;

__device__ __forceinline__ int wave_min(int v) {
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ int wave_max(int v) {
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ int block_min_max(int v, bool is_max, int (*red)[GP_T / 64], int q) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    v = is_max ? wave_max(v) : wave_min(v);
    if (lane == 0) red[q][wv] = v;
    return v;
}

template <int NMOD, typename R>
__global__ void __launch_bounds__(GP_T) k_gather_push(const double* __restrict__ coord, PStride sx, R* __restrict__ u,
                                                      PStride su, const R* __restrict__ w,
                                                      const cplx_t<R>* __restrict__ Fld, GridGeom g_in, double push_dt,
                                                      ExtDevices devs, int np) {
    typedef cplx_t<R> C;
    constexpr int NC = 6 * NMOD;   // (component, mode) planes
    __shared__ C tile[GP_LDS_BYTES / sizeof(C)];
    __shared__ int red[4][GP_T / 64];
    __shared__ int box[4];
    const int tid = threadIdx.x;
    const int ip = xcd_block(blockIdx.x, gridDim.x) * GP_T + tid;
    const bool live = ip < np;
    const GridGeom g = frame_geom(g_in);
    double xp = 0, yp = 0, zp = 0;
    R m[3] = {0, 0, 0};
    if (live) {
        xp = coord[sx.at(ip, 0)];
        yp = coord[sx.at(ip, 1)];
        zp = coord[sx.at(ip, 2)];
        // the momenta load now, so that it is in flight while the field tile loads
        m[0] = u[su.at(ip, 0)];
        m[1] = u[su.at(ip, 1)];
        m[2] = u[su.at(ip, 2)];
    }
    PartGeom pg;
    const bool has = live && w[ip] != 0 && part_geom(pg, xp, yp, zp, g, +1.0);
    block_min_max(has ? (int)pg.ix : INT_MAX, false, red, 0);
    block_min_max(has ? (int)pg.ix : INT_MIN, true, red, 1);
    block_min_max(has ? (int)pg.ir : INT_MAX, false, red, 2);
    block_min_max(has ? (int)pg.ir : INT_MIN, true, red, 3);
    __syncthreads();
    if (tid < 4) {
        int v = red[tid][0];
        for (int k = 1; k < GP_T / 64; k++) v = (tid & 1) ? max(v, red[tid][k]) : min(v, red[tid][k]);
        box[tid] = v;
    }
    __syncthreads();
    const int64_t sr = g.nx + 1, sm = sr * (g.nr + 1), sl = sm * NMOD;
    const int bx0 = box[0], br0 = box[2];
    const int TX = box[1] >= box[0] ? box[1] - box[0] + 2 : 0, TR = box[3] >= box[2] ? box[3] - box[2] + 2 : 0;
    const int nt = TX * TR * NC;
    const bool tiled = nt > 0 && (int64_t)nt * (int64_t)sizeof(C) <= GP_LDS_BYTES;
    if (tiled) {
        // plane lm = l*NMOD + m of the field starts at lm*sm (sl = NMOD*sm)
        for (int e = tid; e < nt; e += GP_T) {
            const int xx = e % TX, rest = e / TX, rr = rest % TR, lm = rest / TR;
            tile[e] = Fld[(bx0 + xx) + (int64_t)(br0 + rr) * sr + (int64_t)lm * sm];
        }
    }
    __syncthreads();
    if (!live) return;
    R f[6] = {0, 0, 0, 0, 0, 0};
    if (has) {
        if (tiled) {
            const C* base = tile + (pg.ix - bx0) + (pg.ir - br0) * TX;
            const int tsl = TX * TR;
            for (int l = 0; l < 6; l++) {
                R acc = 0;
#pragma unroll
                for (int iO = 0; iO < NMOD; iO++) {
                    const C* fl = base + (l * NMOD + iO) * tsl;
                    for (int b = 0; b < 2; b++)
                        for (int a = 0; a < 2; a++) {
                            const C pc = cconv<R>(crs(pg.S[1][b] * pg.S[0][a], pg.ph[iO]));
                            const C v = fl[a + b * TX];
                            acc += pc.x * v.x - pc.y * v.y;
                        }
                }
                f[l] = acc;
            }
        } else {
            const C* base = Fld + pg.ix + pg.ir * sr;
            for (int l = 0; l < 6; l++) {
                R acc = 0;
#pragma unroll
                for (int iO = 0; iO < NMOD; iO++) {
                    const C* fl = base + iO * sm + l * sl;
                    for (int b = 0; b < 2; b++)
                        for (int a = 0; a < 2; a++) {
                            const C pc = cconv<R>(crs(pg.S[1][b] * pg.S[0][a], pg.ph[iO]));
                            const C v = fl[a + b * sr];
                            acc += pc.x * v.x - pc.y * v.y;
                        }
                }
                f[l] = acc;
            }
        }
    }
    if (devs.n) ext_fields<R>(devs, xp, yp, zp, f);
    boris<R>(m, f, (R)(0.5 * push_dt));
    for (int c = 0; c < 3; c++) u[su.at(ip, c)] = m[c];
}

// ------------------------------------------------------------------ fused push + deposition
//
// A block of four waves takes a group of DEP_T * PPL consecutive particles, PPL
// per lane:
//  1. Every lane loads its particles once (coalesced), pushes them
//     (particle_tools.f90:58-82), finds their cells, weights and phases for J
//     (half-step positions) and rho (new positions), and leaves J's in LDS for
//     its wave; the block reduces the node bounding box of both deposits.
//  2. Each wave cuts its particles into segments of one cell, listed in LDS
//     from ballots.  A lane takes one (segment, component, node row of the
//     cell): it sums the particles of the segment on the row's two nodes, all
//     modes, in FP64 registers and adds the sums to the block's LDS tile (real
//     planes: Re of mode 0, then Re and Im of each mode) with ds_add_f64, the
//     waves one after the other.  rho follows J through the same LDS.
//  3. The block hands the tile on:
//      * a tile of at most dep_slot values and no more rows than columns (or
//        DEP_SLOT_R) goes with plain stores, as it is, into the group's own
//        slot, with a descriptor (first node row, first node column, width,
//        rows); k_dep_combine then adds the slots into the grid, so no global
//        atomics;
//      * any other tile is added to the grid with one global atomic per node
//        value; the planes take as many passes as the LDS needs (all four
//        components at once, J then rho, or one component at a time);
//      * a box with no room even for one component's planes (a group that
//        spans the end of one cell row and the start of the next) sends each
//        segment's sums to the grid with global atomics.
// Deposits are unfolded; the forward FB transform applies the ghost fold.
//
// What bounds it: about equally the 104 bytes per particle in and out of HBM
// (with the slots 8.9 GB of traffic for 67.0 M electrons at four modes), the
// segments' arithmetic and their LDS reads and adds; three blocks of a CU share
// them.  There it takes 3.0 ms (2.8 without the fixed order of the adds), and the
// combine 0.9; one pass per component over particles re-read from memory (46 GB)
// took 5.5, with a combine of 1.2.  Mixed precision, 16.7 M at three modes: 0.82 +
// 0.11 ms, before 1.24 + 0.13 and 70 us to sort the slots.  (Loading the next group during the deposit of one, a
// block taking several, changed nothing: the other blocks already hide it.)

template <typename RT>
struct DepArgsT {
    typedef cplx_t<RT> C;
    double* x;          // positions (3, ld), updated when push
    double* xh;         // half-step positions (3, ld): written when push, read otherwise
    const RT* u;        // momenta (3, ld)
    const RT* w;
    int64_t ld;
    int np;
    int push;
    double dt;
    GridGeom gJ, gR;    // geometry for J (leftX at the current deposit) and rho
    C* J;               // (nx+1, nr+1, M, 3) or null
    C* R;               // (nx+1, nr+1, M) or null
    RT* slot;           // [group][dep_slot]: J's components, then rho, each 2M-1 planes of width * rows
                        // values, starting on an even value
    int4* desc;         // [group]: (first node row or -1, first node column, width, rows)
    uint32_t* mask;     // [nr+1][words]: bit b of a node row: a slot of groups 64b..64b+63 covers it (nullable)
    int words;          // 32-bit words per row of mask
    int ngroups;
    int vec;            // particle arrays allow PPL-wide vector access (ld % PPL == 0, aligned bases)
};

constexpr int DEP_T = 256, DEP_WAVES = DEP_T / 64;
// LDS tile in doubles: with the particle data of PPL = 2 (32 KiB) three blocks
// fill the 160 KiB of a CU (allocated 1280 bytes at a time).  At four modes it
// holds J and rho on 85 nodes (512 cell-sorted particles at 16 per cell span
// 33 x 2), J on 114 (in the lattice's own order they span 33 x 3).
constexpr int DEP_POOL = 2400;
// values of a slot: at two modes 341 nodes, more than the 65 x 4 of a sparse
// bunch's 256 particles (4 per cell, drifting over a row boundary); at one mode
// 528, more than the 257 x 2 of one particle per cell, in half the memory
// (serve.slot_bytes counts it)
constexpr int dep_slot(int nmod) { return nmod == 1 ? 2112 : 4096; }
// node rows of a slot that is narrower than that (others: no more rows than
// columns, so 64 at most).  A tall, narrow tile (particles column by column, as a
// RandCell species draws them) is cheaper as global atomics: a wave of the combine would
// meet a slot of two columns for each of its 64 (65536 particles, 16 per cell in
// 128 x 32 cells, FP64, the whole deposit: two modes 118 us with slots and 41
// without, four modes 153 and 46, eight modes 797 and 55).
constexpr int DEP_SLOT_R = 4;
constexpr uint32_t DEP_SKIP = 0xFFFFFFFFu;

__device__ __forceinline__ void lds_add(double* p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// LDS written by some lanes of a wave and read by others of the same wave
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Minimum / maximum over a wave, in lane 63 (row shifts and row broadcasts; a
// lane without a source keeps its own value).
template <bool MAX>
__device__ __forceinline__ int wave_reduce63(int v) {
    auto op = [](int a, int b) { return MAX ? max(a, b) : min(a, b); };
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x111, 0xf, 0xf, false));
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x112, 0xf, 0xf, false));
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x114, 0xf, 0xf, false));
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x118, 0xf, 0xf, false));
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));
    return v;
}

// g = sqrt(a) and h = 1/sqrt(a) for a in [1e-280, 1e300], to about one unit in
// the last place: the hardware estimate (23 bits) refined by two coupled
// Newton steps (Goldschmidt's form), and a residual correction of g.
__device__ __forceinline__ void sqrt_rsqrt(double a, double& g, double& h) {
    const double y = __builtin_amdgcn_rsq(a);
    g = a * y;
    h = 0.5 * y;
    double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    g = fma(fma(-g, g, a), h, g);
    h = h + h;
}

// Cell (ix, ir), linear weights s = (x, r) of the upper nodes and phase
// p1 = (y - i z)/r (0 at r = 0) of one particle (grid_deps.f90:41-66), under
// the conditions of part_geom.
__device__ __forceinline__ bool dep_geom(double xp, double yp, double zp, const GridGeom& g, int& ix, int& ir,
                                         double2& s, double2& p1) {
    const double r2 = yp * yp + zp * zp;
    double rp, inv;
    sqrt_rsqrt(r2, rp, inv);
    if (!(r2 >= 1e-280)) {          // on the axis, or not a number
        rp = sqrt(r2);
        inv = rp > 0.0 ? 1.0 / rp : 0.0;
    }
    const double fx = (xp - g.leftX) * g.dx_inv, fr = (rp - g.r0) * g.dr_inv;
    if (!(rp < g.rmax) || !(fx >= 0.0 && fx < (double)g.nx) || !(fr >= 0.0 && fr < (double)g.nr)) return false;
    const double fix = floor(fx), fir = floor(fr);
    ix = (int)fix;
    ir = (int)fir;
    s = cmk(fx - fix, (rp - g.Rgrid[ir]) * g.dr_inv);
    p1 = cmk(yp * inv, -zp * inv);
    return true;
}

// One wave's LDS: its particles' weights, phases, charges and cells, and its
// segments.  Particle p sits at p + p/16: cells of 16 particles would otherwise
// start on one bank.
template <int PPL>
struct DepWave {
    static constexpr int WP = 64 * PPL, N = WP + WP / 16;
    double2 s[N], p1[N];
    double q[3][N + 7];
    uint32_t cell[WP];
    uint16_t seg[WP + 8];
    __device__ static int pos(int p) { return p + (p >> 4); }
};

// Segments of the wave's particles (keys of this lane's PPL particles in key):
// cut at every change of cell and every `run` particles, with the shortest run
// that keeps all (segment, component, node row) triples in one round of the 64
// lanes.  Returns their number; seg[i] is the first particle of segment i,
// seg[number] = WP.
template <int PPL, int NCOMP>
__device__ __forceinline__ int dep_segments(DepWave<PPL>& L, const uint32_t (&key)[PPL]) {
    constexpr int BUDGET = 32 / NCOMP, WP = DepWave<PPL>::WP;
    const int lane = threadIdx.x & 63;
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t prev = (uint32_t)__builtin_amdgcn_update_dpp((int)DEP_SKIP, (int)key[PPL - 1], 0x138, 0xf, 0xf, false);
    bool head[PPL];
    int nh = 0;
#pragma unroll
    for (int k = 0; k < PPL; k++) {
        head[k] = key[k] != prev;
        prev = key[k];
        nh += __popcll(__ballot(head[k]));
    }
    int run = 4, inv = 65536 / 4;                 // p / run = (p * inv) >> 16 for p < 128
    while (run < WP && nh + (((WP - 1) * inv) >> 16) > BUDGET) {
        run += run >> 1;
        inv = (65536 + run - 1) / run;
    }
    int nseg = 0, at = 0;
#pragma unroll
    for (int k = 0; k < PPL; k++) {
        const int p = lane * PPL + k;
        head[k] = head[k] || p == ((p * inv) >> 16) * run;
        const uint64_t b = __ballot(head[k]);
        nseg += __popcll(b);
        at += __popcll(b & below);
    }
#pragma unroll
    for (int k = 0; k < PPL; k++) {
        const int p = lane * PPL + k;
        L.cell[p] = key[k];
        if (head[k]) L.seg[at++] = (uint16_t)p;
    }
    if (lane == 0) L.seg[nseg] = (uint16_t)WP;
    wave_lds_fence();
    return nseg;
}

// The wave's segments into components c0..c0+NCP-1 (charges L.q[c0..]): to the
// tile (pns values per component: planes of nn nodes, rows of TX; key = node of
// the cell's lower corner), or, untiled, straight to the grid (key = node offset
// in a mode plane).  The lanes of one ds_add_f64 mostly add to different nodes.
// (With all four corners in a lane the segments had to be cut shorter to fill
// the lanes, and several of one cell collided on every add.)
//
// The waves add to the tile in turn, a round of 64 lanes each, so that its sums
// have the same order in every call: a barrier between two turns, and as many
// rounds as the block's wave with the most segments has (nsegs: the number of
// each, exchanged at the first barrier).  No barrier after the last turn.  On
// 67.0 M electrons at four modes, 10 steps after a sort, 4.13 ms with the combine; unordered
// 3.82, but with other last bits in every call.  (Tried: the even waves and then
// the odd ones where their boxes allow it, 4.11; a wave waiting for the waves
// that share nodes with it alone, by counters in LDS, 4.05; the odd waves
// keeping the sums of shared nodes in registers until the others are done, 4.25.)
template <int NMOD, int NCP, int PPL, typename R>
__device__ __forceinline__ void dep_pass(DepWave<PPL>& L, int wv, int nseg, int* nsegs, int c0, bool tiled,
                                         double* tile, int pns, int nn, int TX, cplx_t<R>* grid, int64_t sr, int64_t sm,
                                         int64_t sl) {
    constexpr int PL = 2 * NMOD - 1;
    const int nt = nseg * (2 * NCP);
    int rounds = (nt + 63) >> 6;          // of this wave; at least one
    if (tiled && (threadIdx.x & 63) == 0) nsegs[wv] = nseg;
    for (int r = 0, t = threadIdx.x & 63; r < rounds; r++, t += 64) {
        const bool in = t < nt;
        const int sg = in ? t / (2 * NCP) : 0, rem = in ? t - sg * (2 * NCP) : 0, c = rem >> 1;
        const bool up = rem & 1;
        const int pb = L.seg[sg], pe1 = L.seg[sg + 1];
        const uint32_t key = L.cell[pb];
        const bool on = in && key != DEP_SKIP;
        const int pe = on ? pe1 : pb;
        const double* q = L.q[c0 + c];
        double acc[PL][2];
#pragma unroll
        for (int i = 0; i < PL; i++) acc[i][0] = acc[i][1] = 0.0;
        for (int p = pb; p < pe; p++) {
            const int o = DepWave<PPL>::pos(p);
            const double2 s = L.s[o], p1 = L.p1[o];
            const double qp = q[o] * (up ? s.y : 1.0 - s.y);
            const double w0 = 1.0 - s.x, w1 = s.x;
            acc[0][0] += w0 * qp;
            acc[0][1] += w1 * qp;
            double2 pv = crs(qp, p1);
#pragma unroll
            for (int m = 1; m < NMOD; m++) {
                acc[2 * m - 1][0] += w0 * pv.x;
                acc[2 * m - 1][1] += w1 * pv.x;
                acc[2 * m][0] += w0 * pv.y;
                acc[2 * m][1] += w1 * pv.y;
                if (m + 1 < NMOD) pv = cmul(pv, p1);
            }
        }
        if (tiled) {
            double* tp = tile + c * pns + key + (up ? TX : 0);
            for (int w = 0; w < DEP_WAVES; w++) {
                if (w == wv && on) {
#pragma unroll
                    for (int i = 0; i < PL; i++)
#pragma unroll
                        for (int k = 0; k < 2; k++) lds_add(tp + i * nn + k, acc[i][k]);
                }
                if (w + 1 < DEP_WAVES) __syncthreads();
            }
            if (r == 0) {
                int n = 0;
#pragma unroll
                for (int i = 0; i < DEP_WAVES; i++) n = max(n, nsegs[i]);
                rounds = __builtin_amdgcn_readfirstlane((n * (2 * NCP) + 63) >> 6);
            }
            if (r + 1 < rounds) __syncthreads();
        } else if (on) {
#pragma unroll
            for (int m = 0; m < NMOD; m++)
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    R* dst = reinterpret_cast<R*>(grid + (c0 + c) * sl + m * sm + key + k + (up ? sr : 0));
                    unsafeAtomicAdd(dst, (R)acc[m ? 2 * m - 1 : 0][k]);
                    // the imaginary part of mode 0 is 0 times the real one
                    const double im = m ? acc[2 * m][k] : 0.0 * acc[0][k];
                    if (m || im != 0.0) unsafeAtomicAdd(dst + 1, (R)im);
                }
        }
    }
}

// ncp components of the tile to the group's slot, or, without one, to the grid;
// the tile is left zero for the next pass.
template <int NMOD, typename R>
__device__ __forceinline__ void dep_writeout(double* tile, int ncp, int pns, int nn, int TX, R* slot, cplx_t<R>* grid,
                                             int64_t sr, int64_t sm) {
    typedef R rv2 __attribute__((ext_vector_type(2)));
    const int n = ncp * pns;
    if (slot) {
        for (int i = 2 * threadIdx.x; i < n; i += 2 * DEP_T) {     // pns is even
            const double2 v = *reinterpret_cast<const double2*>(tile + i);
            *reinterpret_cast<double2*>(tile + i) = cmk(0.0, 0.0);
            rv2 t;
            t[0] = (R)v.x, t[1] = (R)v.y;
            *reinterpret_cast<rv2*>(slot + i) = t;
        }
        return;
    }
    for (int i = threadIdx.x; i < n; i += DEP_T) {
        const double v = tile[i];
        tile[i] = 0.0;
        if (v == 0.0) continue;      // (the odd value between components among them)
        const int c = i / pns, at = i - c * pns, k = at / nn, node = at - k * nn, rr = node / TX, xx = node - rr * TX;
        R* dst = reinterpret_cast<R*>(grid + (int64_t)(c * NMOD + (k + 1) / 2) * sm + xx + rr * sr);
        unsafeAtomicAdd(dst + (k > 0 && (k & 1) == 0 ? 1 : 0), (R)v);
        if (k == 0 && 0.0 * v != 0.0) unsafeAtomicAdd(dst + 1, (R)(0.0 * v));    // Im of mode 0: 0 times Re
    }
}

// R: precision of momenta, weights and grids (double, or float in mixed
// precision).  Positions, the push and the cell geometry stay FP64; each
// corner contribution is formed and summed in FP64, and the LDS tile is FP64
// in both precisions, rounded to R when it leaves the block.
template <int NMOD, typename R, int PPL>
__global__ void __launch_bounds__(DEP_T, 3) k_push_deposit(DepArgsT<R> a) {
    typedef double dvp __attribute__((ext_vector_type(PPL)));
    constexpr int PL = 2 * NMOD - 1;
    __shared__ DepWave<PPL> wl[DEP_WAVES];
    __shared__ __align__(16) double tile[DEP_POOL];
    __shared__ int red[DEP_WAVES][4];
    __shared__ int nsegs[2][DEP_WAVES];         // of J, of rho
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const GridGeom gJ = frame_geom(a.gJ), gR = frame_geom(a.gR);
    const int64_t ld = a.ld;
    const bool doJ = a.J != nullptr, doR = a.R != nullptr;
    const int64_t sr = gJ.nx + 1, sm = sr * (gJ.nr + 1), sl = sm * NMOD;
    DepWave<PPL>& L = wl[wv];

    const int grp = xcd_block(blockIdx.x, gridDim.x);
    const int64_t ib = (int64_t)grp * (DEP_T * PPL) + (int64_t)tid * PPL;
    double X[3][PPL], H[3][PPL], U[3][PPL], W[PPL];
    auto load = [&](const auto* p, double (&v)[PPL]) __attribute__((always_inline)) {
        typedef typename std::remove_cv<typename std::remove_pointer<decltype(p)>::type>::type T;
        typedef T tvp __attribute__((ext_vector_type(PPL)));
        if (a.vec && ib + PPL <= a.np) {
            const tvp t = *reinterpret_cast<const tvp*>(p + ib);
#pragma unroll
            for (int k = 0; k < PPL; k++) v[k] = t[k];
        } else {
#pragma unroll
            for (int k = 0; k < PPL; k++) v[k] = ib + k < a.np ? (double)p[ib + k] : 0.0;
        }
    };
    // ---- 1. load, push, store, geometry
    load(a.w, W);
#pragma unroll
    for (int c = 0; c < 3; c++) {
        load(a.x + c * ld, X[c]);
        load(a.u + c * ld, U[c]);
    }
    if (!a.push && doJ) {
#pragma unroll
        for (int c = 0; c < 3; c++) load(a.xh + c * ld, H[c]);
    }
    for (int i = 2 * tid; i < DEP_POOL; i += 2 * DEP_T) *reinterpret_cast<double2*>(tile + i) = cmk(0.0, 0.0);

    double ig[PPL];      // 1/gamma
#pragma unroll
    for (int k = 0; k < PPL; k++) {
        const double g2 = 1.0 + (U[0][k] * U[0][k] + U[1][k] * U[1][k] + U[2][k] * U[2][k]);
        double gam;
        sqrt_rsqrt(g2, gam, ig[k]);
        if (!(g2 <= 1e300)) ig[k] = 1.0 / sqrt(g2);
    }
    if (a.push) {
        // particle_tools.f90:58-82: x += u*dt/gamma; x_half = (x_old + x_new)/2
#pragma unroll
        for (int k = 0; k < PPL; k++) {
            const double dt_gp = a.dt * ig[k];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const double xn = X[c][k] + U[c][k] * dt_gp;
                H[c][k] = 0.5 * (X[c][k] + xn);
                X[c][k] = xn;
            }
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            if (a.vec && ib + PPL <= a.np) {
                dvp t, h;
#pragma unroll
                for (int k = 0; k < PPL; k++) t[k] = X[c][k], h[k] = H[c][k];
                *reinterpret_cast<dvp*>(a.x + c * ld + ib) = t;
                *reinterpret_cast<dvp*>(a.xh + c * ld + ib) = h;
            } else {
#pragma unroll
                for (int k = 0; k < PPL; k++)
                    if (ib + k < a.np) {
                        a.x[c * ld + ib + k] = X[c][k];
                        a.xh[c * ld + ib + k] = H[c][k];
                    }
            }
        }
    }
    int bx0 = INT_MAX, bx1 = INT_MIN, br0 = INT_MAX, br1 = INT_MIN;
    int ixJ[PPL], irJ[PPL], ixR[PPL], irR[PPL];
    bool okJ[PPL], okR[PPL];
    double2 sR[PPL], pR[PPL];
#pragma unroll
    for (int k = 0; k < PPL; k++) {
        double2 s, p1;
        okJ[k] = doJ && W[k] != 0.0 && (fabs(U[0][k]) + fabs(U[1][k]) + fabs(U[2][k])) != 0.0 &&
                 dep_geom(H[0][k], H[1][k], H[2][k], gJ, ixJ[k], irJ[k], s, p1);
        if (okJ[k]) {
            bx0 = min(bx0, ixJ[k]), bx1 = max(bx1, ixJ[k]), br0 = min(br0, irJ[k]), br1 = max(br1, irJ[k]);
            const int o = L.pos(lane * PPL + k);
            const double wg = W[k] * ig[k];
            L.s[o] = s;
            L.p1[o] = p1;
#pragma unroll
            for (int c = 0; c < 3; c++) L.q[c][o] = U[c][k] * wg;
        }
        okR[k] = doR && W[k] != 0.0 && dep_geom(X[0][k], X[1][k], X[2][k], gR, ixR[k], irR[k], sR[k], pR[k]);
        if (okR[k]) bx0 = min(bx0, ixR[k]), bx1 = max(bx1, ixR[k]), br0 = min(br0, irR[k]), br1 = max(br1, irR[k]);
    }
    bx0 = wave_reduce63<false>(bx0);
    bx1 = wave_reduce63<true>(bx1);
    br0 = wave_reduce63<false>(br0);
    br1 = wave_reduce63<true>(br1);
    if (lane == 63) {
        red[wv][0] = bx0, red[wv][1] = bx1, red[wv][2] = br0, red[wv][3] = br1;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < DEP_WAVES; i++) {
        const int b0 = red[i][0], b1 = red[i][1], b2 = red[i][2], b3 = red[i][3];
        bx0 = i ? min(bx0, b0) : b0;
        bx1 = i ? max(bx1, b1) : b1;
        br0 = i ? min(br0, b2) : b2;
        br1 = i ? max(br1, b3) : b3;
    }
    bx0 = __builtin_amdgcn_readfirstlane(bx0);
    bx1 = __builtin_amdgcn_readfirstlane(bx1);
    br0 = __builtin_amdgcn_readfirstlane(br0);
    br1 = __builtin_amdgcn_readfirstlane(br1);

    // ---- 2 and 3
    int4 d = make_int4(-1, 0, 0, 0);
    if (bx1 >= bx0) {
        const int TX = bx1 - bx0 + 2, TR = br1 - br0 + 2;
        const int64_t nn64 = (int64_t)TX * TR;
        const int nc = (doJ ? 3 : 0) + (doR ? 1 : 0);
        const int64_t pns64 = (PL * nn64 + 1) & ~(int64_t)1;        // values per component, even
        // components per pass; 0: no tile
        const int per = nc * pns64 <= DEP_POOL ? nc : 3 * pns64 <= DEP_POOL ? 3 : pns64 <= DEP_POOL ? 1 : 0;
        const bool tiled = per > 0, slotted = tiled && TR <= max(DEP_SLOT_R, TX) && nc * pns64 <= dep_slot(NMOD);
        const int nn = tiled ? (int)nn64 : 1, pns = tiled ? (int)pns64 : 0;
        R* const slot = slotted ? a.slot + (int64_t)grp * dep_slot(NMOD) : nullptr;
        const int rho0 = doJ ? 3 * pns : 0;         // rho in the slot
        const int64_t corner = bx0 + br0 * sr;      // grid node of the tile's first node
        auto keys = [&](const bool (&ok)[PPL], const int (&ix)[PPL], const int (&ir)[PPL], uint32_t (&key)[PPL])
            __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < PPL; k++)
                key[k] = !ok[k] ? DEP_SKIP
                                : tiled ? (uint32_t)((ir[k] - br0) * TX + ix[k] - bx0) : (uint32_t)(ix[k] + ir[k] * sr);
        };
        uint32_t key[PPL];
        if (doJ) {
            keys(okJ, ixJ, irJ, key);
            const int nseg = dep_segments<PPL, 3>(L, key);
            if (per != 1) {
                dep_pass<NMOD, 3, PPL, R>(L, wv, nseg, nsegs[0], 0, tiled, tile, pns, nn, TX, a.J, sr, sm, sl);
                if (per == 3) {
                    __syncthreads();
                    dep_writeout<NMOD, R>(tile, 3, pns, nn, TX, slot, a.J + corner, sr, sm);
                    __syncthreads();
                }
            } else {
#pragma unroll 1
                for (int c = 0; c < 3; c++) {
                    dep_pass<NMOD, 1, PPL, R>(L, wv, nseg, nsegs[0], c, true, tile, pns, nn, TX, a.J, sr, sm, sl);
                    __syncthreads();
                    dep_writeout<NMOD, R>(tile, 1, pns, nn, TX, slot ? slot + c * pns : nullptr,
                                          a.J + c * sl + corner, sr, sm);
                    __syncthreads();
                }
            }
            wave_lds_fence();
        }
        if (doR) {
#pragma unroll
            for (int k = 0; k < PPL; k++)
                if (okR[k]) {
                    const int o = L.pos(lane * PPL + k);
                    L.s[o] = sR[k];
                    L.p1[o] = pR[k];
                    L.q[0][o] = W[k];
                }
            keys(okR, ixR, irR, key);
            const int nseg = dep_segments<PPL, 1>(L, key);
            dep_pass<NMOD, 1, PPL, R>(L, wv, nseg, nsegs[1], 0, tiled, tile + (per == 4 ? rho0 : 0), pns, nn, TX, a.R, sr,
                                      sm, sl);
            if (tiled) {
                __syncthreads();
                if (per != 4) {
                    dep_writeout<NMOD, R>(tile, 1, pns, nn, TX, slot ? slot + rho0 : nullptr, a.R + corner, sr, sm);
                } else if (slot) {
                    dep_writeout<NMOD, R>(tile, 4, pns, nn, TX, slot, nullptr, sr, sm);
                } else {
                    dep_writeout<NMOD, R>(tile, 3, pns, nn, TX, nullptr, a.J + corner, sr, sm);
                    dep_writeout<NMOD, R>(tile + rho0, 1, pns, nn, TX, nullptr, a.R + corner, sr, sm);
                }
            }
        }
        if (slotted) {
            d = make_int4(br0, bx0, TX, TR);
            if (a.mask && tid < TR)                 // (TR <= 64)
                atomicOr(a.mask + (int64_t)(br0 + tid) * a.words + (grp >> 11), 1u << ((grp >> 6) & 31));
        }
    }
    if (tid == 0) a.desc[grp] = d;
}

// ------------------------------------------------------------------ slot combine
//
// One wave per (64 node columns, node row r).  It lists the slots that cover
// its nodes in group order -- the 64 descriptors of one load and a ballot --
// and adds their sums to the grids once, so the order of the sum is fixed.
// The descriptors to look at come from the row's bits of `mask`, or, without
// one (small launches), are all of them.  (A radix sort of the descriptors by
// row, which the mask replaced, took a dozen launches and 70 us at 16.7 M
// particles.)
constexpr int CMB_T = 256;

// Instantiations whose sums the compiler would fit into the registers of eight
// (float) or four (double) waves a SIMD by loading a slot's values one or two at
// a time, a memory latency each.  They are held to cmb_waves and load all of a
// slot's values before adding any: 65536 sorted particles, 16 per cell, in 128 x
// 32 cells, mixed precision: four modes 67 -> 14 us, eight 169 -> 28 (the whole
// deposit 104 -> 52 and 210 -> 68; before it was one pass 81 and 104).
template <int NMOD, typename RT>
constexpr bool cmb_batch() { return NMOD >= (sizeof(RT) == 4 ? 4 : 5); }
template <int NMOD, typename RT>
constexpr int cmb_waves() { return !cmb_batch<NMOD, RT>() ? 8 : sizeof(RT) == 4 ? 4 : 2; }

template <int NMOD, typename RT>
__global__ void __launch_bounds__(CMB_T) __attribute__((amdgpu_waves_per_eu(1, cmb_waves<NMOD, RT>())))
k_dep_combine(DepArgsT<RT> a, int64_t sr, int64_t sm, int nx1) {
    constexpr int PL = 2 * NMOD - 1;
    constexpr bool BATCH = cmb_batch<NMOD, RT>();
    const int r = blockIdx.y, lane = threadIdx.x & 63;
    const int xs = (blockIdx.x * (CMB_T / 64) + (threadIdx.x >> 6)) * 64, x = xs + lane;
    if (xs >= nx1) return;
    const bool doJ = a.J != nullptr, doR = a.R != nullptr;
    RT acc[4][PL];       // J_x, J_y, J_z, rho
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int i = 0; i < PL; i++) acc[c][i] = 0;
    bool hit = false;
    auto look = [&](int batch) __attribute__((always_inline)) {
        const int b = batch * 64 + lane;
        int4 d = make_int4(-1, 0, 0, 0);
        if (b < a.ngroups) d = a.desc[b];
        uint64_t bal = __ballot(d.x >= 0 && r >= d.x && r - d.x < d.w && d.y < xs + 64 && d.y + d.z > xs);
        while (bal) {
            const int j = __builtin_ctzll(bal);
            bal &= bal - 1;
            const int row = __builtin_amdgcn_readlane(d.x, j), col = __builtin_amdgcn_readlane(d.y, j);
            const int width = __builtin_amdgcn_readlane(d.z, j), rows = __builtin_amdgcn_readlane(d.w, j);
            const int nn = width * rows, pns = (PL * nn + 1) & ~1, o = x - col;
            if (o >= 0 && o < width) {
                hit = true;
                const RT* sp = a.slot + (int64_t)(batch * 64 + j) * dep_slot(NMOD) + (r - row) * width + o;
                if constexpr (BATCH) {
                    RT v[4][PL];
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        if (c < 3 ? !doJ : !doR) continue;
                        const RT* q = sp + (c < 3 || doJ ? c * pns : 0);
#pragma unroll
                        for (int i = 0; i < PL; i++) v[c][i] = q[i * nn];
                    }
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        if (c < 3 ? !doJ : !doR) continue;
#pragma unroll
                        for (int i = 0; i < PL; i++) acc[c][i] += v[c][i];
                    }
                } else {
                    if (doJ) {
#pragma unroll
                        for (int c = 0; c < 3; c++)
#pragma unroll
                            for (int i = 0; i < PL; i++) acc[c][i] += sp[c * pns + i * nn];
                        sp += 3 * pns;
                    }
                    if (doR) {
#pragma unroll
                        for (int i = 0; i < PL; i++) acc[3][i] += sp[i * nn];
                    }
                }
            }
        }
    };
    if (a.mask) {
        const uint32_t* mask = a.mask + (int64_t)r * a.words;
        for (int w0 = 0; w0 < a.words; w0 += 64) {
            const uint32_t word = w0 + lane < a.words ? mask[w0 + lane] : 0u;
            uint64_t wb = __ballot(word != 0u);
            while (wb) {
                const int j = __builtin_ctzll(wb);
                wb &= wb - 1;
                uint32_t bits = (uint32_t)__builtin_amdgcn_readlane((int)word, j);
                while (bits) {
                    look((w0 + j) * 32 + __builtin_ctz(bits));
                    bits &= bits - 1;
                }
            }
        }
    } else {
        for (int i = 0; i * 64 < a.ngroups; i++) look(i);
    }
    if (!hit || x >= nx1) return;
    const int64_t node = x + (int64_t)r * sr;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        if (c < 3 ? !doJ : !doR) continue;
        cplx_t<RT>* gp = (c < 3 ? a.J + c * NMOD * sm : a.R) + node;
#pragma unroll
        for (int m = 0; m < NMOD; m++) {
            // the imaginary part of mode 0 is 0 times the real one
            const cplx_t<RT> v = m ? cmake<RT>(acc[c][2 * m - 1], acc[c][2 * m]) : cmake<RT>(acc[c][0], 0 * acc[c][0]);
            gp[m * sm] = cadd(gp[m * sm], v);
        }
    }
}

// Stable compaction: flags, exclusive scan, scatter of every particle array.
__global__ void k_keep_flags(const double* __restrict__ coord, int64_t ld, double l0, double l1, double l2, double l3,
                             int32_t* __restrict__ flag, int np) {
    const int ip = blockIdx.x * blockDim.x + threadIdx.x;
    if (ip >= np) return;
    const double x = coord[ip], y = coord[ld + ip], z = coord[2 * ld + ip];
    // rounded as written (no contraction), as in the selection of k_cell_keys
    const double r2 = __dadd_rn(__dmul_rn(y, y), __dmul_rn(z, z));
    flag[ip] = (x >= l0 && x <= l1 && r2 >= l2 && r2 <= l3) ? 1 : 0;
}

template <typename T>
__global__ void k_compact_scatter(const int32_t* __restrict__ flag, const int64_t* __restrict__ pos,
                                  const T* __restrict__ src, T* __restrict__ dst, int64_t ld_src,
                                  int64_t ld_dst, int ncomp, int np) {
    const int ip = blockIdx.x * blockDim.x + threadIdx.x;
    if (ip >= np || !flag[ip]) return;
    const int64_t o = pos[ip];
    for (int c = 0; c < ncomp; c++) dst[c * ld_dst + o] = src[c * ld_src + ip];
}

// Launch kernel template K<NMOD> for NMOD = nkO + 1 (check_resident bounds nkO).
#define CH_MODE_SWITCH(nkO, LAUNCH)                  \
    switch ((nkO) + 1) {                             \
        case 1: LAUNCH(1); break;                    \
        case 2: LAUNCH(2); break;                    \
        case 3: LAUNCH(3); break;                    \
        case 4: LAUNCH(4); break;                    \
        case 5: LAUNCH(5); break;                    \
        case 6: LAUNCH(6); break;                    \
        case 7: LAUNCH(7); break;                    \
        default: LAUNCH(8); break;                   \
    }

static int32_t check_resident(int np, int64_t ld, int nkO) {
    if (np < 0 || ld < np) return fail(ST_EINVAL, "resident particles: np=%d ld=%lld", np, (long long)ld);
    if (nkO < 0 || nkO >= MAX_MODES)
        return fail(ST_EUNSUP, "azimuthal modes 0..%d requested; this build supports up to %d modes", nkO, MAX_MODES);
    return ST_OK;
}

// get_dens_on_grid (species.py:400-427): dens(nx+1, nr+1, nkO+1) = the
// deposited density (grid_deps.f90:89-147, ghost fold included) times
// VGrid[ir] per radial row; dens is overwritten.
template <typename W>
static int32_t dens_on_grid_impl(const double* coord, const W* wghts, int64_t ld, int32_t np, double* dens,
                                 double leftX, const double* Rgrid, double dx_inv, double dr_inv, double r0,
                                 double rmax, int32_t nx, int32_t nr, int32_t nkO, const double* vgrid) {
    CH_TRY(check_resident(np, ld, nkO));
    if (nx < 1 || nr < 1 || !dens || !vgrid || !is_device_ptr(dens) || !is_device_ptr(vgrid))
        return fail(ST_EINVAL, "dens_on_grid: nx=%d nr=%d; dens and vgrid are device arrays", nx, nr);
    double2* D = reinterpret_cast<double2*>(dens);
    CH_TRY(fill_bytes(D, 0, (size_t)(nx + 1) * (nr + 1) * (nkO + 1) * sizeof(double2)));
    if (np > 0) {
        const GridGeom g = resident_geom(leftX, Rgrid, dx_inv, dr_inv, r0, rmax, nx, nr, nkO);
        CH_TRY(launch_dep_dens<W>(coord, PStride{1, ld}, wghts, D, g, 0, np));
    }
    CH_TRY(ghost_fold<double>(D, nx + 1, nr + 1, nkO + 1));
    return scale_rows(D, vgrid, nx + 1, nr + 1, nkO + 1);
}

// ------------------------------------------------------------------ counting sort by cell
//
// key = ir*nx + ix for a particle in cell (ix, ir) of the grid, nx*nr for a
// kept particle outside the grid, nx*nr + 1 for a particle outside lims (it is
// dropped).  The cell comes from the same expressions as grid_deps.f90:46-47,
// evaluated with explicitly rounded operations so that the integer key of a
// particle does not depend on contraction choices of the compiler.
constexpr int KEYS_T = 256, KEYS_MAX_BLOCKS = 2048;
__global__ void __launch_bounds__(KEYS_T) k_cell_keys(const double* __restrict__ x, const double* __restrict__ xh,
                                                       int64_t ld, int np, double leftX, double dx_inv, double dr_inv,
                                                       double r0, int nx, int nr, int use_lims, double l0, double l1,
                                                       double l2, double l3, int test_half,
                                                       uint32_t* __restrict__ keys, int32_t* __restrict__ kept) {
    __shared__ int32_t wkept[KEYS_T / 64];
    const uint32_t ncell = (uint32_t)nx * (uint32_t)nr;
    int32_t nkept = 0;    // this wave's kept particles (the same in every lane)
    // grid-stride: a bounded number of blocks, one counter update per block
    for (int64_t ip = (int64_t)blockIdx.x * KEYS_T + threadIdx.x; ip - threadIdx.x < np;
         ip += (int64_t)gridDim.x * KEYS_T) {
        const bool valid = ip < np;
        uint32_t key = 0;
        if (valid) {
            const double px = x[ip], py = x[ld + ip], pz = x[2 * ld + ip];
            bool drop = false;
            if (use_lims) {
                const double* t = test_half ? xh : x;
                const double tx = t[ip], ty = t[ld + ip], tz = t[2 * ld + ip];
                const double r2 = __dadd_rn(__dmul_rn(ty, ty), __dmul_rn(tz, tz));
                drop = !(tx >= l0 && tx <= l1 && r2 >= l2 && r2 <= l3);
            }
            if (drop) {
                key = ncell + 1;
            } else {
                const double rp = sqrt(__dadd_rn(__dmul_rn(py, py), __dmul_rn(pz, pz)));
                const double fx = __dmul_rn(__dsub_rn(px, leftX), dx_inv);
                const double fr = __dmul_rn(__dsub_rn(rp, r0), dr_inv);
                if (fx >= 0.0 && fx < (double)nx && fr >= 0.0 && fr < (double)nr)
                    key = (uint32_t)floor(fr) * (uint32_t)nx + (uint32_t)floor(fx);
                else
                    key = ncell;
            }
            keys[ip] = key;
        }
        nkept += (int32_t)__popcll(__ballot(valid && key <= ncell));
    }
    if ((threadIdx.x & 63) == 0) wkept[threadIdx.x >> 6] = nkept;
    __syncthreads();
    if (threadIdx.x == 0) {
        int32_t t = 0;
        for (int w = 0; w < KEYS_T / 64; w++) t += wkept[w];
        if (t) atomicAdd(kept, t);
    }
}

template <typename R>
__global__ void k_gather_particles(const int32_t* __restrict__ idx, int n, const double* __restrict__ x,
                                   const double* __restrict__ xh, const R* __restrict__ u,
                                   const R* __restrict__ w, int64_t ld, double* __restrict__ x2,
                                   double* __restrict__ xh2, R* __restrict__ u2, R* __restrict__ w2,
                                   int64_t ld2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t j = idx[i];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        x2[c * ld2 + i] = x[c * ld + j];
        xh2[c * ld2 + i] = xh[c * ld + j];
        u2[c * ld2 + i] = u[c * ld + j];
    }
    w2[i] = w[j];
}

}  // namespace chimera

using namespace chimera;

template <typename R>
static int32_t sort_cells_impl(const double* coord, const double* coord_half, const R* momenta, const R* wghts,
                               int64_t ld, int32_t np, double* coord2, double* coord_half2, R* momenta2, R* wghts2,
                               int64_t ld2, double leftX, double dx_inv, double dr_inv, double r0, int32_t nx,
                               int32_t nr, const double* lims, int32_t test_half, int32_t* np_out, int32_t* perm) {
    CH_TRY(check_resident(np, ld, 0));
    if (np_out == nullptr || ld2 < np || nx < 1 || nr < 1) return fail(ST_EINVAL, "soa_sort_cells: bad arguments");
    if ((int64_t)nx * nr + 2 > (int64_t)UINT32_MAX) return fail(ST_EINVAL, "soa_sort_cells: too many cells");
    if (np == 0) {
        *np_out = 0;
        return ST_OK;
    }
    KTimer kt(KF_SORT);
    uint32_t* keys = static_cast<uint32_t*>(scratch(8, (size_t)np * sizeof(uint32_t)));
    int32_t* idx = perm ? perm : static_cast<int32_t*>(scratch(9, (size_t)np * sizeof(int32_t)));
    uint32_t* ktmp = static_cast<uint32_t*>(scratch(10, (size_t)np * sizeof(uint32_t)));
    int32_t* itmp = static_cast<int32_t*>(scratch(11, (size_t)np * sizeof(int32_t)));
    int32_t* kept = static_cast<int32_t*>(scratch(15, 256));
    if (!keys || !idx || !ktmp || !itmp || !kept) return ST_ENOMEM;
    CH_HIP(hipMemsetAsync(kept, 0, sizeof(int32_t), stream()));
    double L[4] = {0, 0, 0, 0};
    if (lims) memcpy(L, lims, sizeof L);
    const int64_t kb = (np + KEYS_T - 1) / KEYS_T;
    hipLaunchKernelGGL(k_cell_keys, (unsigned)(kb < KEYS_MAX_BLOCKS ? kb : KEYS_MAX_BLOCKS), KEYS_T, 0, stream(), coord,
                       coord_half, ld, np, leftX, dx_inv,
                       dr_inv, r0, nx, nr, lims ? 1 : 0, L[0], L[1], L[2], L[3], test_half, keys, kept);
    CH_LAUNCH_CHECK("k_cell_keys");
    const uint64_t maxkey = (uint64_t)nx * nr + 1;
    int bits = 1;
    while ((1ull << bits) <= maxkey) bits++;
    CH_TRY(radix_sort_keys(keys, idx, ktmp, itmp, np, bits, 12, 13));
    int32_t hk = 0;
    CH_HIP(hipMemcpyAsync(&hk, kept, sizeof hk, hipMemcpyDeviceToHost, stream()));
    CH_HIP(hipStreamSynchronize(stream()));
    hipLaunchKernelGGL(k_gather_particles<R>, blocks_for(hk, 256), 256, 0, stream(), idx, hk, coord, coord_half, momenta,
                       wghts, ld, coord2, coord_half2, momenta2, wghts2, ld2);
    CH_LAUNCH_CHECK("k_gather_particles");
    *np_out = hk;
    return ST_OK;
}

// The device list of a resident gather-push: none, or the one analytic
// undulator of undul_params (host, 4 doubles), or the described devices.
static int32_t undul_devices(ExtDevices& devs, const double* undul_params) {
    memset(&devs, 0, sizeof devs);
    if (!undul_params) return ST_OK;
    devs.n = 1;
    return make_ext_device(devs.d[0], DEV_UNDUL, undul_params, 4, nullptr, 0, 0.0);
}


template <typename R>
static int32_t gather_push_impl(const double* coord, R* momenta, const R* wghts, int64_t ld, int32_t np,
                                const cplx_t<R>* Fld, double leftX, const double* Rgrid, double dx_inv, double dr_inv,
                                double r0, double rmax, int32_t nx, int32_t nr, int32_t nkO, double push_dt,
                                const ExtDevices& devs, const double* frame) {
    CH_TRY(check_resident(np, ld, nkO));
    if (np == 0) return ST_OK;
    const PStride s = {1, ld};
    GridGeom g = resident_geom(leftX, Rgrid, dx_inv, dr_inv, r0, rmax, nx, nr, nkO);
    g.leftX_dev = frame;
    KTimer kt(KF_GATHER_PUSH);
#define GATHER_LAUNCH(N)                                                                                      \
    hipLaunchKernelGGL((k_gather_push<N, R>), blocks_for(np, GP_T), GP_T, 0, stream(), coord, s, momenta, s, wghts, \
                       Fld, g, push_dt, devs, np)
    CH_MODE_SWITCH(nkO, GATHER_LAUNCH)
#undef GATHER_LAUNCH
    CH_LAUNCH_CHECK("k_gather_push");
    return ST_OK;
}

// Stable removal of the particles outside lims.  With destination arrays
// (dst, leading dimension ld_dst) the kept particles are scattered there and
// the sources are left as they were; without, they are scattered to scratch
// memory and copied back in place.
template <typename R>
static int32_t compact_impl(double* coord, double* coord_half, R* momenta, R* wghts, int64_t ld, int32_t np,
                            const double* lims, int32_t test_half, int32_t* np_out, double* d_coord = nullptr,
                            double* d_half = nullptr, R* d_mom = nullptr, R* d_w = nullptr, int64_t ld_dst = 0) {
    CH_TRY(check_resident(np, ld, 0));
    if (lims == nullptr || np_out == nullptr) return fail(ST_EINVAL, "soa_compact: null lims/np_out");
    if (np == 0) {
        *np_out = 0;
        return ST_OK;
    }
    const bool into = d_coord != nullptr;
    if (into && (!d_half || !d_mom || !d_w || ld_dst < np))
        return fail(ST_EINVAL, "soa_compact_into: four destination arrays of leading dimension >= np");
    int32_t* flag = static_cast<int32_t*>(scratch(4, (size_t)np * sizeof(int32_t)));
    int64_t* pos = static_cast<int64_t*>(scratch(5, ((size_t)np + 8) * sizeof(int64_t)));
    double* tmp = into ? nullptr : static_cast<double*>(scratch(7, (size_t)np * 3 * sizeof(double)));
    if (!flag || !pos || (!into && !tmp)) return ST_ENOMEM;
    int64_t* total = pos + np;
    const double* test = test_half ? coord_half : coord;
    KTimer kt(KF_SORT);
    hipLaunchKernelGGL(k_keep_flags, blocks_for(np, 256), 256, 0, stream(), test, ld, lims[0], lims[1], lims[2],
                       lims[3], flag, np);
    CH_LAUNCH_CHECK("k_keep_flags");
    CH_TRY(exclusive_scan(flag, pos, np, total, 6));
    // each array: scatter the kept particles to the destination, or to the
    // work buffer and back
    auto one = [&](auto* arr, decltype(arr) dst, int nc) -> int32_t {
        typedef typename std::remove_pointer<decltype(arr)>::type T;
        if (into) {
            hipLaunchKernelGGL((k_compact_scatter<T>), blocks_for(np, 256), 256, 0, stream(), flag, pos, arr, dst, ld,
                               ld_dst, nc, np);
            CH_LAUNCH_CHECK("k_compact_scatter");
            return ST_OK;
        }
        T* t = reinterpret_cast<T*>(tmp);
        hipLaunchKernelGGL((k_compact_scatter<T>), blocks_for(np, 256), 256, 0, stream(), flag, pos, arr, t, ld,
                           (int64_t)np, nc, np);
        CH_LAUNCH_CHECK("k_compact_scatter");
        CH_HIP(hipMemcpy2DAsync(arr, ld * sizeof(T), t, (size_t)np * sizeof(T), (size_t)np * sizeof(T), nc,
                                hipMemcpyDeviceToDevice, stream()));
        return ST_OK;
    };
    CH_TRY(one(coord, d_coord, 3));
    CH_TRY(one(coord_half, d_half, 3));
    CH_TRY(one(momenta, d_mom, 3));
    CH_TRY(one(wghts, d_w, 1));
    int64_t h = 0;
    CH_HIP(hipMemcpyAsync(&h, total, sizeof h, hipMemcpyDeviceToHost, stream()));
    CH_HIP(hipStreamSynchronize(stream()));
    *np_out = (int32_t)h;
    return ST_OK;
}

template <typename R>
static int32_t push_deposit_impl(double* coord, double* coord_half, const R* momenta, const R* wghts, int64_t ld,
                                 int32_t np, double dt, double leftX_J, double leftX_rho, const double* Rgrid,
                                 double dx_inv, double dr_inv, double r0, double rmax, int32_t nx, int32_t nr,
                                 int32_t nkO, cplx_t<R>* curr, cplx_t<R>* dens, const double* frame) {
    CH_TRY(check_resident(np, ld, nkO));
    if (np == 0) return ST_OK;
    DepArgsT<R> a;
    a.x = coord;
    a.xh = coord_half;
    a.u = momenta;
    a.w = wghts;
    a.ld = ld;
    a.np = np;
    a.push = dt != 0.0;
    a.dt = dt;
    a.gJ = resident_geom(leftX_J, Rgrid, dx_inv, dr_inv, r0, rmax, nx, nr, nkO);
    a.gR = resident_geom(leftX_rho, Rgrid, dx_inv, dr_inv, r0, rmax, nx, nr, nkO);
    a.gJ.leftX_dev = frame;
    a.gR.leftX_dev = frame ? frame + 1 : nullptr;
    a.J = curr;
    a.R = dens;
    if (!a.J && !a.R) return ST_OK;
    if ((int64_t)(nx + 1) * (nr + 1) >= (int64_t)DEP_SKIP)
        return fail(ST_EUNSUP, "push_deposit: %d x %d nodes per mode", nx + 1, nr + 1);
    // groups of 512 particles where they average 8 or more per cell and fill
    // the chip twice over in such groups; else of 256
    const bool big = (int64_t)np >= (int64_t)8 * nx * nr && np >= 512 * 512;
    const int ppl = big ? 2 : 1;
    {
        auto al = [](const void* p, size_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; };
        a.vec = ld % ppl == 0 && al(coord, 8 * ppl) && al(coord_half, 8 * ppl) && al(momenta, sizeof(R) * ppl) &&
                al(wghts, sizeof(R) * ppl);
    }
    a.ngroups = (int)blocks_for(np, DEP_T * ppl);
    // up to 1024 descriptors a combine wave reads them all (16 KiB in L2);
    // beyond, the deposit marks those of each row
    const int nbatch = (a.ngroups + 63) / 64;
    a.words = (nbatch + 31) / 32;
    const size_t mask_bytes = nbatch > 16 ? (size_t)(nr + 1) * a.words * sizeof(uint32_t) : 0;
    a.slot = static_cast<R*>(scratch(16, (size_t)a.ngroups * dep_slot(nkO + 1) * sizeof(R)));
    a.desc = static_cast<int4*>(scratch(18, (size_t)a.ngroups * sizeof(int4)));
    a.mask = mask_bytes ? static_cast<uint32_t*>(scratch(19, mask_bytes)) : nullptr;
    if (!a.slot || !a.desc || (mask_bytes && !a.mask)) return ST_ENOMEM;
    KTimer kt(a.J ? KF_DEP_CURR : KF_DEP_DENS);
    if (a.mask) CH_TRY(fill_bytes(a.mask, 0, mask_bytes));
#define DEP_LAUNCH(N)                                                                       \
    do {                                                                                    \
        if (big)                                                                            \
            hipLaunchKernelGGL((k_push_deposit<N, R, 2>), a.ngroups, DEP_T, 0, stream(), a);      \
        else                                                                                \
            hipLaunchKernelGGL((k_push_deposit<N, R, 1>), a.ngroups, DEP_T, 0, stream(), a);      \
    } while (0)
    CH_MODE_SWITCH(nkO, DEP_LAUNCH)
#undef DEP_LAUNCH
    CH_LAUNCH_CHECK("k_push_deposit");
    const int64_t sr = nx + 1, sm = sr * (nr + 1);
    const dim3 grid((unsigned)((nx + 1 + CMB_T - 1) / CMB_T), (unsigned)(nr + 1));
#define CMB_LAUNCH(N) hipLaunchKernelGGL((k_dep_combine<N, R>), grid, CMB_T, 0, stream(), a, sr, sm, nx + 1)
    CH_MODE_SWITCH(nkO, CMB_LAUNCH)
#undef CMB_LAUNCH
    CH_LAUNCH_CHECK("k_dep_combine");
    return ST_OK;
}

extern "C" {

int32_t chimera_soa_push_coords(double* coord, double* coord_half, const double* momenta, int64_t ld, int32_t np,
                                double dt) {
    CH_TRY(check_resident(np, ld, 0));
    if (np == 0) return ST_OK;
    const PStride s = {1, ld};
    return launch_push_coords(coord, s, momenta, s, coord_half, s, dt, np);
}

int32_t chimera_soa_dep_curr(const double* coord, const double* momenta, const double* wghts, int64_t ld, int32_t np,
                             double* curr, double leftX, const double* Rgrid, double dx_inv, double dr_inv, double r0,
                             double rmax, int32_t nx, int32_t nr, int32_t nkO) {
    CH_TRY(check_resident(np, ld, nkO));
    if (np == 0) return ST_OK;
    const PStride s = {1, ld};
    const GridGeom g = resident_geom(leftX, Rgrid, dx_inv, dr_inv, r0, rmax, nx, nr, nkO);
    return launch_dep_curr(coord, s, momenta, s, wghts, reinterpret_cast<double2*>(curr), g, 0, np);
}

int32_t chimera_soa_dep_dens(const double* coord, const double* wghts, int64_t ld, int32_t np, double* dens,
                             double leftX, const double* Rgrid, double dx_inv, double dr_inv, double r0, double rmax,
                             int32_t nx, int32_t nr, int32_t nkO) {
    CH_TRY(check_resident(np, ld, nkO));
    if (np == 0) return ST_OK;
    const PStride s = {1, ld};
    const GridGeom g = resident_geom(leftX, Rgrid, dx_inv, dr_inv, r0, rmax, nx, nr, nkO);
    return launch_dep_dens(coord, s, wghts, reinterpret_cast<double2*>(dens), g, 0, np);
}

int32_t chimera_soa_dens_on_grid(const double* coord, const double* wghts, int64_t ld, int32_t np, double* dens,
                                 double leftX, const double* Rgrid, double dx_inv, double dr_inv, double r0,
                                 double rmax, int32_t nx, int32_t nr, int32_t nkO, const double* vgrid) {
    return dens_on_grid_impl<double>(coord, wghts, ld, np, dens, leftX, Rgrid, dx_inv, dr_inv, r0, rmax, nx, nr, nkO,
                                     vgrid);
}

int32_t chimera_soa_dens_on_grid_mixed(const double* coord, const float* wghts, int64_t ld, int32_t np,
                                       double* dens, double leftX, const double* Rgrid, double dx_inv, double dr_inv,
                                       double r0, double rmax, int32_t nx, int32_t nr, int32_t nkO,
                                       const double* vgrid) {
    return dens_on_grid_impl<float>(coord, wghts, ld, np, dens, leftX, Rgrid, dx_inv, dr_inv, r0, rmax, nx, nr, nkO,
                                    vgrid);
}

int32_t chimera_soa_gather_push(const double* coord, double* momenta, const double* wghts, int64_t ld, int32_t np,
                                const double* Fld, double leftX, const double* Rgrid, double dx_inv, double dr_inv,
                                double r0, double rmax, int32_t nx, int32_t nr, int32_t nkO, double push_dt,
                                const double* undul_params, const double* frame) {
    ExtDevices devs;
    CH_TRY(undul_devices(devs, undul_params));
    return gather_push_impl<double>(coord, momenta, wghts, ld, np, reinterpret_cast<const double2*>(Fld), leftX, Rgrid,
                                    dx_inv, dr_inv, r0, rmax, nx, nr, nkO, push_dt, devs, frame);
}

int32_t chimera_soa_gather_push_mixed(const double* coord, float* momenta, const float* wghts, int64_t ld, int32_t np,
                                      const float* Fld, double leftX, const double* Rgrid, double dx_inv,
                                      double dr_inv, double r0, double rmax, int32_t nx, int32_t nr, int32_t nkO,
                                      double push_dt, const double* undul_params, const double* frame) {
    ExtDevices devs;
    CH_TRY(undul_devices(devs, undul_params));
    return gather_push_impl<float>(coord, momenta, wghts, ld, np, reinterpret_cast<const float2*>(Fld), leftX, Rgrid,
                                   dx_inv, dr_inv, r0, rmax, nx, nr, nkO, push_dt, devs, frame);
}

int32_t chimera_soa_gather_push_dev(const double* coord, double* momenta, const double* wghts, int64_t ld,
                                    int32_t np, const double* Fld, double leftX, const double* Rgrid, double dx_inv,
                                    double dr_inv, double r0, double rmax, int32_t nx, int32_t nr, int32_t nkO,
                                    double push_dt, const chimera_device_t* devices, int32_t ndev, double t,
                                    const double* frame) {
    ExtDevices devs;
    CH_TRY(ext_devices(devs, devices, ndev, t));
    return gather_push_impl<double>(coord, momenta, wghts, ld, np, reinterpret_cast<const double2*>(Fld), leftX, Rgrid,
                                    dx_inv, dr_inv, r0, rmax, nx, nr, nkO, push_dt, devs, frame);
}

int32_t chimera_soa_gather_push_dev_mixed(const double* coord, float* momenta, const float* wghts, int64_t ld,
                                          int32_t np, const float* Fld, double leftX, const double* Rgrid,
                                          double dx_inv, double dr_inv, double r0, double rmax, int32_t nx, int32_t nr,
                                          int32_t nkO, double push_dt, const chimera_device_t* devices, int32_t ndev,
                                          double t, const double* frame) {
    ExtDevices devs;
    CH_TRY(ext_devices(devs, devices, ndev, t));
    return gather_push_impl<float>(coord, momenta, wghts, ld, np, reinterpret_cast<const float2*>(Fld), leftX, Rgrid,
                                   dx_inv, dr_inv, r0, rmax, nx, nr, nkO, push_dt, devs, frame);
}

// Advance of a device-side window frame, as move_frame forms the new edge
// (chimera_main.py:286-291: Xgrid + shiftX, leftX = Xgrid[0]).
__global__ void k_frame_step(double* __restrict__ f, double shift1, double shift2) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const double a = f[1] + shift1;
    f[0] = a;
    f[1] = a + shift2;
}

int32_t chimera_frame_step(double* frame, double shift1, double shift2) {
    if (!is_device_ptr(frame)) return fail(ST_EINVAL, "frame_step: the frame is a device pointer");
    hipLaunchKernelGGL(k_frame_step, 1, 64, 0, stream(), frame, shift1, shift2);
    CH_LAUNCH_CHECK("k_frame_step");
    return ST_OK;
}

int32_t chimera_soa_compact(double* coord, double* coord_half, double* momenta, double* wghts, int64_t ld, int32_t np,
                            const double* lims, int32_t test_half, int32_t* np_out) {
    return compact_impl<double>(coord, coord_half, momenta, wghts, ld, np, lims, test_half, np_out);
}

int32_t chimera_soa_compact_mixed(double* coord, double* coord_half, float* momenta, float* wghts, int64_t ld,
                                  int32_t np, const double* lims, int32_t test_half, int32_t* np_out) {
    return compact_impl<float>(coord, coord_half, momenta, wghts, ld, np, lims, test_half, np_out);
}

int32_t chimera_soa_compact_into(const double* coord, const double* coord_half, const double* momenta,
                                 const double* wghts, int64_t ld, int32_t np, double* d_coord, double* d_half,
                                 double* d_mom, double* d_w, int64_t ld_dst, const double* lims, int32_t test_half,
                                 int32_t* np_out) {
    if (!d_coord) return fail(ST_EINVAL, "soa_compact_into: null destination");
    return compact_impl<double>(const_cast<double*>(coord), const_cast<double*>(coord_half),
                                const_cast<double*>(momenta), const_cast<double*>(wghts), ld, np, lims, test_half,
                                np_out, d_coord, d_half, d_mom, d_w, ld_dst);
}

int32_t chimera_soa_compact_into_mixed(const double* coord, const double* coord_half, const float* momenta,
                                       const float* wghts, int64_t ld, int32_t np, double* d_coord, double* d_half,
                                       float* d_mom, float* d_w, int64_t ld_dst, const double* lims,
                                       int32_t test_half, int32_t* np_out) {
    if (!d_coord) return fail(ST_EINVAL, "soa_compact_into: null destination");
    return compact_impl<float>(const_cast<double*>(coord), const_cast<double*>(coord_half),
                               const_cast<float*>(momenta), const_cast<float*>(wghts), ld, np, lims, test_half,
                               np_out, d_coord, d_half, d_mom, d_w, ld_dst);
}


int32_t chimera_soa_push_deposit(double* coord, double* coord_half, const double* momenta, const double* wghts,
                                 int64_t ld, int32_t np, double dt, double leftX_J, double leftX_rho,
                                 const double* Rgrid, double dx_inv, double dr_inv, double r0, double rmax, int32_t nx,
                                 int32_t nr, int32_t nkO, double* curr, double* dens, const double* frame) {
    return push_deposit_impl<double>(coord, coord_half, momenta, wghts, ld, np, dt, leftX_J, leftX_rho, Rgrid, dx_inv,
                                     dr_inv, r0, rmax, nx, nr, nkO, reinterpret_cast<double2*>(curr),
                                     reinterpret_cast<double2*>(dens), frame);
}

int32_t chimera_soa_push_deposit_mixed(double* coord, double* coord_half, const float* momenta, const float* wghts,
                                       int64_t ld, int32_t np, double dt, double leftX_J, double leftX_rho,
                                       const double* Rgrid, double dx_inv, double dr_inv, double r0, double rmax,
                                       int32_t nx, int32_t nr, int32_t nkO, float* curr, float* dens,
                                       const double* frame) {
    return push_deposit_impl<float>(coord, coord_half, momenta, wghts, ld, np, dt, leftX_J, leftX_rho, Rgrid, dx_inv,
                                    dr_inv, r0, rmax, nx, nr, nkO, reinterpret_cast<float2*>(curr),
                                    reinterpret_cast<float2*>(dens), frame);
}


int32_t chimera_soa_sort_cells(const double* coord, const double* coord_half, const double* momenta,
                               const double* wghts, int64_t ld, int32_t np, double* coord2, double* coord_half2,
                               double* momenta2, double* wghts2, int64_t ld2, double leftX, double dx_inv,
                               double dr_inv, double r0, int32_t nx, int32_t nr, const double* lims, int32_t test_half,
                               int32_t* np_out, int32_t* perm) {
    return sort_cells_impl<double>(coord, coord_half, momenta, wghts, ld, np, coord2, coord_half2, momenta2, wghts2,
                                   ld2, leftX, dx_inv, dr_inv, r0, nx, nr, lims, test_half, np_out, perm);
}

int32_t chimera_soa_sort_cells_mixed(const double* coord, const double* coord_half, const float* momenta,
                                     const float* wghts, int64_t ld, int32_t np, double* coord2, double* coord_half2,
                                     float* momenta2, float* wghts2, int64_t ld2, double leftX, double dx_inv,
                                     double dr_inv, double r0, int32_t nx, int32_t nr, const double* lims,
                                     int32_t test_half, int32_t* np_out, int32_t* perm) {
    return sort_cells_impl<float>(coord, coord_half, momenta, wghts, ld, np, coord2, coord_half2, momenta2, wghts2,
                                  ld2, leftX, dx_inv, dr_inv, r0, nx, nr, lims, test_half, np_out, perm);
}

}  // extern "C"
