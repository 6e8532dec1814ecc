// poisson.hip — pressure Poisson solve: multigrid-preconditioned CG.
//
// Replaces SetPressureVector + PoissonSolver (PETSc KSPSolve, GMRES(30) +
// BoomerAMG) + GetLocalArray (poisson.F90:107-186).
//
// Operator (poisson.F90:74-94, initialization.F90:105-173): the 7-point
// -lap_h with wall neighbours omitted (Neumann) and periodic neighbours
// wrapped; (Ax)_i = diag_i x_i - nbsum_i, nbsum = (xw+xe)/hx^2 +
// (xs+xn)/hy^2 + (xb+xt)/hz^2, wall neighbours contributing 0.
// The reference pins row P'(1,1,1) to the identity with b[0] = 0
// (poisson.F90:78,97-100,126); that system's solution is the solution of
// the singular system with b[0] := -sum_{i>0} b[i], shifted so that
// P'(1,1,1) = 0, which is what is solved here.
// Inflow sides are Neumann like walls. An outflow side (no counterpart in
// the reference) holds P' = 0 on the face: the ghost is -P', which adds
// 2/h^2 to the diagonal of the last cell; the operator is then
// non-singular, and there is no pinned row and no gauge shift.
//
// Preconditioner: one symmetric V-cycle. Smoother red-black Gauss-Seidel
// (pre: red then black, post: black then red); coarsest level: symmetric
// red-black sweeps in one work-group (damped Jacobi if a periodic dimension
// is odd); transfers: cell-centred trilinear prolongation (3/4, 1/4 per
// dimension) and restriction = prolongation^T / 8, with wall mirror and
// periodic wrap index rules. In the mixed form the whole V-cycle runs in
// FP32 on FP32 level arrays; the CG vectors, matrix-vector product, inner
// products and the stopping test stay FP64.
//
// Reductions have a fixed association (fixed block counts, LDS trees), so
// results are run-to-run identical.
#include "common.hpp"
#include "batched.hpp"

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <new>
#include <type_traits>

namespace {

using namespace bk;

constexpr int RB = 256;           // threads per block for level kernels
constexpr int RED_BLOCKS = 1024;
constexpr int RED_T = 256;

struct LaunchShape {
    dim3 grid, block;
};

// Barrier of one wavefront over LDS: its LDS operations complete in program
// order, so a compiler-level fence suffices.
__device__ __forceinline__ void wave_barrier_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
int pow2ceil(int v) {
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}
LaunchShape shape_for(int nx, int ny, int nz);
// Blocks always hold RB threads (bx * by = RB, rows past the level masked),
// so a launch over a batch of cases can run every case's blocks with one
// block size and the same block decomposition as the case's own launch.
LaunchShape shape_for(int nx, int ny, int nz) {
    (void)ny;
    int bx = std::min(64, pow2ceil(nx));
    int by = RB / bx;
    return {dim3(div_up(nx, bx), div_up(ny, by), nz), dim3(bx, by, 1)};
}

// nbsum in the oracle's association: ((xw+xe)*ihx2 + (xs+xn)*ihy2) + (xb+xt)*ihz2,
// wall neighbours 0, periodic neighbours wrapped; x(o) is the value at
// storage position o
template <typename T, typename F>
__device__ __forceinline__ T nbsum_f(const F &x, const LevelDev &L, int i, int j, int k) {
    const T ihx2 = T(L.ihx2), ihy2 = T(L.ihy2), ihz2 = T(L.ihz2);
    const bool pxw = L.bt[0] == IBMDEM_BC_PERIODIC, pyw = L.bt[2] == IBMDEM_BC_PERIODIC,
               pzw = L.bt[4] == IBMDEM_BC_PERIODIC;
    const bool hw = i > 0 || pxw, he = i < L.nx - 1 || pxw;
    const bool hs = j > 0 || pyw, hn = j < L.ny - 1 || pyw;
    const bool hb = k > 0 || pzw, ht = k < L.nz - 1 || pzw;
    const int iw = i > 0 ? i - 1 : L.nx - 1, ie = i < L.nx - 1 ? i + 1 : 0;
    const int js = j > 0 ? j - 1 : L.ny - 1, jn = j < L.ny - 1 ? j + 1 : 0;
    const int kb = k > 0 ? k - 1 : L.nz - 1, kt = k < L.nz - 1 ? k + 1 : 0;
    const T xw = hw ? x(lidx(L, iw, j, k)) : T(0), xe = he ? x(lidx(L, ie, j, k)) : T(0);
    const T xs = hs ? x(lidx(L, i, js, k)) : T(0), xn = hn ? x(lidx(L, i, jn, k)) : T(0);
    const T xb = hb ? x(lidx(L, i, j, kb)) : T(0), xt = ht ? x(lidx(L, i, j, kt)) : T(0);
    const T sx = (xw + xe) * ihx2;
    const T syy = (xs + xn) * ihy2;
    const T szz = (xb + xt) * ihz2;
    return sx + syy + szz;
}
template <typename T>
__device__ __forceinline__ T nbsum(const T *__restrict__ x, const LevelDev &L, int i, int j, int k) {
    return nbsum_f<T>([&](int o) { return x[o]; }, L, i, j, k);
}

// per-dimension diagonal count: 1 per present neighbour, 2 for an outflow
// (Dirichlet) face
__device__ __forceinline__ int diag_count(int i, int n, int lo, int hi) {
    int c = 2 - ((i == 0 && lo != IBMDEM_BC_PERIODIC) ? 1 : 0) - ((i == n - 1 && hi != IBMDEM_BC_PERIODIC) ? 1 : 0);
    if (i == n - 1 && hi == IBMDEM_BC_OUTFLOW) c += 2;
    return c;
}
// the diagonal table entry of a cell with both neighbours in all three
// dimensions (counts 2, 2, 2)
constexpr int DIAG_INTERIOR = 2 * 16 + 2 * 4 + 2;
__device__ __forceinline__ int diag_index(const LevelDev &L, int i, int j, int k) {
    return diag_count(i, L.nx, L.bt[0], L.bt[1]) * 16 + diag_count(j, L.ny, L.bt[2], L.bt[3]) * 4 +
           diag_count(k, L.nz, L.bt[4], L.bt[5]);
}

// The x-pair (2p, 2p+1) of row (j, k) in colour-split storage: both cells
// sit at position pos of their colour halves (the even cell in half ca), and
// every neighbour of either cell lies in the other cell's half, at pos or pos
// plus one of these offsets (wrapped across a periodic side; the h* flags
// are false across any other side). With these the stencils below evaluate
// nbsum's expression without per-neighbour index arithmetic.
struct PairGeo {
    int pos, ca;
    int dw, de, ds, dn, db, dt;   // even cell's west, odd cell's east, then y and z
    bool hw, he, hs, hn, hb, ht;
    int cx0, cx1, cyz;            // diagonal counts: x of the even / odd cell, cy*4 + cz
};
__device__ __forceinline__ PairGeo pair_geo(const LevelDev &L, int p, int j, int k) {
    const int rl = L.nx >> 1, pl = rl * L.ny;
    const bool px = L.bt[0] == IBMDEM_BC_PERIODIC, py = L.bt[2] == IBMDEM_BC_PERIODIC,
               pz = L.bt[4] == IBMDEM_BC_PERIODIC;
    PairGeo g;
    g.pos = (k * L.ny + j) * rl + p;
    g.ca = (j + k) & 1;
    g.hw = p > 0 || px;          g.dw = p > 0 ? -1 : rl - 1;
    g.he = p < rl - 1 || px;     g.de = p < rl - 1 ? 1 : 1 - rl;
    g.hs = j > 0 || py;          g.ds = j > 0 ? -rl : (L.ny - 1) * rl;
    g.hn = j < L.ny - 1 || py;   g.dn = j < L.ny - 1 ? rl : -(L.ny - 1) * rl;
    g.hb = k > 0 || pz;          g.db = k > 0 ? -pl : (L.nz - 1) * pl;
    g.ht = k < L.nz - 1 || pz;   g.dt = k < L.nz - 1 ? pl : -(L.nz - 1) * pl;
    g.cx0 = diag_count(2 * p, L.nx, L.bt[0], L.bt[1]);
    g.cx1 = diag_count(2 * p + 1, L.nx, L.bt[0], L.bt[1]);
    g.cyz = diag_count(j, L.ny, L.bt[2], L.bt[3]) * 4 + diag_count(k, L.nz, L.bt[4], L.bt[5]);
    return g;
}
// nbsum of the pair's even (h = 0) or odd (h = 1) cell from the loaded values:
// the pair's other one, the other x neighbour (west for h = 0, east for h = 1),
// south, north, below, above (each read at offset 0, the pair's own position,
// when absent, and replaced by 0 here: loads without a branch are all in flight
// at once)
template <typename T>
__device__ __forceinline__ T nbsum_pair_vals(const PairGeo &g, int h, T part, T xo, T ys, T yn, T zb, T zt,
                                             const LevelDev &L) {
    const T ihx2 = T(L.ihx2), ihy2 = T(L.ihy2), ihz2 = T(L.ihz2);
    const bool pw = h == 0 ? g.hw : true, pe = h == 0 ? true : g.he;
    const T vw = h == 0 ? xo : part, ve = h == 0 ? part : xo;
    const T xw = pw ? vw : T(0), xe = pe ? ve : T(0);
    const T xs = g.hs ? ys : T(0), xn = g.hn ? yn : T(0);
    const T xb = g.hb ? zb : T(0), xt = g.ht ? zt : T(0);
    const T sx = (xw + xe) * ihx2;
    const T syy = (xs + xn) * ihy2;
    const T szz = (xb + xt) * ihz2;
    return sx + syy + szz;
}

// Two-value accesses of a colour half (8 bytes in FP32, 16 in FP64).
template <typename T>
struct Vec2;
template <>
struct Vec2<float> { using type = float2; };
template <>
struct Vec2<double> { using type = double2; };
template <typename T>
__device__ __forceinline__ void ld2(const T *p, T &v0, T &v1) {
    const typename Vec2<T>::type v = *reinterpret_cast<const typename Vec2<T>::type *>(p);
    v0 = v.x;
    v1 = v.y;
}
template <typename T>
__device__ __forceinline__ void st2(T *p, T v0, T v1) {
    typename Vec2<T>::type v;
    v.x = v0;
    v.y = v1;
    *reinterpret_cast<typename Vec2<T>::type *>(p) = v;
}

// The matrix-vector product's launch on a level: two rows per thread, two-pair
// threads where the level is split and its rows hold an even number of
// pairs, else one pair per thread.
struct SweepShape {
    dim3 grid, block;
    bool x2;
};
SweepShape sweep_shape(const LevelDev &d) {
    const bool x2 = d.split && (d.nx >> 1) % 2 == 0;
    const LaunchShape sh = shape_for(x2 ? d.nx / 4 : div_up(d.nx, 2), d.ny, d.nz);
    return {dim3(sh.grid.x, div_up(d.ny, 2 * (int)sh.block.y), sh.grid.z), sh.block, x2};
}

// cell index of a virtual coordinate one step beyond the level: a wall side
// clamps to the edge (a coarse cell's restriction weighs the edge fine cell
// twice; a fine cell's neighbour parent there is its own parent, see
// parents), a periodic side wraps. Coordinates further out only occur in the
// unused part of a tile and are clamped to some valid cell.
__device__ __forceinline__ int tile_coord(int v, int n, int lo, int hi) {
    if (v < 0) v = lo != IBMDEM_BC_PERIODIC ? 0 : v + n;
    else if (v >= n) v = hi != IBMDEM_BC_PERIODIC ? n - 1 : v - n;
    return min(max(v, 0), n - 1);
}

__device__ __forceinline__ void parents(int f, int nc, int lo, int hi, int &p0, int &p1) {
    int cc = f / 2;
    int nb = (f & 1) ? cc + 1 : cc - 1;
    if (nb < 0) nb = lo != IBMDEM_BC_PERIODIC ? cc : nb + nc;
    else if (nb >= nc) nb = hi != IBMDEM_BC_PERIODIC ? cc : nb - nc;
    p0 = cc; p1 = nb;
}

#include "mgmarch.hpp"
#include "mgtile.hpp"

// ---------------------------------------------------------------------------
// The coarsest level of a hierarchy: `sweeps` symmetric pairs of red-black
// Gauss-Seidel sweeps from x = 0, colours 0, 1, 0, 1, ... and then 1, 0, 1,
// 0, ... . Where the order turns, colour 1 would be swept twice in a row; a
// cell's update reads only the other colour, so the second pass writes the
// same values and is left out: 4 sweeps - 1 half sweeps of strictly
// alternating colour, the same result bit for bit. A level whose colouring is
// inconsistent (an odd periodic extent) runs 2 sweeps damped Jacobi sweeps.
//
// How far halving gets depends on the extents: multiples of 32 end at a few
// hundred cells, other even extents at thousands or 10^5. Three forms, by
// the level's size (each cell's arithmetic is the same in all of them):
//   coarse_wg    up to CWG_PAIRS x-pairs: one work-group with x in LDS and
//                each thread's pairs in registers. Bound by the chain of
//                half sweeps (LDS round, six dependent FP64 operations,
//                barrier): 24 us a solve at 455 cells, 73 us at 7,920, 137 us
//                at 15,700.
//   coarse_jac   Jacobi levels of up to CJ_CELLS cells, likewise.
//   coarse_tile  larger levels of either kind: the level in tiles over the
//                whole chip, CT_H half sweeps a launch on a tile with a
//                CT_H-cell halo in LDS. One work-group over the whole level
//                in global memory took 9.6 ms a solve at 50x38x65 (123,500
//                cells).
// ---------------------------------------------------------------------------
constexpr int COARSE_LDS = 512;

__device__ __forceinline__ int coarse_half_sweeps(int sweeps) { return 4 * sweeps - 1; }

// One work-group of NT threads, CP x-pairs per thread (pair q = t + NT m).
// x is kept in LDS in two colour halves of one slot per pair; slot hs of each
// half is 0 and stands for missing neighbours.
constexpr int CWG_PAIRS = 8192;
template <typename T, int NT, int CP>
__device__ __forceinline__ void coarse_wg_body(const Blk &kb, const LevelDev &L, T *__restrict__ xg,
                                               const T *__restrict__ bg, int sweeps,
                                               const double *__restrict__ stop) {
    static_assert(NT * CP <= CWG_PAIRS, "pairs fit the LDS halves");
    if (*stop != 0.0) return;
    __shared__ T xs[2 * (NT * CP + 1)];
    const int t = threadIdx.x;
    const int rl = (L.nx + 1) >> 1, hs = rl * L.ny * L.nz;   // pairs (an odd row's last pair has one cell)
    const int H = hs + 1;
    const bool px = L.bt[0] == IBMDEM_BC_PERIODIC, py = L.bt[2] == IBMDEM_BC_PERIODIC,
               pz = L.bt[4] == IBMDEM_BC_PERIODIC;
    const T ihx2 = T(L.ihx2), ihy2 = T(L.ihy2), ihz2 = T(L.ihz2);
    // per pair: its parity (the colour of its even cell; -1: no pair), the
    // slots of its neighbours within the other colour's half (two per
    // register) and, by cell, right-hand side and 1/diagonal
    int ca[CP], nx2[CP], ny2[CP], nz2[CP];
    T bv[CP][2], id[CP][2];
#pragma unroll
    for (int m = 0; m < CP; ++m) {
        const int q = t + NT * m;
        ca[m] = -1;
        nx2[m] = ny2[m] = nz2[m] = 0;
        bv[m][0] = bv[m][1] = id[m][0] = id[m][1] = T(0);
        if (q >= hs) continue;
        const int row = q / rl, p = q - row * rl, k = row / L.ny, j = row - k * L.ny;
        const int i = 2 * p, last = L.nx - 1;
        ca[m] = (j + k) & 1;
        // the even cell's west neighbour is an odd cell, the odd cell's east
        // neighbour an even one (periodic x: nx is even)
        const int w = p > 0 ? q - 1 : (px ? q + rl - 1 : hs);
        const int e = i + 2 <= last ? q + 1 : (px ? q + 1 - rl : hs);
        const int s = j > 0 ? q - rl : (py ? q + (L.ny - 1) * rl : hs);
        const int n = j < L.ny - 1 ? q + rl : (py ? q - (L.ny - 1) * rl : hs);
        const int pl = rl * L.ny;
        const int b = k > 0 ? q - pl : (pz ? q + (L.nz - 1) * pl : hs);
        const int u = k < L.nz - 1 ? q + pl : (pz ? q - (L.nz - 1) * pl : hs);
        nx2[m] = w | e << 16;
        ny2[m] = s | n << 16;
        nz2[m] = b | u << 16;
        bv[m][0] = bg[lidx(L, i, j, k)];
        id[m][0] = T(L.idiag[diag_index(L, i, j, k)]);
        if (i < last) {   // else the odd cell does not exist: it stays 0
            bv[m][1] = bg[lidx(L, i + 1, j, k)];
            id[m][1] = T(L.idiag[diag_index(L, i + 1, j, k)]);
        }
    }
    for (int q = t; q < 2 * H; q += NT) xs[q] = T(0);
    __syncthreads();
    const int ns = coarse_half_sweeps(sweeps);
    for (int s = 0; s < ns; ++s) {
        const int color = s & 1;
        T *own = xs + color * H;
        const T *oth = xs + (1 - color) * H;
#pragma unroll
        for (int m = 0; m < CP; ++m) {
            if (ca[m] < 0) continue;
            const int q = t + NT * m;
            const bool even = ca[m] == color;
            const T part = oth[q], xo = oth[even ? nx2[m] & 0xffff : nx2[m] >> 16];
            const T sx = ((even ? xo : part) + (even ? part : xo)) * ihx2;
            const T sy = (oth[ny2[m] & 0xffff] + oth[ny2[m] >> 16]) * ihy2;
            const T sz = (oth[nz2[m] & 0xffff] + oth[nz2[m] >> 16]) * ihz2;
            own[q] = ((even ? bv[m][0] : bv[m][1]) + (sx + sy + sz)) * (even ? id[m][0] : id[m][1]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < CP; ++m) {
        if (ca[m] < 0) continue;
        const int q = t + NT * m, row = q / rl, p = q - row * rl, k = row / L.ny, j = row - k * L.ny;
        xg[lidx(L, 2 * p, j, k)] = xs[ca[m] * H + q];
        if (2 * p + 1 < L.nx) xg[lidx(L, 2 * p + 1, j, k)] = xs[(1 - ca[m]) * H + q];
    }
}
template <typename T, int NT, int CP>
__global__ __launch_bounds__(NT) void k_coarse_wg(LevelDev L, T *__restrict__ xg, const T *__restrict__ bg, int sweeps,
                                                  const double *__restrict__ stop) {
    coarse_wg_body<T, NT, CP>(hw_blk(), L, xg, bg, sweeps, stop);
}

// Jacobi levels in one work-group: CP cells per thread (cell q = t + NT m, x
// fastest), the iterate in two LDS arrays read and written in turn, so a
// sweep is one LDS round and one barrier; slot n of both is 0 and stands for
// missing neighbours. One wavefront with the cells in table-driven rounds and
// two barriers a sweep took 55 us at 8x6x7 and 65 us at 15x2x15; this takes
// 10 us at both.
constexpr int CJ_CELLS = 8192;
template <typename T, int NT, int CP>
__device__ __forceinline__ void coarse_jac_body(const Blk &kb, const LevelDev &L, T *__restrict__ xg,
                                                const T *__restrict__ bg, int sweeps,
                                                const double *__restrict__ stop) {
    static_assert(NT * CP <= CJ_CELLS, "16-bit neighbour slots");
    if (*stop != 0.0) return;
    __shared__ T xs[2][NT * CP + 1];
    const int t = threadIdx.x, n = L.nx * L.ny * L.nz, pl = L.nx * L.ny;
    const bool px = L.bt[0] == IBMDEM_BC_PERIODIC, py = L.bt[2] == IBMDEM_BC_PERIODIC,
               pz = L.bt[4] == IBMDEM_BC_PERIODIC;
    const T ihx2 = T(L.ihx2), ihy2 = T(L.ihy2), ihz2 = T(L.ihz2), om = T(0.8);
    int nbx[CP], nby[CP], nbz[CP];   // two neighbour slots each
    T bv[CP], id[CP], xv[CP];
#pragma unroll
    for (int m = 0; m < CP; ++m) {
        const int q = t + NT * m;
        nbx[m] = nby[m] = nbz[m] = 0;
        bv[m] = id[m] = xv[m] = T(0);
        if (q >= n) continue;
        const int row = q / L.nx, i = q - row * L.nx, k = row / L.ny, j = row - k * L.ny;
        const int w = i > 0 ? q - 1 : (px ? q + L.nx - 1 : n), e = i < L.nx - 1 ? q + 1 : (px ? q - L.nx + 1 : n);
        const int s = j > 0 ? q - L.nx : (py ? q + pl - L.nx : n),
                  r = j < L.ny - 1 ? q + L.nx : (py ? q - pl + L.nx : n);
        const int b = k > 0 ? q - pl : (pz ? q + n - pl : n), u = k < L.nz - 1 ? q + pl : (pz ? q - n + pl : n);
        nbx[m] = w | e << 16;
        nby[m] = s | r << 16;
        nbz[m] = b | u << 16;
        bv[m] = bg[lidx(L, i, j, k)];
        id[m] = T(L.idiag[diag_index(L, i, j, k)]);
        xs[0][q] = T(0);
    }
    if (t == 0) xs[0][n] = xs[1][n] = T(0);
    __syncthreads();
    for (int s = 0; s < 2 * sweeps; ++s) {
        const T *x = xs[s & 1];
        T *y = xs[1 - (s & 1)];
#pragma unroll
        for (int m = 0; m < CP; ++m) {
            const int q = t + NT * m;
            if (q >= n) continue;
            const T sx = (x[nbx[m] & 0xffff] + x[nbx[m] >> 16]) * ihx2;
            const T sy = (x[nby[m] & 0xffff] + x[nby[m] >> 16]) * ihy2;
            const T sz = (x[nbz[m] & 0xffff] + x[nbz[m] >> 16]) * ihz2;
            const T xn = (bv[m] + (sx + sy + sz)) * id[m];
            xv[m] = xv[m] + om * (xn - xv[m]);
            y[q] = xv[m];
        }
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < CP; ++m) {
        const int q = t + NT * m;
        if (q >= n) continue;
        const int row = q / L.nx, i = q - row * L.nx, k = row / L.ny, j = row - k * L.ny;
        xg[lidx(L, i, j, k)] = xv[m];
    }
}
template <typename T, int NT, int CP>
__global__ __launch_bounds__(NT) void k_coarse_jac(LevelDev L, T *__restrict__ xg, const T *__restrict__ bg, int sweeps,
                                                   const double *__restrict__ stop) {
    coarse_jac_body<T, NT, CP>(hw_blk(), L, xg, bg, sweeps, stop);
}

// Tiles of CT_X x CT_Y x CT_Z cells, CT_H half sweeps (Jacobi: sweeps) s0 ..
// s0 + ns - 1 from xin to xout (s0 = 0: from x = 0). The tile is loaded with a
// halo of CT_H cells (wrapped across periodic sides, inactive zeros beyond
// the others) and swept; after s half sweeps the cells s layers in are exact
// (the planes further out are left alone), and the tile itself is exact after
// CT_H. Halo cells are the neighbouring tiles' cells with their own
// arithmetic, so the result does not depend on the tiling. Red-black launches
// begin with a red sweep, which reads black cells alone: only those are
// loaded, and only those are stored by all but the last launch (all_out).
// A thread has CT_M pairs above each other, their values by colour in
// registers: a neighbour in z is mostly a register, its plane's index
// arithmetic the wavefront's, and LDS serves x and y. At 50x38x65 in FP64
// (180 blocks): 7.3 us a launch of four half sweeps, the solve 0.18 ms; with
// strided pairs and every neighbour from LDS 9.1 us, most of it index
// arithmetic.
constexpr int CT_X = 16, CT_Y = 8, CT_Z = 8, CT_H = 4, CT_M = 4;
constexpr int CT_RL = (CT_X + 2 * CT_H) / 2, CT_EY = CT_Y + 2 * CT_H, CT_EZ = CT_Z + 2 * CT_H;
constexpr int CT_NP = CT_RL * CT_EY * CT_EZ, CT_PL = CT_RL * CT_EY;   // x-pairs of a tile, of a plane
constexpr int CT_T = CT_NP / CT_M;
static_assert(CT_PL % 64 == 0 && CT_EZ % CT_M == 0 && CT_T <= 1024, "wavefronts within a plane");
static_assert(CT_T % 256 == 0 && CT_X % 2 == 0 && CT_H % 2 == 0, "whole x-pairs, launches that begin with red");
// the level's index of an unwrapped one, -1 beyond a side that is not periodic
__device__ __forceinline__ int ct_map(int v, int n, int lo) {
    if (v >= 0 && v < n) return v;
    if (lo != IBMDEM_BC_PERIODIC) return -1;
    v += v < 0 ? n : -n;
    if (v < 0 || v >= n) {   // levels smaller than the halo or the tile
        v %= n;
        v += v < 0 ? n : 0;
    }
    return v;
}
template <typename T, bool JAC>
__device__ __forceinline__ void coarse_tile_body(const Blk &kb, const LevelDev &L, const T *__restrict__ xin,
                                                 T *__restrict__ xout, const T *__restrict__ bg, int s0, int ns,
                                                 bool all_out, const double *__restrict__ stop) {
    const double stopped = *stop;
    __shared__ T xs[2 * CT_NP];
    const int t = threadIdx.x;
    const int seg = __builtin_amdgcn_readfirstlane(t / CT_PL), col = t - seg * CT_PL;
    const int y = col / CT_RL, p = col - y * CT_RL, z0 = seg * CT_M, q0 = z0 * CT_PL + col;
    const int ox = kb.bx * CT_X - CT_H, oy = kb.by * CT_Y - CT_H, oz = kb.bz * CT_Z - CT_H;
    const T ihx2 = T(L.ihx2), ihy2 = T(L.ihy2), ihz2 = T(L.ihz2);
    const int ca0 = (oy + y + oz + z0) & 1;   // colour of the first pair's even cell (ox is even)
    // cell (m, c): pair m's cell of colour c, even or odd as h(m, c) is 0 or 1
    auto h = [&](int m, int c) { return (ca0 + m + c) & 1; };
    T xv[CT_M][2], bv[CT_M][2], id[CT_M][2];
    bool act[CT_M][2];
    {
        const int rl = L.split ? L.nx >> 1 : L.nx;
        const int j = ct_map(oy + y, L.ny, L.bt[2]);
        const int i0 = ct_map(ox + 2 * p, L.nx, L.bt[0]), i1 = ct_map(ox + 2 * p + 1, L.nx, L.bt[0]);
        const int cy = 4 * diag_count(j, L.ny, L.bt[2], L.bt[3]);
        const int cx0 = 16 * diag_count(i0, L.nx, L.bt[0], L.bt[1]), cx1 = 16 * diag_count(i1, L.nx, L.bt[0], L.bt[1]);
        const T id_int = T(L.idiag[DIAG_INTERIOR]);
#pragma unroll
        for (int m = 0; m < CT_M; ++m) {
            const int k = ct_map(oz + z0 + m, L.nz, L.bt[4]);
            const int cz = diag_count(k, L.nz, L.bt[4], L.bt[5]), row = (k * L.ny + j) * rl;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int i = h(m, c) ? i1 : i0;
                act[m][c] = i >= 0 && j >= 0 && k >= 0;
                // lidx(L, i, j, k); inactive cells load cell 0 and drop it
                int g = L.split ? (((i ^ j ^ k) & 1) ? L.half : 0) + row + (i >> 1) : row + i;
                int d = (h(m, c) ? cx1 : cx0) + cy + cz;
                g = act[m][c] ? g : 0;
                d = act[m][c] ? d : DIAG_INTERIOR;
                const T bl = bg[g], xl = s0 > 0 && (JAC || c == 1) ? xin[g] : T(0);
                T il = id_int;
                if (d != DIAG_INTERIOR) il = T(L.idiag[d]);
                bv[m][c] = bl;
                id[m][c] = il;
                xv[m][c] = act[m][c] ? xl : T(0);
            }
        }
    }
    // every load is in flight before the first is used
    if (stopped != 0.0) return;
#pragma unroll
    for (int m = 0; m < CT_M; ++m)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            xs[c * CT_NP + q0 + m * CT_PL] = xv[m][c];
            // the outermost layer in x and y is not updated
            act[m][c] = act[m][c] && y > 0 && y < CT_EY - 1 && (h(m, c) ? p < CT_RL - 1 : p > 0);
        }
    __syncthreads();
    // nbsum of cell (m, c): its x neighbours are the pair's other cell and the
    // same colour's cell of the pair beside
    auto nb = [&](int m, int c) {
        const T *oth = xs + (1 - c) * CT_NP + q0 + m * CT_PL;
        const T sx = (xv[m][1 - c] + oth[h(m, c) ? 1 : -1]) * ihx2;
        const T syy = (oth[-CT_RL] + oth[CT_RL]) * ihy2;
        const T zb = m > 0 ? xv[m > 0 ? m - 1 : 0][1 - c] : oth[-CT_PL];
        const T zt = m < CT_M - 1 ? xv[m < CT_M - 1 ? m + 1 : 0][1 - c] : oth[CT_PL];
        const T szz = (zb + zt) * ihz2;
        return sx + syy + szz;
    };
    // planes s + 1 layers in and more take part in half sweep s
    auto inner = [&](int m, int s) { return z0 + m > s && z0 + m < CT_EZ - 1 - s; };
    for (int s = 0; s < ns; ++s) {
        if (JAC) {
            const T om = T(0.8);
            T nv[CT_M][2];
#pragma unroll
            for (int m = 0; m < CT_M; ++m)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    nv[m][c] = xv[m][c];
                    if (inner(m, s) && act[m][c]) {
                        const T xn = (bv[m][c] + nb(m, c)) * id[m][c];
                        nv[m][c] = xv[m][c] + om * (xn - xv[m][c]);
                    }
                }
            __syncthreads();
#pragma unroll
            for (int m = 0; m < CT_M; ++m)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    xv[m][c] = nv[m][c];
                    xs[c * CT_NP + q0 + m * CT_PL] = nv[m][c];
                }
            __syncthreads();
        } else {
            auto half = [&](int c) {
#pragma unroll
                for (int m = 0; m < CT_M; ++m)
                    if (inner(m, s) && act[m][c]) {
                        xv[m][c] = (bv[m][c] + nb(m, c)) * id[m][c];
                        xs[c * CT_NP + q0 + m * CT_PL] = xv[m][c];
                    }
                __syncthreads();
            };
            half(0);
            if (++s == ns) break;
            half(1);
        }
    }
    if (y < CT_H || y >= CT_Y + CT_H || p < CT_H / 2 || p >= (CT_X + CT_H) / 2) return;
    const int j = oy + y;
    if (j >= L.ny) return;
#pragma unroll
    for (int m = 0; m < CT_M; ++m) {
        const int z = z0 + m, k = oz + z;
        if (z < CT_H || z >= CT_Z + CT_H || k >= L.nz) continue;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int i = ox + 2 * p + h(m, c);
            if (i < L.nx && (JAC || c == 1 || all_out)) xout[lidx(L, i, j, k)] = xv[m][c];
        }
    }
}
template <typename T, bool JAC>
__global__ __launch_bounds__(CT_T) void k_coarse_tile(const LevelDev *__restrict__ lev,
                                                      const T *__restrict__ xin, T *__restrict__ xout,
                                                      const T *__restrict__ bg, int s0, int ns, bool all_out,
                                                      const double *__restrict__ stop) {
    coarse_tile_body<T, JAC>(hw_blk(), *lev, xin, xout, bg, s0, ns, all_out, stop);
}

// Which form a coarsest level takes: one work-group where the level fits its
// LDS and registers, with as few wavefronts as hold the level in one or two
// rounds (a barrier of four is faster than one of sixteen), tiles above. At
// the line, CWG_PAIRS pairs in FP64, one work-group takes 137 us and the
// tiles' 24 launches took 190 us (at 9.5 us each; 7.3 now).
enum CoarseForm { CF_WG256, CF_WG1, CF_WG2, CF_WG4, CF_WG8, CF_JAC512, CF_JAC2, CF_JAC8, CF_TILE, CF_TILE_JAC };
CoarseForm coarse_form(const LevelDev &d) {
    const long n = (long)d.nx * d.ny * d.nz, pairs = (long)((d.nx + 1) / 2) * d.ny * d.nz;
    if (!d.rb_valid) return n <= 512 ? CF_JAC512 : n <= 2048 ? CF_JAC2 : n <= CJ_CELLS ? CF_JAC8 : CF_TILE_JAC;
    if (pairs <= 512) return CF_WG256;
    return pairs <= 1024 ? CF_WG1 : pairs <= 2048 ? CF_WG2 : pairs <= 4096 ? CF_WG4 : pairs <= CWG_PAIRS ? CF_WG8 : CF_TILE;
}
int coarse_threads(CoarseForm f) { return f == CF_WG256 ? 256 : f == CF_JAC512 ? 512 : 1024; }
// the tile form's launches: launch q of n does half sweeps s0 .. s0 + ns - 1
// and reads what launch q - 1 wrote; the last one writes x (not tmp)
struct CoarseTileStep {
    int s0, ns;
    bool to_x, all_out;
};
int coarse_tile_launches(bool jac, int sweeps) { return div_up(jac ? 2 * sweeps : 4 * sweeps - 1, CT_H); }
CoarseTileStep coarse_tile_step(bool jac, int sweeps, int q) {
    const int total = jac ? 2 * sweeps : 4 * sweeps - 1, n = coarse_tile_launches(jac, sweeps);
    return {q * CT_H, std::min(CT_H, total - q * CT_H), (n - 1 - q) % 2 == 0, q == n - 1};
}
dim3 coarse_tile_grid(const LevelDev &d) { return dim3(div_up(d.nx, CT_X), div_up(d.ny, CT_Y), div_up(d.nz, CT_Z)); }

// The symmetric red-black sweeps of a coarsest level of n <= 64 CQ cells on
// one wavefront (lane l owns the cells q = l + 64 t): the lane's neighbour
// indices, 1/diagonal, right-hand side and colour are read from the tables
// once into registers, so a half sweep is one round of LDS loads of x (the
// zero slot x[n] for a missing neighbour). Cells of one colour do not read
// each other, so the lane's order over them does not matter; each cell's
// expression is the table sweep's.
template <int CQ, typename T>
__device__ __forceinline__ void coarse_reg_sweeps(T *x, const T *b, const short (*nb)[COARSE_LDS], const T *id,
                                                  const unsigned char *col, int n, int sweeps, T ihx2, T ihy2,
                                                  T ihz2) {
    const int lane = threadIdx.x & 63;
    int nbr[CQ][6], cr[CQ];
    T br[CQ], idr[CQ];
#pragma unroll
    for (int t = 0; t < CQ; ++t) {
        const int q = lane + 64 * t;
        cr[t] = -1;
        br[t] = T(0);
        idr[t] = T(0);
        for (int d = 0; d < 6; ++d) nbr[t][d] = n;
        if (q < n) {
            for (int d = 0; d < 6; ++d) nbr[t][d] = nb[d][q];
            br[t] = b[q];
            idr[t] = id[q];
            cr[t] = col[q];
        }
    }
    auto half = [&](int color) {
#pragma unroll
        for (int t = 0; t < CQ; ++t)
            if (cr[t] == color) {
                const T sx = (x[nbr[t][0]] + x[nbr[t][1]]) * ihx2;
                const T sy = (x[nbr[t][2]] + x[nbr[t][3]]) * ihy2;
                const T sz = (x[nbr[t][4]] + x[nbr[t][5]]) * ihz2;
                x[lane + 64 * t] = (br[t] + (sx + sy + sz)) * idr[t];
            }
        wave_barrier_lds();
    };
    for (int s = 1; s < 2 * sweeps; ++s) { half(0); half(1); }
    half(0);
}
// the register-held sweeps for levels of up to 256 cells; false: larger
template <typename T>
__device__ __forceinline__ bool coarse_sweeps_small(T *x, const T *b, const short (*nb)[COARSE_LDS], const T *id,
                                                    const unsigned char *col, int n, int sweeps, T ihx2, T ihy2,
                                                    T ihz2) {
    if (n <= 64) coarse_reg_sweeps<1, T>(x, b, nb, id, col, n, sweeps, ihx2, ihy2, ihz2);
    else if (n <= 128) coarse_reg_sweeps<2, T>(x, b, nb, id, col, n, sweeps, ihx2, ihy2, ihz2);
    else if (n <= 256) coarse_reg_sweeps<4, T>(x, b, nb, id, col, n, sweeps, ihx2, ihy2, ihz2);
    else return false;
    return true;
}

// the coarsest level's solve on the context's stream (dd: d on the device)
template <typename T>
void launch_coarsest(hipStream_t s, const LevelDev &d, const LevelDev *dd, T *x, const T *b, T *tmp, int sweeps,
                     const double *stop) {
    const CoarseForm f = coarse_form(d);
    const dim3 one(1);
    switch (f) {
    case CF_WG8: hipLaunchKernelGGL((k_coarse_wg<T, 1024, 8>), one, dim3(1024), 0, s, d, x, b, sweeps, stop); break;
    case CF_JAC512: hipLaunchKernelGGL((k_coarse_jac<T, 512, 1>), one, dim3(512), 0, s, d, x, b, sweeps, stop); break;
    case CF_JAC2: hipLaunchKernelGGL((k_coarse_jac<T, 1024, 2>), one, dim3(1024), 0, s, d, x, b, sweeps, stop); break;
    case CF_JAC8: hipLaunchKernelGGL((k_coarse_jac<T, 1024, 8>), one, dim3(1024), 0, s, d, x, b, sweeps, stop); break;
    case CF_WG256: hipLaunchKernelGGL((k_coarse_wg<T, 256, 2>), one, dim3(256), 0, s, d, x, b, sweeps, stop); break;
    case CF_WG1: hipLaunchKernelGGL((k_coarse_wg<T, 1024, 1>), one, dim3(1024), 0, s, d, x, b, sweeps, stop); break;
    case CF_WG2: hipLaunchKernelGGL((k_coarse_wg<T, 1024, 2>), one, dim3(1024), 0, s, d, x, b, sweeps, stop); break;
    case CF_WG4: hipLaunchKernelGGL((k_coarse_wg<T, 1024, 4>), one, dim3(1024), 0, s, d, x, b, sweeps, stop); break;
    default: {
        const bool jac = f == CF_TILE_JAC;
        const int n = coarse_tile_launches(jac, sweeps);
        for (int q = 0; q < n; ++q) {
            const CoarseTileStep st = coarse_tile_step(jac, sweeps, q);
            const T *in = st.to_x ? tmp : x;
            T *out = st.to_x ? x : tmp;
            if (jac)
                hipLaunchKernelGGL((k_coarse_tile<T, true>), coarse_tile_grid(d), dim3(CT_T), 0, s, dd, in, out, b,
                                   st.s0, st.ns, st.all_out, stop);
            else
                hipLaunchKernelGGL((k_coarse_tile<T, false>), coarse_tile_grid(d), dim3(CT_T), 0, s, dd, in, out, b,
                                   st.s0, st.ns, st.all_out, stop);
        }
    }
    }
}

// ---------------------------------------------------------------------------
// The small levels of the hierarchy as one work-group: from level `first`
// down to the coarsest, the whole V-cycle (smoothing, residual, restriction,
// coarse sweeps, prolongation) runs in LDS with a barrier between phases, in
// place of a few dozen launches that each cost more than their work. The
// coarsest level sweeps on one wavefront from neighbour tables. Every cell's
// arithmetic is the multi-launch path's, so the result is the same bit for
// bit; b of level `first` comes from global memory and its x goes back there
// for the prolongation to the level above. One CU's instruction issue bounds
// the larger levels and a chain of LDS round trips the coarsest. With the
// geometry in registers: levels 16^3, 8^3, 4^3, 2^3 in FP64 44 -> 31 us,
// 16x12x20 down to 4x3x5 38 -> 27 us, FP32 43 -> 33 us.
// ---------------------------------------------------------------------------
constexpr int TAIL_T = 1024;
constexpr int TAIL_BYTES = 112 * 1024;   // x (one extra zero slot on the coarsest level), b, r of the levels
constexpr int TAIL_MAXLEV = 6;           // levels of one tail (their descriptors are copied to LDS)
static_assert(sizeof(LevelDev) % 4 == 0, "level descriptors copied by words");
// (the tail's levels hold at most TAIL_BYTES / 12 cells, so its index
// divisions go through udiv_small)
static_assert(TAIL_BYTES / 12 < (1 << 14), "tail levels small enough for udiv_small");

// The x-pairs of a level above the coarsest (split) that one thread of NT
// sweeps: pairs t, t + NT, .... Where a pair's neighbours stand and what its
// cells are divided by is worked out once per visit and kept in registers, as
// is b, so a half sweep is six LDS loads and the sum (index arithmetic and
// table loads took two thirds of it). A missing neighbour is position `half`,
// a zero word behind each colour's cells.
template <typename T, int Q, int NT>
struct TailPairs {
    int o[Q][4], ox[Q][2];   // south, north, below, above; the other x neighbour of either colour's cell
    int di[Q][2];
    T id[Q][2], b[Q][2];
    T ihx2, ihy2, ihz2;
    const LevelDev &L;
    __device__ __forceinline__ TailPairs(const LevelDev &lev, const T *bl) : L(lev) {
        ihx2 = T(L.ihx2);
        ihy2 = T(L.ihy2);
        ihz2 = T(L.ihz2);
        const int rl = L.nx >> 1, none = L.half;
#pragma unroll
        for (int u = 0; u < Q; ++u) {
            const int p = threadIdx.x + u * NT;
            if (p >= L.half) continue;
            const int row = udiv_small(p, rl, L.m_row), kr = udiv_small(row, L.ny, L.m_ny);
            const PairGeo g = pair_geo(L, p - row * rl, row - kr * L.ny, kr);
            o[u][0] = g.hs ? p + g.ds : none;
            o[u][1] = g.hn ? p + g.dn : none;
            o[u][2] = g.hb ? p + g.db : none;
            o[u][3] = g.ht ? p + g.dt : none;
            const int w = g.hw ? p + g.dw : none, e = g.he ? p + g.de : none;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const int h = g.ca ^ c;   // the pair's cell of colour c: even (0) or odd (1)
                ox[u][c] = h ? e : w;
                di[u][c] = (h ? g.cx1 : g.cx0) * 16 + g.cyz;
                id[u][c] = T(L.idiag[di[u][c]]);
                b[u][c] = bl[c * L.half + p];
            }
        }
    }
    // the black cells stand behind the red ones and their zero word
    __device__ __forceinline__ int base(int c) const { return c ? L.half + 1 : 0; }
    // nbsum of the cell of colour c of pair u
    __device__ __forceinline__ T nbsum(const T *x, int u, int c) const {
        const T *oth = x + base(1 - c);
        const T sx = (oth[threadIdx.x + u * NT] + oth[ox[u][c]]) * ihx2;
        const T syy = (oth[o[u][0]] + oth[o[u][1]]) * ihy2;
        const T szz = (oth[o[u][2]] + oth[o[u][3]]) * ihz2;
        return sx + syy + szz;
    }
    template <typename F>
    __device__ __forceinline__ void each(const F &f) const {
#pragma unroll
        for (int u = 0; u < Q; ++u)
            if (threadIdx.x + u * NT < L.half) f(u, threadIdx.x + u * NT);
    }
    __device__ __forceinline__ void sync() const {
        if (NT == 64) wave_barrier_lds();
        else __syncthreads();
    }
    __device__ __forceinline__ void half_sweep(T *x, T (&own)[Q][2], int c) const {
        each([&](int u, int p) {
            own[u][c] = (b[u][c] + nbsum(x, u, c)) * id[u][c];
            x[base(c) + p] = own[u][c];
        });
        sync();
    }
};

// The way down through one level: the pre-smoothing from x = 0 (the first red
// sweep reads no neighbour, the black one after it red cells alone) and the
// residual after the last black sweep, in FP64 of the red cells alone as in
// the passes of mgmarch.hpp.
template <typename T, int Q, int NT>
__device__ __forceinline__ void tail_down(const LevelDev &L, T *x, const T *bl, T *r, int pre) {
    const TailPairs<T, Q, NT> P(L, bl);
    T own[Q][2];
    if (threadIdx.x < 2) x[P.base(threadIdx.x) + L.half] = T(0);
    P.each([&](int u, int p) {
        own[u][0] = (P.b[u][0] + T(0)) * P.id[u][0];
        x[p] = own[u][0];
    });
    P.sync();
    P.half_sweep(x, own, 1);
    for (int q = 1; q < pre; ++q) {
        P.half_sweep(x, own, 0);
        P.half_sweep(x, own, 1);
    }
    P.each([&](int u, int p) {
#pragma unroll
        for (int c = 0; c < (RES_BLACK<T> ? 2 : 1); ++c)
            r[c * L.half + p] = P.b[u][c] - (T(L.diag[P.di[u][c]]) * own[u][c] - P.nbsum(x, u, c));
    });
    P.sync();
}

// restrict_body's sum from the level's residual in LDS
template <typename T, int NT>
__device__ __forceinline__ void tail_restrict(const LevelDev &F, const T *rf, const LevelDev &Cl, T *bc) {
    const T wt[4] = {T(0.25), T(0.75), T(0.75), T(0.25)};
    const int n = Cl.nx * Cl.ny * Cl.nz, rl = F.nx >> 1;
    const bool px = F.bt[0] == IBMDEM_BC_PERIODIC;
    for (int q = threadIdx.x; q < n; q += NT) {
        int I, J, K;
        lcell_small(Cl, q, I, J, K);
        const bool lo = I == 0 && !px, hi = I == Cl.nx - 1 && !px;
        // the row's pairs I - 1, I, I + 1 (wrapped; unused beyond other sides)
        const int pm = I > 0 ? I - 1 : (px ? rl - 1 : 0), pp = I < rl - 1 ? I + 1 : (px ? 0 : I);
        int fj[4];
#pragma unroll
        for (int c2 = 0; c2 < 4; ++c2) fj[c2] = tile_coord(2 * J - 1 + c2, F.ny, F.bt[2], F.bt[3]);
        T s = T(0);
#pragma unroll
        for (int c3 = 0; c3 < 4; ++c3) {
            const int fk = tile_coord(2 * K - 1 + c3, F.nz, F.bt[4], F.bt[5]);
#pragma unroll
            for (int c2 = 0; c2 < 4; ++c2) {
                const T *row = rf + (fk * F.ny + fj[c2]) * rl;
                s = restrict_row(s, wt[c3] * wt[c2], ((fj[c2] + fk) & 1) == 0, lo, hi,
                                 [&](int d) { return row[d < 0 ? pm : (d > 0 ? pp : I)]; },
                                 [&](int d) { return row[F.half + (d < 0 ? pm : (d > 0 ? pp : I))]; });
            }
        }
        bc[q] = T(0.125) * s;
    }
    if (NT == 64) wave_barrier_lds();
    else __syncthreads();
}

// The way up: the correction of the red cells from the coarser level (hs:
// words from its red to its black cells; the fine black cells are swept next)
// and the post-smoothing. xg: the level's x in global memory, or null.
template <typename T, int Q, int NT>
__device__ __forceinline__ void tail_up(const LevelDev &F, T *xf, const T *bl, const LevelDev &Cl, const T *xc, int hs,
                                        int post, T *xg) {
    const TailPairs<T, Q, NT> P(F, bl);
    const T wt[2] = {T(0.75), T(0.25)};
    const int rl = Cl.split ? Cl.nx >> 1 : Cl.nx, fr = F.nx >> 1;
    T own[Q][2];
    P.each([&](int u, int q) {
        const int row = udiv_small(q, fr, F.m_row), k = udiv_small(row, F.ny, F.m_ny), j = row - k * F.ny;
        const int i = 2 * (q - row * fr) + ((j + k) & 1);
        int pi[2], pj[2], pk[2];
        parents(i, Cl.nx, Cl.bt[0], Cl.bt[1], pi[0], pi[1]);
        parents(j, Cl.ny, Cl.bt[2], Cl.bt[3], pj[0], pj[1]);
        parents(k, Cl.nz, Cl.bt[4], Cl.bt[5], pk[0], pk[1]);
        // lidx(Cl, i, j, k) = ((i & 1) ^ ((j + k) & 1)) * half + row(j, k) + (i >> 1)
        // when split, row(j, k) + i otherwise: its parts per parent coordinate
        int xo[2], xp[2], ro[4], rp[4];
        for (int a = 0; a < 2; ++a) {
            xo[a] = Cl.split ? pi[a] >> 1 : pi[a];
            xp[a] = pi[a] & 1;
        }
        for (int c3 = 0; c3 < 2; ++c3)
            for (int c2 = 0; c2 < 2; ++c2) {
                ro[2 * c3 + c2] = (pk[c3] * Cl.ny + pj[c2]) * rl;
                rp[2 * c3 + c2] = (pj[c2] + pk[c3]) & 1;
            }
        T s = T(0);
        for (int c3 = 0; c3 < 2; ++c3)
            for (int c2 = 0; c2 < 2; ++c2)
                for (int c1 = 0; c1 < 2; ++c1) {
                    T w = wt[c3] * wt[c2] * wt[c1];
                    const int r = 2 * c3 + c2;
                    s = s + w * xc[(xp[c1] ^ rp[r]) * hs + ro[r] + xo[c1]];
                }
        own[u][0] = xf[q] + s;
        xf[q] = own[u][0];
        own[u][1] = xf[P.base(1) + q];
    });
    P.sync();
    for (int q = 0; q < post; ++q) {
        P.half_sweep(xf, own, 1);
        P.half_sweep(xf, own, 0);
    }
    if (xg)
        P.each([&](int u, int p) {
            xg[p] = own[u][0];
            xg[F.half + p] = own[u][1];
        });
}

// The coarsest level (n <= COARSE_LDS cells, consistent red-black colouring)
// on wavefront 0: neighbour tables whose missing (wall) neighbours point at
// the zero slot x[n], then the symmetric sweeps of coarse_wg (colour 1 once
// where the order turns).
template <typename T>
__device__ __forceinline__ void tail_coarse(const LevelDev &L, T *x, const T *b, int sweeps,
                                            short (*nb)[COARSE_LDS], T *id, unsigned char *col) {
    const int n = L.nx * L.ny * L.nz;
    const int m[3] = {L.nx, L.ny, L.nz};
    for (int q = threadIdx.x; q < n; q += 64) {
        int a[3];
        lcell_small(L, q, a[0], a[1], a[2]);
        for (int d = 0; d < 3; ++d)
            for (int dir = 0; dir < 2; ++dir) {
                int p[3] = {a[0], a[1], a[2]};
                const int v = p[d] + (dir ? 1 : -1);
                int idx;
                if (v < 0) idx = L.bt[2 * d] != IBMDEM_BC_PERIODIC ? -1 : v + m[d];
                else if (v >= m[d]) idx = L.bt[2 * d + 1] != IBMDEM_BC_PERIODIC ? -1 : v - m[d];
                else idx = v;
                p[d] = idx;
                nb[2 * d + dir][q] = (short)(idx < 0 ? n : lidx(L, p[0], p[1], p[2]));
            }
        id[q] = T(L.idiag[diag_index(L, a[0], a[1], a[2])]);
        col[q] = (unsigned char)((a[0] + a[1] + a[2]) & 1);
        x[q] = T(0);
    }
    if (threadIdx.x == 0) x[n] = T(0);
    wave_barrier_lds();
    const T ihx2 = T(L.ihx2), ihy2 = T(L.ihy2), ihz2 = T(L.ihz2);
    auto half = [&](int color) {
        for (int q = threadIdx.x; q < n; q += 64)
            if (col[q] == color) {
                const T sx = (x[nb[0][q]] + x[nb[1][q]]) * ihx2;
                const T sy = (x[nb[2][q]] + x[nb[3][q]]) * ihy2;
                const T sz = (x[nb[4][q]] + x[nb[5][q]]) * ihz2;
                x[q] = (b[q] + (sx + sy + sz)) * id[q];
            }
        wave_barrier_lds();
    };
    if (coarse_sweeps_small<T>(x, b, nb, id, col, n, sweeps, ihx2, ihy2, ihz2)) return;
    for (int s = 1; s < 2 * sweeps; ++s) { half(0); half(1); }
    half(0);
}

template <typename T>
__device__ __forceinline__ void vcycle_tail_body(const Blk &kb, const LevelDev *__restrict__ lev, int first, int last,
                                                        const T *__restrict__ bg, T *__restrict__ xg, int pre,
                                                        int post, int coarse_sweeps,
                                                        const double *__restrict__ stop) {
    if (*stop != 0.0) return;
    __shared__ T mem[TAIL_BYTES / sizeof(T) + 2 * TAIL_MAXLEV];
    __shared__ short s_nb[6][COARSE_LDS];
    __shared__ T s_id[COARSE_LDS];
    __shared__ unsigned char s_col[COARSE_LDS];
    __shared__ int s_off[IBMDEM_MAX_LEVELS + 1];   // level l: x at off, then b, then r
    // the levels' descriptors (sizes, boundary types, diagonal tables) in
    // LDS: every phase reads them, and a level's first phase would otherwise
    // wait on its scalar and table loads from global memory
    __shared__ LevelDev s_lev[TAIL_MAXLEV];
    {
        const int nw = (last - first + 1) * (int)(sizeof(LevelDev) / 4);
        const int *src = (const int *)(lev + first);
        int *dst = (int *)s_lev;
        for (int w = kb.tx; w < nw; w += TAIL_T) dst[w] = src[w];
    }
    if (kb.tx == 0) {
        int off = 0;
        for (int l = first; l <= last; ++l) {
            s_off[l] = off;
            off += 3 * lev[l].nx * lev[l].ny * lev[l].nz + (l == last ? 1 : 2);
        }
    }
    __syncthreads();
    constexpr int QM = (TAIL_BYTES / (3 * sizeof(T)) / 2 + TAIL_T - 1) / TAIL_T;   // pairs of the largest level
    auto LV = [&](int l) -> const LevelDev & { return s_lev[l - first]; };
    auto cells = [&](int l) { return LV(l).nx * LV(l).ny * LV(l).nz; };
    auto X = [&](int l) { return mem + s_off[l]; };
    auto B = [&](int l) { return mem + s_off[l] + cells(l) + (l == last ? 1 : 2); };
    auto R = [&](int l) { return B(l) + cells(l); };
    auto HS = [&](int l) { return l == last ? LV(l).half : LV(l).half + 1; };   // red to black cells of x
    // the levels from `wave` on have at most a pair per lane of one wavefront,
    // which runs them without a work-group barrier
    int wave = first;
    while (wave < last && LV(wave).half > 64) ++wave;
    for (int l = first; l < wave; ++l) {
        const T *b = l == first ? bg : B(l);
        if (LV(l).half > TAIL_T) tail_down<T, QM, TAIL_T>(LV(l), X(l), b, R(l), pre);
        else tail_down<T, 1, TAIL_T>(LV(l), X(l), b, R(l), pre);
        tail_restrict<T, TAIL_T>(LV(l), R(l), LV(l + 1), B(l + 1));
    }
    if (kb.tx < 64) {
        for (int l = wave; l < last; ++l) {
            tail_down<T, 1, 64>(LV(l), X(l), l == first ? bg : B(l), R(l), pre);
            tail_restrict<T, 64>(LV(l), R(l), LV(l + 1), B(l + 1));
        }
        tail_coarse(LV(last), X(last), B(last), coarse_sweeps, s_nb, s_id, s_col);
        for (int l = last - 1; l >= wave; --l)
            tail_up<T, 1, 64>(LV(l), X(l), l == first ? bg : B(l), LV(l + 1), X(l + 1), HS(l + 1), post,
                              l == first ? xg : nullptr);
    }
    __syncthreads();
    for (int l = wave - 1; l >= first; --l) {
        const T *b = l == first ? bg : B(l);
        T *g = l == first ? xg : nullptr;
        if (LV(l).half > TAIL_T) tail_up<T, QM, TAIL_T>(LV(l), X(l), b, LV(l + 1), X(l + 1), HS(l + 1), post, g);
        else tail_up<T, 1, TAIL_T>(LV(l), X(l), b, LV(l + 1), X(l + 1), HS(l + 1), post, g);
    }
}
template <typename T>
__global__ __launch_bounds__(TAIL_T) void k_vcycle_tail(const LevelDev *__restrict__ lev, int first, int last,
                                                        const T *__restrict__ bg, T *__restrict__ xg, int pre,
                                                        int post, int coarse_sweeps,
                                                        const double *__restrict__ stop) {
    vcycle_tail_body<T>(hw_blk(), lev, first, last, bg, xg, pre, post, coarse_sweeps, stop);
}

// ---------------------------------------------------------------------------
// CG kernels (FP64)
// ---------------------------------------------------------------------------
// Ap = A p and one partial sum of p.Ap per block. A thread owns an x-pair
// (both colours), a block 64 x 4 pairs of one plane: a block's plane
// neighbours are read by the block
// gridDim.x * gridDim.y positions away, a multiple of the XCD count for the
// level-0 shapes, so they are served by the same L2.
__device__ __forceinline__ void matvec_dot_body(const Blk &kb, const LevelDev &L, const double *__restrict__ p,
                                                   double *__restrict__ Ap, double *__restrict__ partial,
                                                   const double *__restrict__ scal) {
    if (scal[SC_CONV] != 0.0) return;
    __shared__ double red[RB];
    // a thread takes the x-pair ip of two adjacent rows j0, j0 + 1 (blocks as
    // sweep_shape's); when both rows exist, a cell's north neighbour in row
    // j0 is row j0 + 1's value of the same cell of its pair, and a cell's
    // south neighbour in row j0 + 1 is row j0's: those loads are shared
    const int ip = kb.bx * kb.dx + kb.tx;
    const int j0 = (kb.by * kb.dy + kb.ty) * 2, k = kb.bz;
    double s = 0.0;
    if (L.split) {
        const int ipc = min(ip, (L.nx >> 1) - 1);
        const double dg_int = L.diag[DIAG_INTERIOR];
        const bool adj = j0 + 1 < L.ny;
        PairGeo g[2];
        bool ok[2];
        long oo[2][2];
        double pv[2][2], dgv[2][2], a[2][2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            ok[r] = j0 + r < L.ny && ip < (L.nx >> 1);
            g[r] = pair_geo(L, ipc, min(j0 + r, L.ny - 1), k);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                oo[r][h] = (long)(h ? 1 - g[r].ca : g[r].ca) * L.half + g[r].pos;
                const int di = (h ? g[r].cx1 : g[r].cx0) * 16 + g[r].cyz;
                double dg;
                if (di == DIAG_INTERIOR) dg = dg_int;
                else dg = L.diag[di];
                dgv[r][h] = dg;
                pv[r][h] = p[oo[r][h]];
            }
        }
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const PairGeo &G = g[r];
                const double *q = p + (long)(h ? G.ca : 1 - G.ca) * L.half + G.pos;
                const double xo = q[h == 0 ? (G.hw ? G.dw : 0) : (G.he ? G.de : 0)];
                const double zb = q[G.hb ? G.db : 0], zt = q[G.ht ? G.dt : 0];
                double ys, yn;
                if (r == 0) {
                    ys = q[G.hs ? G.ds : 0];
                    if (adj) yn = pv[1][h];
                    else yn = q[G.hn ? G.dn : 0];
                } else {
                    yn = q[G.hn ? G.dn : 0];
                    if (adj) ys = pv[0][h];
                    else ys = q[G.hs ? G.ds : 0];
                }
                a[r][h] = dgv[r][h] * pv[r][h] - nbsum_pair_vals(G, h, pv[r][1 - h], xo, ys, yn, zb, zt, L);
            }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            if (!ok[r]) continue;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                Ap[oo[r][h]] = a[r][h];
                s += pv[r][h] * a[r][h];
            }
        }
    } else {
        for (int r = 0; r < 2; ++r) {
            const int j = j0 + r;
            if (j >= L.ny) break;
            for (int h = 0; h < 2; ++h) {
                const int i = 2 * ip + h;
                if (i >= L.nx) break;
                const int o = lidx(L, i, j, k);
                const double av = L.diag[diag_index(L, i, j, k)] * p[o] - nbsum(p, L, i, j, k);
                Ap[o] = av;
                s += p[o] * av;
            }
        }
    }
    const int t = kb.ty * kb.dx + kb.tx;
    s = tree_sum<RB>(s, t, red);
    if (t == 0) partial[((long)kb.bz * kb.gy + kb.by) * kb.gx + kb.bx] = s;
}
__global__ __launch_bounds__(RB) void k_matvec_dot(LevelDev L, const double *__restrict__ p,
                                                   double *__restrict__ Ap, double *__restrict__ partial,
                                                   const double *__restrict__ scal) {
    matvec_dot_body(hw_blk(), L, p, Ap, partial, scal);
}

// The same product with each thread on two adjacent x-pairs (pc, pc + 1,
// pc even) of its two rows, on split levels whose rows hold an even number
// of pairs (sweep_shape's condition and launch shape): both cells of the two
// pairs come from two-value loads of the two colour halves, and a cell's
// x neighbours are mostly its pairs' other cells. Each Ap value is
// matvec_dot_body's (the same diagonal product less nbsum_pair_vals' sum);
// the partial sums follow this kernel's blocks.
__device__ __forceinline__ void matvec2_dot_body(const Blk &kb, const LevelDev &L, const double *__restrict__ p,
                                                 double *__restrict__ Ap, double *__restrict__ partial,
                                                 const double *__restrict__ scal) {
    if (scal[SC_CONV] != 0.0) return;
    __shared__ double red[RB];
    const double ihx2 = L.ihx2, ihy2 = L.ihy2, ihz2 = L.ihz2;
    const double dg_int = L.diag[DIAG_INTERIOR];
    const int rl = L.nx >> 1, pl = rl * L.ny;
    const int p0 = 2 * (kb.bx * kb.dx + kb.tx), k = kb.bz;
    const int j0 = (kb.by * kb.dy + kb.ty) * 2;
    const bool px = L.bt[0] == IBMDEM_BC_PERIODIC, py = L.bt[2] == IBMDEM_BC_PERIODIC,
               pz = L.bt[4] == IBMDEM_BC_PERIODIC;
    const int pc = min(p0, rl - 2);
    const bool hw = pc > 0 || px, he = pc + 2 < rl || px;
    const int dw = pc > 0 ? -1 : rl - 1, de = pc + 2 < rl ? 2 : 2 - rl;
    const bool hb = k > 0 || pz, ht = k < L.nz - 1 || pz;
    const int db = k > 0 ? -pl : (L.nz - 1) * pl, dt = k < L.nz - 1 ? pl : -(L.nz - 1) * pl;
    const int cz = diag_count(k, L.nz, L.bt[4], L.bt[5]);
    const bool adj = j0 + 1 < L.ny;
    // per row: v[r][hh][c] = the value of cell h = hh of pair pc + c (hh 0:
    // the even cell, in half ca; 1: the odd cell, in half 1 - ca)
    bool ok[2], hs[2], hn[2];
    int pos[2], ca[2], cyz[2];
    double v[2][2][2], zb[2][2][2], zt[2][2][2], xw0[2], xe1[2], ys[2][2][2], yn[2][2][2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int j = min(j0 + r, L.ny - 1);
        ok[r] = j0 + r < L.ny && p0 < rl;
        pos[r] = (k * L.ny + j) * rl + pc;
        ca[r] = (j + k) & 1;
        hs[r] = j > 0 || py;
        hn[r] = j < L.ny - 1 || py;
        cyz[r] = diag_count(j, L.ny, L.bt[2], L.bt[3]) * 4 + cz;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const double *q = p + (long)(hh ? 1 - ca[r] : ca[r]) * L.half + pos[r];
            ld2(q, v[r][hh][0], v[r][hh][1]);
            ld2(q + (hb ? db : 0), zb[r][hh][0], zb[r][hh][1]);
            ld2(q + (ht ? dt : 0), zt[r][hh][0], zt[r][hh][1]);
        }
        // the west neighbour of pair pc's even cell (the odd cell of pair
        // pc - 1) and the east neighbour of pair pc + 1's odd cell (the even
        // cell of pair pc + 2)
        xw0[r] = p[(long)(1 - ca[r]) * L.half + pos[r] + (hw ? dw : 0)];
        xe1[r] = p[(long)ca[r] * L.half + pos[r] + (he ? de : 0)];
    }
    // y neighbours: cell (i, j +- 1) is in the other half of its row at the
    // same pair position; row 0's north and row 1's south are the other
    // row's values when both rows exist
    {
        const int jr0 = min(j0, L.ny - 1), jr1 = min(j0 + 1, L.ny - 1);
        const int ds0 = jr0 > 0 ? -rl : (L.ny - 1) * rl, dn1 = jr1 < L.ny - 1 ? rl : -(L.ny - 1) * rl;
        const int dn0 = jr0 < L.ny - 1 ? rl : -(L.ny - 1) * rl;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            // cell h of row 0 has colour ca[0] ^ h; its south neighbour lies in
            // the half of that colour's opposite, i.e. half (ca[0] ^ h) ^ 1 of row jr0 - 1
            const double *q0 = p + (long)((ca[0] ^ hh) ^ 1) * L.half + pos[0];
            const double *q1 = p + (long)((ca[1] ^ hh) ^ 1) * L.half + pos[1];
            ld2(q0 + (hs[0] ? ds0 : 0), ys[0][hh][0], ys[0][hh][1]);
            ld2(q1 + (hn[1] ? dn1 : 0), yn[1][hh][0], yn[1][hh][1]);
            if (adj) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    yn[0][hh][c] = v[1][hh][c];
                    ys[1][hh][c] = v[0][hh][c];
                }
            } else {
                ld2(q0 + (hn[0] ? dn0 : 0), yn[0][hh][0], yn[0][hh][1]);
                ys[1][hh][0] = ys[0][hh][0];
                ys[1][hh][1] = ys[0][hh][1];
            }
        }
    }
    double s = 0.0;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        double a[2][2];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                // nbsum_pair_vals of cell hh of pair pc + c: its pair's other
                // cell and its other x neighbour (the adjacent pair's cell)
                const double part = v[r][1 - hh][c];
                double xo;
                bool pw = true, pe = true;
                if (hh == 0) {
                    xo = c == 0 ? xw0[r] : v[r][1][0];
                    pw = c == 0 ? hw : true;
                } else {
                    xo = c == 0 ? v[r][0][1] : xe1[r];
                    pe = c == 0 ? true : he;
                }
                const double vw = hh == 0 ? xo : part, ve = hh == 0 ? part : xo;
                const double xw = pw ? vw : 0.0, xe = pe ? ve : 0.0;
                const double xs = hs[r] ? ys[r][hh][c] : 0.0, xn = hn[r] ? yn[r][hh][c] : 0.0;
                const double xb = hb ? zb[r][1 - hh][c] : 0.0, xt = ht ? zt[r][1 - hh][c] : 0.0;
                const double sx = (xw + xe) * ihx2;
                const double syy = (xs + xn) * ihy2;
                const double szz = (xb + xt) * ihz2;
                const int di = diag_count(2 * (pc + c) + hh, L.nx, L.bt[0], L.bt[1]) * 16 + cyz[r];
                const double dg = di == DIAG_INTERIOR ? dg_int : L.diag[di];
                a[hh][c] = dg * v[r][hh][c] - (sx + syy + szz);
            }
        if (!ok[r]) continue;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            st2(Ap + (long)(hh ? 1 - ca[r] : ca[r]) * L.half + pos[r], a[hh][0], a[hh][1]);
#pragma unroll
            for (int c = 0; c < 2; ++c) s += v[r][hh][c] * a[hh][c];
        }
    }
    const int t = kb.ty * kb.dx + kb.tx;
    s = tree_sum<RB>(s, t, red);
    if (t == 0) partial[((long)kb.bz * kb.gy + kb.by) * kb.gx + kb.bx] = s;
}
__global__ __launch_bounds__(RB) void k_matvec2_dot(LevelDev L, const double *__restrict__ p,
                                                    double *__restrict__ Ap, double *__restrict__ partial,
                                                    const double *__restrict__ scal) {
    matvec2_dot_body(hw_blk(), L, p, Ap, partial, scal);
}

// CG iteration k >= 2, first kernel: p_k = z_k + beta_{k-1} p_{k-1} in place,
// and the deferred x_k = x_{k-1} + alpha_{k-1} p_{k-1}
// (z in the V-cycle's precision; bound by memory: 104 us at 256^3 in FP64,
// 89 us with the mixed form's FP32 z read as it is)
template <typename T>
__device__ __forceinline__ void cg_px_body(const Blk &kb, long n, double *__restrict__ p, const T *__restrict__ z,
                                           double *__restrict__ x, const double *__restrict__ scal) {
    if (scal[SC_CONV] != 0.0) return;
    const double beta = scal[SC_BETA], alpha = scal[SC_ALPHA];
    for (long q = (long)kb.bx * RED_T + kb.tx; q < n; q += (long)kb.gx * RED_T) {
        const double po = p[q];
        p[q] = double(z[q]) + beta * po;
        x[q] = x[q] + alpha * po;
    }
}
template <typename T>
__global__ __launch_bounds__(RED_T) void k_cg_px(long n, double *__restrict__ p, const T *__restrict__ z,
                                                 double *__restrict__ x, const double *__restrict__ scal) {
    cg_px_body(hw_blk(), n, p, z, x, scal);
}

// r -= alpha Ap; partial sums of r.r (x is updated one iteration later, by
// k_cg_px or, after the last iteration, by k_gauge)
// (and, in the mixed form, the FP32 copy of r the V-cycle reads)
__device__ __forceinline__ void cg_update_r_body(const Blk &kb, long n, double *__restrict__ r, const double *__restrict__ Ap,
                                                       const double *__restrict__ scal, double *__restrict__ partial,
                                                       float *__restrict__ r32) {
    __shared__ double red[RED_T];
    const double conv = scal[SC_CONV], alpha = scal[SC_ALPHA];
    const long chunk = (n + kb.gx - 1) / kb.gx;
    const long lo = (long)kb.bx * chunk, hi = min(n, lo + chunk);
    double s = 0.0, ro = 0.0, ap = 0.0;
    // a round's loads before the round ahead of it is stored, the first
    // before the wait for the scalars
    auto load = [&](long a) {
        if (a < hi) { ro = r[a]; ap = Ap[a]; }
    };
    long q = lo + kb.tx;
    load(q);
    if (conv != 0.0) return;
    while (q < hi) {
        const double rq = ro - alpha * ap;
        load(q + RED_T);
        r[q] = rq;
        if (r32) r32[q] = float(rq);
        s += rq * rq;
        q += RED_T;
    }
    const double t = tree_sum<RED_T>(s, kb.tx, red);
    if (kb.tx == 0) partial[kb.bx] = t;
}
__global__ __launch_bounds__(RED_T) void k_cg_update_r(long n, double *__restrict__ r, const double *__restrict__ Ap,
                                                       const double *__restrict__ scal, double *__restrict__ partial,
                                                       float *__restrict__ r32) {
    cg_update_r_body(hw_blk(), n, r, Ap, scal, partial, r32);
}

// partial sums of a.b
__device__ __forceinline__ void dot_body(const Blk &kb, long n, const double *__restrict__ a,
                                         const double *__restrict__ b, double *__restrict__ partial,
                                         const double *__restrict__ scal) {
    if (scal[SC_CONV] != 0.0) return;
    __shared__ double red[RED_T];
    const long chunk = (n + kb.gx - 1) / kb.gx;
    const long lo = (long)kb.bx * chunk, hi = min(n, lo + chunk);
    // four independent sums over the thread's strided elements (four
    // rounds of loads in flight), then (s0 + s1) + (s2 + s3): a fixed
    // association set by (n, grid, RED_T)
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    long q = lo + kb.tx;
    for (; q + 3 * RED_T < hi; q += 4 * RED_T) {
        s0 += a[q] * b[q];
        s1 += a[q + RED_T] * b[q + RED_T];
        s2 += a[q + 2 * RED_T] * b[q + 2 * RED_T];
        s3 += a[q + 3 * RED_T] * b[q + 3 * RED_T];
    }
    for (; q < hi; q += RED_T) s0 += a[q] * b[q];
    const double t = tree_sum<RED_T>((s0 + s1) + (s2 + s3), kb.tx, red);
    if (kb.tx == 0) partial[kb.bx] = t;
}
__global__ __launch_bounds__(RED_T) void k_dot(long n, const double *__restrict__ a, const double *__restrict__ b,
                                               double *__restrict__ partial, const double *__restrict__ scal) {
    dot_body(hw_blk(), n, a, b, partial, scal);
}

// finalize a partial sum into scal[slot]; op: 0 store, 1 alpha = rz/pAp,
// 2 beta = rz_new/rz and rz = rz_new, 3 r.r and the convergence test of
// iteration it, 4 ||b||^2 and tol = rtol ||b||
// Each thread sums its strided partials with four independent accumulators
// (the loads of a round are in flight together), then a tree.
constexpr int FIN_T = 1024;
__device__ __forceinline__ void final_body(const Blk &kb, const double *__restrict__ partial, int np, double *__restrict__ scal,
                                                 int slot, int op, int it, double rtol) {
    __shared__ double red[FIN_T];
    // one block, bound by its chain of latencies: the stop flag and the
    // scalars are waited for with the partial sums (at 128^3 in FP64 the
    // solve's three reductions an iteration take 1 to 1.5 % of a step less
    // than with a wait of its own for the flag and a barrier per tree level)
    const double conv = scal[SC_CONV], rz = scal[SC_RZ], tol = scal[SC_TOL];
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    int q = kb.tx;
    for (; q + 3 * FIN_T < np; q += 4 * FIN_T)
        for (int u = 0; u < 4; ++u) a[u] += partial[q + u * FIN_T];
    for (int u = 0; q < np; q += FIN_T, ++u) a[u] += partial[q];
    const double t = tree_sum<FIN_T>((a[0] + a[1]) + (a[2] + a[3]), kb.tx, red);
    if (conv != 0.0) return;
    if (kb.tx == 0) {
        scal[slot] = t;
        if (op == 1) scal[SC_ALPHA] = rz / t;
        if (op == 2) { scal[SC_BETA] = t / rz; scal[SC_RZ] = t; }
        if (op == 3) scal[SC_DONE] = it;
        if (op == 3 && (sqrt(t) <= tol || !(t == t))) { scal[SC_CONV] = 1.0; scal[SC_ITER] = it; }
        if (op == 4) {
            scal[SC_TOL] = rtol * sqrt(t);
            if (t == 0.0) { scal[SC_CONV] = 1.0; scal[SC_ITER] = 0; scal[SC_RR] = 0.0; }
        }
    }
}
__global__ __launch_bounds__(FIN_T) void k_final(const double *__restrict__ partial, int np, double *__restrict__ scal,
                                                 int slot, int op, int it, double rtol) {
    final_body(hw_blk(), partial, np, scal, slot, op, it, rtol);
}


// r = rhs with the pinned row, x = 0; r and x in level-0 storage, rhs in
// field order (cell (0,0,0) is position 0 of both). A thread takes the
// x-pair (2p, 2p+1) of row (j, k), blocks of shape_for over the level's x-pairs.
__device__ __forceinline__ void cg_init_body(const Blk &kb, const LevelDev &L, const double *__restrict__ rhs,
                                             double *__restrict__ r, double *__restrict__ x,
                                             double *__restrict__ scal, float *__restrict__ r32) {
    const int ip = kb.bx * kb.dx + kb.tx;
    const int j = kb.by * kb.dy + kb.ty, k = kb.bz;
    const double pin = scal[SC_PIN];
    if (kb.bx == 0 && kb.by == 0 && kb.bz == 0 && kb.tx == 0 && kb.ty == 0) {
        scal[SC_CONV] = 0.0;
        scal[SC_ITER] = 0.0;
        scal[SC_DONE] = 0.0;
    }
    if (j >= L.ny || 2 * ip >= L.nx) return;
    // both cells' right-hand sides are loaded before the stores (the second
    // from the first's place when the row ends at an odd length)
    const bool two = 2 * ip + 1 < L.nx;
    const long f0 = ((long)k * L.ny + j) * L.nx + 2 * ip;
    const double v[2] = {rhs[f0], rhs[f0 + (two ? 1 : 0)]};
    for (int h = 0; h < (two ? 2 : 1); ++h) {
        const int q = lidx(L, 2 * ip + h, j, k);
        const double rq = (q == 0 && !L.dirichlet) ? -pin : v[h];
        r[q] = rq;
        if (r32) r32[q] = float(rq);   // the mixed form's FP32 copy
        x[q] = 0.0;
    }
}
__global__ __launch_bounds__(RB) void k_cg_init(LevelDev L, const double *__restrict__ rhs,
                                                double *__restrict__ r, double *__restrict__ x,
                                                double *__restrict__ scal, float *__restrict__ r32) {
    cg_init_body(hw_blk(), L, rhs, r, x, scal, r32);
}

template <typename T>
__device__ __forceinline__ void copy_body(const Blk &kb, long n, double *__restrict__ d, const T *__restrict__ s) {
    for (long q = (long)kb.bx * RED_T + kb.tx; q < n; q += (long)kb.gx * RED_T) d[q] = s[q];
}
template <typename T>
__global__ __launch_bounds__(RED_T) void k_copy(long n, double *__restrict__ d, const T *__restrict__ s) {
    copy_body(hw_blk(), n, d, s);
}
template <typename TD, typename TS>
__global__ __launch_bounds__(RED_T) void k_convert(long n, TD *__restrict__ d, const TS *__restrict__ s,
                                                   const double *__restrict__ stop) {
    if (*stop != 0.0) return;
    for (long q = (long)blockIdx.x * RED_T + threadIdx.x; q < n; q += (long)gridDim.x * RED_T) d[q] = TD(s[q]);
}

// gauge P'(1,1,1) = 0: pcorr = x - x(1,1,1), x in level-0 storage, pcorr in
// field order (no shift with an outflow side, where P' = 0 on the face), x
// taking the last completed CG iteration's deferred update x + alpha p
// (thread per x-pair of a row, blocks of shape_for over the x-pairs)
__device__ __forceinline__ void gauge_body(const Blk &kb, const LevelDev &L, const double *__restrict__ x,
                                              const double *__restrict__ p, const double *__restrict__ scal,
                                              double *__restrict__ pc) {
    const int done = (int)scal[SC_DONE];
    const double alpha = done > 0 ? scal[SC_ALPHA] : 0.0;
    auto xv = [&](long q) { return done > 0 ? x[q] + alpha * p[q] : x[q]; };
    const double x0 = L.dirichlet ? 0.0 : xv(0);
    const int ip = kb.bx * kb.dx + kb.tx;
    const int j = kb.by * kb.dy + kb.ty, k = kb.bz;
    if (j >= L.ny || 2 * ip >= L.nx) return;
    // both cells' values are loaded before the stores (the second from the
    // first's place when the row ends at an odd length)
    const bool two = 2 * ip + 1 < L.nx;
    const double v0 = xv(lidx(L, 2 * ip, j, k)), v1 = xv(lidx(L, two ? 2 * ip + 1 : 2 * ip, j, k));
    const long f0 = ((long)k * L.ny + j) * L.nx + 2 * ip;
    pc[f0] = v0 - x0;
    if (two) pc[f0 + 1] = v1 - x0;
}
__global__ __launch_bounds__(RB) void k_gauge(LevelDev L, const double *__restrict__ x,
                                              const double *__restrict__ p, const double *__restrict__ scal,
                                              double *__restrict__ pc) {
    gauge_body(hw_blk(), L, x, p, scal, pc);
}

int stream_blocks(long n) { return (int)std::min<long>(4096, std::max<long>(1, (n + RED_T - 1) / RED_T)); }

LevelDev make_level(int nx, int ny, int nz, const int bt[6], const double h[3]) {
    LevelDev L;
    std::memset(&L, 0, sizeof L);
    L.nx = nx; L.ny = ny; L.nz = nz;
    for (int s = 0; s < 6; ++s) L.bt[s] = bt[s];
    L.ihx2 = 1.0 / (h[0] * h[0]);
    L.ihy2 = 1.0 / (h[1] * h[1]);
    L.ihz2 = 1.0 / (h[2] * h[2]);
    for (int cx = 0; cx < 4; ++cx)
        for (int cy = 0; cy < 4; ++cy)
            for (int cz = 0; cz < 4; ++cz) {
                double dsum0 = cx * L.ihx2, dsum1 = cy * L.ihy2, dsum2 = cz * L.ihz2;
                double d = dsum0 + dsum1 + dsum2;
                L.diag[cx * 16 + cy * 4 + cz] = d;
                L.idiag[cx * 16 + cy * 4 + cz] = d > 0 ? 1.0 / d : 0.0;
            }
    L.dirichlet = 0;
    for (int s = 0; s < 6; ++s)
        if (bt[s] == IBMDEM_BC_OUTFLOW) L.dirichlet = 1;
    const int n[3] = {nx, ny, nz};
    L.rb_valid = 1;
    for (int d = 0; d < 3; ++d)
        if (bt[2 * d] == IBMDEM_BC_PERIODIC && (n[d] % 2)) L.rb_valid = 0;
    L.split = (nx % 2) == 0 ? 1 : 0;
    L.half = L.split ? nx * ny * nz / 2 : 0;
    L.m_row = udiv_magic(L.split ? nx / 2 : nx);
    L.m_ny = udiv_magic(ny);
    L.m_nxy = udiv_magic(nx * ny);
    return L;
}

// pairs per thread of a level's passes: two where its rows hold an even number
int march_pw(const LevelDev &d) { return (d.nx >> 1) % 2 == 0 ? 2 : 1; }

// Levels of up to tile_cells() cells smooth in tiles (mgtile.hpp: two launches
// a visit with up to two sweeps each way), larger ones in marching passes
// (mgmarch.hpp: five, six in FP32). Tiles save launches and gaps, passes the
// halo's work. A CG iteration with the level in tiles and in passes, us, by
// (pre, post), in FP64 with 0.51 M cells (80^3), 0.74 M (80x96x96), 0.88 M
// (96^3), 1.05 M (64x64x256) and 1.12 M (104^3):
//   (2,2)  152/187  182/193  185/193  196/187  210/205
//   (4,4)  224/290  267/291  273/298  290/286  306/306
//   (1,1)  140/147  168/160  168/156  177/152  194/167
//   (2,1)  148/168  178/178  179/176  189/170  205/186
//   (3,3)  215/254  256/256  261/259  277/251  294/269
// A launch of one sweep has the halo of two, so odd counts end earlier. Level 1
// in FP32 meets later (0.51 M 327/362, 0.88 M 433/452, 1.12 M 518/523, 1.40 M
// 680/677, 2.10 M 781/732), by 1 % or less where the line would differ. The
// mixed form's level 0 always marches (its r.z sums, rz_half_body).
long tile_cells(int pre, int post) { return (pre | post) & 1 ? 600000 : 900000; }
template <typename T>
bool tile_level(const ibmdem_ctx *c, int l) {
    return (l > 0 || std::is_same<T, double>::value) && c->lev64[l].n <= tile_cells(c->cs.mg_pre, c->cs.mg_post);
}

template <typename T, int MODE, bool FROMB, bool PRO = false>
void launch_march(hipStream_t s, const LevelDev &d, const T *xin, const T *b, T *out, T *out2, double *partial,
                  const double *stop, const T *xc = nullptr) {
    const int pw = march_pw(d);
    const MarchShape sh = march_shape<T>(d, pw);
    const dim3 grid(8 * div_up(sh.ntx * sh.nty * sh.nzc, 8)), block(MT);
    if (pw == 2)
        hipLaunchKernelGGL((k_march<T, 2, MODE, FROMB, PRO>), grid, block, 0, s, d, xin, b, out, out2, partial, xc,
                           stop);
    else
        hipLaunchKernelGGL((k_march<T, 1, MODE, FROMB, PRO>), grid, block, 0, s, d, xin, b, out, out2, partial, xc,
                           stop);
}

// the launches of a level in tiles (mgtile.hpp)
template <typename T>
void launch_tile_down(hipStream_t s, TileSrc src, const MGLevel<T> &L, const MGLevel<T> &C, const T *xin, bool more,
                      T *xr, const double *stop) {
    const dim3 grid = tile_grid(L.d), block(TileDown::NT);
    if (src == TS_B)
        hipLaunchKernelGGL((k_tile_down<T, TS_B>), grid, block, 0, s, L.d, L.b, xin, more, xr, C.d, C.b, stop);
    else
        hipLaunchKernelGGL((k_tile_down<T, TS_X>), grid, block, 0, s, L.d, L.b, xin, more, xr, C.d, C.b, stop);
}
template <typename T>
void launch_tile_up(hipStream_t s, TileSrc src, const MGLevel<T> &L, const MGLevel<T> &C, const T *xr, T *x, T *xb,
                    bool two, double *partial, const double *stop) {
    const dim3 grid = tile_grid(L.d), block(TileUp::NT);
    if (src == TS_PROLONG)
        hipLaunchKernelGGL((k_tile_up<T, TS_PROLONG>), grid, block, 0, s, L.d, L.b, xr, x, xb, two, C.d, C.x, partial,
                           stop);
    else if (src == TS_X)
        hipLaunchKernelGGL((k_tile_up<T, TS_X>), grid, block, 0, s, L.d, L.b, xr, x, xb, two, C.d, C.x, partial, stop);
    else
        hipLaunchKernelGGL((k_tile_up<T, TS_B>), grid, block, 0, s, L.d, L.b, xr, x, xb, two, C.d, C.x, partial, stop);
}

// the mixed form's last two sweeps at level 0: the red cells' x from xr, the
// black ones' to x1 and the red ones' to x0
void launch_rz(hipStream_t s, const LevelDev &d, const float *xr, float *x0, float *x1, const double *r64,
               double *partial, const double *stop) {
    const SweepShape sw = sweep_shape(d);
    const long nb = (long)sw.grid.x * sw.grid.y * sw.grid.z;
    for (int q = 0; q < 2; ++q) {   // black, red
        const float *oth = q ? x1 : xr;
        float *own = q ? x0 : x1;
        if (sw.x2)
            hipLaunchKernelGGL(k_rz_half<2>, sw.grid, sw.block, 0, s, d, oth, own, 1 - q, r64, partial, q * nb, stop);
        else
            hipLaunchKernelGGL(k_rz_half<1>, sw.grid, sw.block, 0, s, d, oth, own, 1 - q, r64, partial, q * nb, stop);
    }
}

// Whether a marching level's prolongation is part of its first post-smoothing
// pass (in FP64, when another pass follows that finalizes x). The pass's steps
// take half as long again, which the launch and the traffic saved outweigh on
// large levels: 66 us in place of 41 + 41 at 256^3, 20 in place of 12.7 + 8.7
// at 128^3; on the smallest that march they meet: 19.7 and 12.0 + 7.9 at
// 100x76x130, 18.5 and 11.3 + 6.7 at 64x64x256, with one launch less.
template <typename T>
constexpr bool prolong_fused(int post) {
    return std::is_same<T, double>::value && post >= 2;
}

template <typename T>
int vcycle(ibmdem_ctx *c, MGLevel<T> *lev, int l, bool dot = false) {
    MGLevel<T> &L = lev[l];
    const LevelDev &d = L.d;
    hipStream_t s = c->stream;
    if (l >= c->tail_first) {
        hipLaunchKernelGGL((k_vcycle_tail<T>), dim3(1), dim3(TAIL_T), 0, s, c->dlev, l, c->nlev - 1, L.b, L.x,
                           c->cs.mg_pre, c->cs.mg_post, c->cs.mg_coarse_sweeps, c->scal + SC_CONV);
        CHECK_LAUNCH(c);
        return IBMDEM_OK;
    }
    if (l == c->nlev - 1) {
        launch_coarsest<T>(s, d, c->dlev + l, L.x, L.b, L.r, c->cs.mg_coarse_sweeps, c->scal + SC_CONV);
        CHECK_LAUNCH(c);
        return IBMDEM_OK;
    }
    // Passes of two half sweeps (mgmarch.hpp) on the red half, out of place
    // between the halves of x and r: the pre-smoothing passes in x, the
    // residual in r's red half; the correction into r, the post-smoothing
    // passes in r, the last one into x. At level 0 the pre- and the
    // post-smoothing passes are each timed as one group of launches; a
    // pass's bytes are its red input, b (of both colours) and what it writes
    // (the mixed form's last pass: the FP64 r and z).
    const double *stop = c->scal + SC_CONV;
    T *x0 = L.x, *x1 = L.x + d.half, *r0 = L.r, *r1 = L.r + d.half, *cur = nullptr;
    const double cell = sizeof(T) * (double)L.n;
    double bytes = 0.0;
    MGLevel<T> &C = lev[l + 1];
    if (tile_level<T>(c, l)) {
        // profiled at level 0: b (and from the second launch on the red
        // cells' x) read, the red cells' x written; on the way up b, x read
        // and the red cells' x written, the last time both colours'
        const int pre = c->cs.mg_pre, post = c->cs.mg_post, ns = tile_smooths(pre), nu = tile_ups(post);
        if (l == 0) prof_begin(c, IBMDEM_K_MG_SMOOTH);
        for (int q = 0; q < ns; ++q) {
            T *to = q & 1 ? x1 : x0;
            launch_tile_up<T>(s, q ? TS_X : TS_B, L, C, cur, to, nullptr, tile_smooth_two(pre, q), nullptr, stop);
            CHECK_LAUNCH(c);
            cur = to;
        }
        launch_tile_down<T>(s, ns ? TS_X : TS_B, L, C, cur, pre > 1, r0, stop);
        CHECK_LAUNCH(c);
        if (l == 0) prof_end(c, IBMDEM_K_MG_SMOOTH, (1.5 + 2.0 * ns) * cell, 1 + ns);
        const int rc = vcycle<T>(c, lev, l + 1);
        if (rc) return rc;
        if (l == 0) prof_begin(c, IBMDEM_K_MG_SMOOTH);
        for (int q = 0; q < nu; ++q) {
            const bool last = q == nu - 1;
            T *from = q & 1 ? r1 : r0;
            launch_tile_up<T>(s, q ? TS_X : TS_PROLONG, L, C, from, last ? x0 : (q & 1 ? r0 : r1),
                              last ? x1 : (T *)nullptr, tile_up_two(post, q),
                              dot && l == 0 && last ? c->partial : (double *)nullptr, stop);
            CHECK_LAUNCH(c);
        }
        if (l == 0) prof_end(c, IBMDEM_K_MG_SMOOTH, (2.0 * nu + 0.5) * cell, nu);
        return IBMDEM_OK;
    }
    if (l == 0) prof_begin(c, IBMDEM_K_MG_SMOOTH);
    for (int q = 0; q < c->cs.mg_pre; ++q) {
        if (q == c->cs.mg_pre - 1) {
            if (q == 0) {
                launch_march<T, 1, true>(s, d, nullptr, L.b, r0, x0, nullptr, stop);
                cur = x0;
            } else {
                launch_march<T, 1, false>(s, d, cur, L.b, r0, nullptr, nullptr, stop);
            }
            bytes += (RES_BLACK<T> ? 2.5 : 2.0) * cell;
        } else {
            T *to = cur == x0 ? x1 : x0;
            if (q == 0) launch_march<T, 0, true>(s, d, nullptr, L.b, to, nullptr, nullptr, stop);
            else launch_march<T, 0, false>(s, d, cur, L.b, to, nullptr, nullptr, stop);
            bytes += (q == 0 ? 1.5 : 2.0) * cell;
            cur = to;
        }
        CHECK_LAUNCH(c);
    }
    if (l == 0) prof_end(c, IBMDEM_K_MG_SMOOTH, bytes, c->cs.mg_pre);
    const dim3 cs(div_up(C.d.nx, RS_CX), div_up(C.d.ny, RS_CY), C.d.nz);
    hipLaunchKernelGGL((k_restrict<T>), cs, dim3(RB), 0, s, d, r0, C.d, C.b, stop);
    CHECK_LAUNCH(c);
    int rc = vcycle<T>(c, lev, l + 1);
    if (rc) return rc;
    const bool fused = prolong_fused<T>(c->cs.mg_post);
    const LaunchShape ps = shape_for(d.nx / 2 / march_pw(d), d.ny, d.nz);
    if (!fused) {
        if (march_pw(d) == 2)
            hipLaunchKernelGGL((k_prolong_red<T, 2>), ps.grid, ps.block, 0, s, d, cur, r0, C.d, C.x, stop);
        else
            hipLaunchKernelGGL((k_prolong_red<T, 1>), ps.grid, ps.block, 0, s, d, cur, r0, C.d, C.x, stop);
        CHECK_LAUNCH(c);
    }
    const T *uncorrected = cur;
    cur = r0;
    bytes = 0.0;
    int launches = c->cs.mg_post;
    if (l == 0) prof_begin(c, IBMDEM_K_MG_SMOOTH);
    for (int q = 0; q < c->cs.mg_post; ++q) {
        if (q < c->cs.mg_post - 1) {
            T *to = cur == r0 ? r1 : r0;
            if (q == 0 && fused) {
                if constexpr (std::is_same<T, double>::value)
                    launch_march<T, 0, false, true>(s, d, uncorrected, L.b, to, nullptr, nullptr, stop, C.x);
            } else {
                launch_march<T, 0, false>(s, d, cur, L.b, to, nullptr, nullptr, stop);
            }
            bytes += 2.0 * cell;
            cur = to;
        } else if (dot && l == 0) {
            // the last pass at level 0 finalizes z and leaves the partial
            // sums of r.z (the mixed form reads the FP64 r)
            if constexpr (std::is_same<T, double>::value) {
                launch_march<T, 2, false>(s, d, cur, L.b, x0, x1, c->partial, stop);
                bytes += 2.5 * cell;
            } else {
                launch_rz(s, d, cur, x0, x1, c->cg_r, c->partial, stop);
                ++launches;   // its two sweeps are a launch each
                bytes += 2.0 * cell + 8.0 * (double)L.n;
            }
        } else {
            launch_march<T, 3, false>(s, d, cur, L.b, x0, x1, nullptr, stop);
            bytes += 2.5 * cell;
        }
        CHECK_LAUNCH(c);
    }
    if (l == 0) prof_end(c, IBMDEM_K_MG_SMOOTH, bytes, launches);
    return IBMDEM_OK;
}

// partial sums of r.z the last level-0 launches leave
int rz_blocks(const ibmdem_ctx *c) {
    const LevelDev &d = c->lev64[0].d;
    if (c->cs.precision == IBMDEM_MIXED) {
        const dim3 g = sweep_shape(d).grid;
        return 2 * (int)(g.x * g.y * g.z);
    }
    if (tile_level<double>(c, 0)) {
        const dim3 g = tile_grid(d);
        return (int)(g.x * g.y * g.z);
    }
    const MarchShape sh = march_shape<double>(d, march_pw(d));
    return sh.ntx * sh.nty * sh.nzc;
}

int dot_into(ibmdem_ctx *c, const double *a, const double *b, int slot, int op);

// z = M^{-1} r
int precondition(ibmdem_ctx *c) {
    const long n = c->n;
    if (c->cs.precision == IBMDEM_MIXED) {
        hipLaunchKernelGGL((k_convert<float, double>), dim3(stream_blocks(n)), dim3(RED_T), 0, c->stream, n,
                           c->lev32[0].b, c->cg_r, c->scal + SC_CONV);
        CHECK_LAUNCH(c);
        int rc = vcycle<float>(c, c->lev32, 0);
        if (rc) return rc;
        hipLaunchKernelGGL((k_convert<double, float>), dim3(stream_blocks(n)), dim3(RED_T), 0, c->stream, n,
                           c->cg_z, c->lev32[0].x, c->scal + SC_CONV);
        CHECK_LAUNCH(c);
        return IBMDEM_OK;
    }
    c->lev64[0].b = c->cg_r;
    c->lev64[0].x = c->cg_z;
    return vcycle<double>(c, c->lev64, 0);
}

// z = M^{-1} r, then r.z into scal[slot] with k_final's op. In the FP64 form
// with post-smoothing the last level-0 launches leave the partial sums of r.z
// (rz_blocks), so z is not read again.
int precondition_dot(ibmdem_ctx *c, int slot, int op) {
    if (c->cs.mg_post < 1 || c->nlev < 2) {
        int rc = precondition(c);
        if (rc) return rc;
        return dot_into(c, c->cg_r, c->cg_z, slot, op);
    }
    int rc;
    if (c->cs.precision == IBMDEM_MIXED) {
        // the FP32 copy of r was written with r (k_cg_init, k_cg_update_r);
        // the last level-0 sweeps read the FP64 r
        rc = vcycle<float>(c, c->lev32, 0, true);
    } else {
        c->lev64[0].b = c->cg_r;
        c->lev64[0].x = c->cg_z;
        rc = vcycle<double>(c, c->lev64, 0, true);
    }
    if (rc) return rc;
    const int np = rz_blocks(c);
    hipLaunchKernelGGL(k_final, dim3(1), dim3(FIN_T), 0, c->stream, c->partial, np, c->scal, slot, op, 0,
                       c->cs.poisson_rtol);
    CHECK_LAUNCH(c);
    return IBMDEM_OK;
}

int dot_into(ibmdem_ctx *c, const double *a, const double *b, int slot, int op) {
    hipLaunchKernelGGL(k_dot, dim3(RED_BLOCKS), dim3(RED_T), 0, c->stream, c->n, a, b, c->partial, c->scal);
    CHECK_LAUNCH(c);
    hipLaunchKernelGGL(k_final, dim3(1), dim3(FIN_T), 0, c->stream, c->partial, RED_BLOCKS, c->scal, slot, op, 0,
                       c->cs.poisson_rtol);
    CHECK_LAUNCH(c);
    return IBMDEM_OK;
}

int read_scalars(ibmdem_ctx *c) {
    HIPX(c, hipMemcpyAsync(c->scal_host, c->scal, SC_COUNT * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIPX(c, hipStreamSynchronize(c->stream));
    return IBMDEM_OK;
}

}  // namespace

// room for the partial sums of the level-0 matrix-vector product and of the
// last level-0 launches with r.z, in any form
long poisson_partials(int nx, int ny, int nz) {
    const LaunchShape mv = shape_for(div_up(nx, 2), ny, nz);
    long most = (long)mv.grid.x * mv.grid.y * mv.grid.z;
    if (nx % 2 == 0) {
        LevelDev d{};
        d.nx = nx;
        d.ny = ny;
        d.nz = nz;
        d.split = 1;
        const dim3 sw = sweep_shape(d).grid, tl = tile_grid(d);
        const MarchShape ma = march_shape<double>(d, march_pw(d));
        most = std::max(most, 2L * sw.x * sw.y * sw.z);
        most = std::max(most, (long)tl.x * tl.y * tl.z);
        most = std::max(most, (long)ma.ntx * ma.nty * ma.nzc);
    }
    return most;
}

int poisson_setup(ibmdem_ctx *c) {
    int bt[6];
    for (int s = 0; s < 6; ++s) bt[s] = c->g.bt[s];
    double h[3] = {c->g.dx, c->g.dy, c->g.dz};
    int nx = c->g.nx, ny = c->g.ny, nz = c->g.nz;
    const int maxl = c->cs.mg_max_levels > 0 ? std::min(c->cs.mg_max_levels, IBMDEM_MAX_LEVELS) : IBMDEM_MAX_LEVELS;
    c->nlev = 0;
    while (true) {
        LevelDev L = make_level(nx, ny, nz, bt, h);
        long n = (long)nx * ny * nz;
        const int l = c->nlev;
        c->lev64[l].d = L; c->lev64[l].n = n;
        c->lev32[l].d = L; c->lev32[l].n = n;
        int rc;
        if (c->cs.precision == IBMDEM_MIXED) {
            if ((rc = dev_alloc(c, &c->lev32[l].x, n))) return rc;
            if ((rc = dev_alloc(c, &c->lev32[l].b, n))) return rc;
            if ((rc = dev_alloc(c, &c->lev32[l].r, n))) return rc;
        } else {
            if (l > 0) {
                if ((rc = dev_alloc(c, &c->lev64[l].x, n))) return rc;
                if ((rc = dev_alloc(c, &c->lev64[l].b, n))) return rc;
            }
            if ((rc = dev_alloc(c, &c->lev64[l].r, n))) return rc;
        }
        c->nlev++;
        if (c->nlev >= maxl) break;
        if ((nx % 2) || (ny % 2) || (nz % 2)) break;
        if (nx < 4 || ny < 4 || nz < 4) break;
        nx /= 2; ny /= 2; nz /= 2;
        h[0] *= 2; h[1] *= 2; h[2] *= 2;
    }
    int rc;
    // the mixed form reads z where its V-cycle leaves it, in FP32, but for a
    // hierarchy of one level (precondition)
    if ((c->cs.precision != IBMDEM_MIXED || c->nlev < 2) && (rc = dev_alloc(c, &c->cg_z, c->n))) return rc;
    // the small levels whose x, b and r fit the tail work-group's LDS
    // together run as one launch per V-cycle, when the coarsest level suits
    // the one-wavefront table sweeps (IBMDEM_NO_TAIL=1 keeps one launch per
    // operation, for comparison)
    const size_t elem = c->cs.precision == IBMDEM_MIXED ? sizeof(float) : sizeof(double);
    const LevelDev &lc = c->lev64[c->nlev - 1].d;
    c->tail_first = c->nlev;
    if (c->nlev >= 2 && lc.rb_valid && c->lev64[c->nlev - 1].n <= COARSE_LDS) {
        size_t need = elem;   // the zero slot
        for (int l = c->nlev - 1; l >= 1; --l) {
            need += 3 * (size_t)c->lev64[l].n * elem;
            if (need > (size_t)TAIL_BYTES || c->nlev - l > TAIL_MAXLEV) break;
            c->tail_first = l;
        }
        if (c->tail_first == c->nlev - 1) c->tail_first = c->nlev;   // the coarsest alone: one launch as well
    }
    const char *nt = std::getenv("IBMDEM_NO_TAIL");
    if (nt && *nt && *nt != '0') c->tail_first = c->nlev;
    if ((rc = dev_alloc(c, &c->dlev, (size_t)c->nlev))) return rc;
    LevelDev host[IBMDEM_MAX_LEVELS];
    for (int l = 0; l < c->nlev; ++l) host[l] = c->lev64[l].d;
    HIPX(c, hipMemcpyAsync(c->dlev, host, c->nlev * sizeof(LevelDev), hipMemcpyHostToDevice, c->stream));
    HIPX(c, hipStreamSynchronize(c->stream));
    return IBMDEM_OK;
}

namespace {

// one CG iteration (it is its 1-based number), queued without any host wait
int cg_iteration(ibmdem_ctx *c, int it) {
    const long n = c->n;
    hipStream_t s = c->stream;
    int rc;
    const LevelDev &L0 = c->lev64[0].d;
    const SweepShape mv = sweep_shape(L0);   // two rows per thread, two pairs where the level allows
    const int mv_blocks = (int)(mv.grid.x * mv.grid.y * mv.grid.z);
    if (it > 1) {
        if (c->cs.precision == IBMDEM_MIXED)
            hipLaunchKernelGGL(k_cg_px<float>, dim3(stream_blocks(n)), dim3(RED_T), 0, s, n, c->cg_p, c->lev32[0].x,
                               c->cg_x, c->scal);
        else
            hipLaunchKernelGGL(k_cg_px<double>, dim3(stream_blocks(n)), dim3(RED_T), 0, s, n, c->cg_p, c->cg_z,
                               c->cg_x, c->scal);
        CHECK_LAUNCH(c);
    }
    prof_begin(c, IBMDEM_K_MATVEC);
    if (mv.x2)
        hipLaunchKernelGGL(k_matvec2_dot, mv.grid, mv.block, 0, s, L0, c->cg_p, c->cg_Ap, c->partial, c->scal);
    else
        hipLaunchKernelGGL(k_matvec_dot, mv.grid, mv.block, 0, s, L0, c->cg_p, c->cg_Ap, c->partial, c->scal);
    prof_end(c, IBMDEM_K_MATVEC, 2.0 * 8.0 * (double)n);
    CHECK_LAUNCH(c);
    hipLaunchKernelGGL(k_final, dim3(1), dim3(FIN_T), 0, s, c->partial, mv_blocks, c->scal, SC_PAP, 1, it,
                       c->cs.poisson_rtol);
    CHECK_LAUNCH(c);
    prof_begin(c, IBMDEM_K_CG_UPDATE);
    hipLaunchKernelGGL(k_cg_update_r, dim3(RED_BLOCKS), dim3(RED_T), 0, s, n, c->cg_r, c->cg_Ap, c->scal,
                       c->partial, c->cs.precision == IBMDEM_MIXED ? c->lev32[0].b : (float *)nullptr);
    prof_end(c, IBMDEM_K_CG_UPDATE, 3.0 * 8.0 * (double)n);
    CHECK_LAUNCH(c);
    hipLaunchKernelGGL(k_final, dim3(1), dim3(FIN_T), 0, s, c->partial, RED_BLOCKS, c->scal, SC_RR, 3, it,
                       c->cs.poisson_rtol);
    CHECK_LAUNCH(c);
    return precondition_dot(c, SC_RZ_NEW, 2);
}

}  // namespace

// Start of the solve, queued without any host wait, in two parts: first
// the pinned-row right-hand side, r = b, x = 0, ||b|| and the tolerance (a
// zero right-hand side converges at once); then z = M^-1 r, p = z, r.z
// (which a batch runs for all its cases at once).
int poisson_begin_rhs(ibmdem_ctx *c) {
    const long n = c->n;
    hipStream_t s = c->stream;
    int rc;
    // pinned row: b[0] = -sum_{q>0} b[q] (none with an outflow side)
    if (!c->lev64[0].d.dirichlet && (rc = reduce_sum(c, c->rhs, nullptr, n, SC_PIN, 1))) return rc;
    const LevelDev &L0 = c->lev64[0].d;
    const LaunchShape fs = shape_for(div_up(L0.nx, 2), L0.ny, L0.nz);
    hipLaunchKernelGGL(k_cg_init, fs.grid, fs.block, 0, s, L0, c->rhs, c->cg_r, c->cg_x, c->scal,
                       c->cs.precision == IBMDEM_MIXED ? c->lev32[0].b : (float *)nullptr);
    CHECK_LAUNCH(c);
    return dot_into(c, c->cg_r, c->cg_r, SC_BNORM2, 4);
}

int poisson_begin_precondition(ibmdem_ctx *c) {
    int rc;
    if ((rc = precondition_dot(c, SC_RZ, 0))) return rc;
    if (c->cs.precision == IBMDEM_MIXED)
        hipLaunchKernelGGL(k_copy<float>, dim3(stream_blocks(c->n)), dim3(RED_T), 0, c->stream, c->n, c->cg_p,
                           c->lev32[0].x);
    else
        hipLaunchKernelGGL(k_copy<double>, dim3(stream_blocks(c->n)), dim3(RED_T), 0, c->stream, c->n, c->cg_p,
                           c->cg_z);
    CHECK_LAUNCH(c);
    return IBMDEM_OK;
}

int poisson_begin(ibmdem_ctx *c) {
    int rc;
    if ((rc = poisson_begin_rhs(c))) return rc;
    return poisson_begin_precondition(c);
}

// Iterations first..last, queued without any host wait. Once the device sets
// SC_CONV every later CG kernel returns at once, so x is the iterate of the
// converging iteration however many iterations were queued.
int poisson_iterations(ibmdem_ctx *c, int first, int last) {
    for (int it = first; it <= last; ++it) {
        int rc = cg_iteration(c, it);
        if (rc) return rc;
    }
    return IBMDEM_OK;
}

// Iterations from `first` until convergence or the cap: the host keeps at
// most two iterations in flight and reads the convergence flag of the older
// one, so the stream never drains inside the solve.
int poisson_iterate_to_convergence(ibmdem_ctx *c, int first) {
    hipStream_t s = c->stream;
    const int maxit = c->cs.poisson_max_iter;
    for (int q = 0; q <= maxit + 1; ++q) c->conv_host[q] = 0.0;
    HIPX(c, hipMemcpyAsync(c->conv_host + first - 1, c->scal + SC_CONV, sizeof(double), hipMemcpyDeviceToHost, s));
    HIPX(c, hipEventRecord(c->iter_ev[(first - 1) & 1], s));
    for (int it = first; it <= maxit; ++it) {
        int rc = cg_iteration(c, it);
        if (rc) return rc;
        HIPX(c, hipMemcpyAsync(c->conv_host + it, c->scal + SC_CONV, sizeof(double), hipMemcpyDeviceToHost, s));
        HIPX(c, hipEventRecord(c->iter_ev[it & 1], s));
        // wait for the previous iteration, then look at its flag
        HIPX(c, hipEventSynchronize(c->iter_ev[(it - 1) & 1]));
        if (c->conv_host[it - 1] != 0.0) break;
    }
    return IBMDEM_OK;
}

// Wait for the solve, report it, fail on a non-converged or non-finite one.
int poisson_check(ibmdem_ctx *c, ibmdem_solve_info *info) {
    int rc;
    if ((rc = read_scalars(c))) return rc;
    return poisson_check_scalars(c, nullptr, info);
}

// The same report from solver scalars already on the host (scal, or the
// context's own copy when null).
int poisson_check_scalars(ibmdem_ctx *c, const double *scal, ibmdem_solve_info *info) {
    if (scal) std::memcpy(c->scal_host, scal, SC_COUNT * sizeof(double));
    const double bnorm = std::sqrt(c->scal_host[SC_BNORM2]);
    const int conv = c->scal_host[SC_CONV] != 0.0;
    const double rr = bnorm > 0 ? c->scal_host[SC_RR] : 0.0;
    const int it = conv ? (int)c->scal_host[SC_ITER] : c->cs.poisson_max_iter;
    c->last_cg_iterations = it;
    if (info) {
        info->iterations = it;
        info->converged = conv;
        info->rel_residual = bnorm > 0 ? std::sqrt(rr) / bnorm : 0.0;
        info->rhs_norm = bnorm;
    }
    // a non-finite right-hand side (||b|| is then NaN or inf) or residual
    if (!(bnorm - bnorm == 0.0) || !(rr == rr))
        return set_error(c, IBMDEM_ERR_NAN, "non-finite right-hand side or residual in the Poisson solve");
    if (!conv) return set_error(c, IBMDEM_ERR_NOT_CONVERGED, "Poisson solve did not converge");
    return IBMDEM_OK;
}

// P' = x - x(1,1,1): the reference's gauge (poisson.F90:78,97-100)
int poisson_gauge(ibmdem_ctx *c) {
    const LevelDev &L0 = c->lev64[0].d;
    const LaunchShape fs = shape_for(div_up(L0.nx, 2), L0.ny, L0.nz);
    hipLaunchKernelGGL(k_gauge, fs.grid, fs.block, 0, c->stream, L0, c->cg_x, c->cg_p, c->scal, c->pcorr);
    CHECK_LAUNCH(c);
    return IBMDEM_OK;
}

int poisson_solve(ibmdem_ctx *c, ibmdem_solve_info *info) {
    int rc;
    if ((rc = poisson_begin(c))) return rc;
    if ((rc = poisson_iterate_to_convergence(c, 1))) return rc;
    // an unconverged solve still delivers its last iterate, as the oracle does
    const int chk = poisson_check(c, info);
    if (chk && chk != IBMDEM_ERR_NOT_CONVERGED) return chk;
    if ((rc = poisson_gauge(c))) return rc;
    return chk;
}

// ---------------------------------------------------------------------------
// The batched solve: one launch per solver operation over a group of cases.
//
// A group's cases share the precision, the smoothing counts and the
// iteration cap; grids, level counts, where the one-work-group tail starts
// and the coarsest-level sweeps are per case. A launch runs the body of the
// members' own launches, and a member sees its operations in the order its own
// solve queues them. Where a sum's association follows the decomposition (the
// inner products, the last pass with r.z) that is the member's own; the level
// passes, whose cells do not depend on it, choose tiles or marching and the
// chunk length by the whole launch. So a member's arithmetic is bitwise that
// of solving it alone. A
// block finds its case in a table of first blocks (each a multiple of 8, so
// a case's blocks keep the XCD placement of its own launch); a member that
// has converged returns at once, as it does alone.
// ---------------------------------------------------------------------------
namespace {

template <typename T>
struct MaArg {
    BGrid g;
    const LevelDev *L;
    const T *xin, *b;
    T *out, *out2;
    double *partial;
    int nzp;   // planes of a chunk
    int nty;   // the grid's y holds the rows' tiles chunk after chunk, so that
               // batch_for deals the blocks evenly (by planes, a chunk more or less an XCD)
    const T *xc;
    const double *stop;
};
template <typename T, int PW, int MODE, bool FROMB, bool PRO>
__global__ __launch_bounds__(MT, (MARCH_WAVES<T, MODE>)) void kb_march(BTable<MaArg<T>> tab) {
    batch_for(tab, [&](const MaArg<T> &a, const Blk &kt) {
        Blk kb = kt;
        kb.bz = kt.by / a.nty;
        kb.by = kt.by - kb.bz * a.nty;
        march_body<T, PW, MODE, FROMB, PRO>(kb, *cst(a.L), glb(a.xin), glb(a.b), glb(a.out), glb(a.out2),
                                            glb(a.partial), a.nzp, glb(a.xc), glb(a.stop));
    });
}

struct RzArg {
    BGrid g;
    const LevelDev *L;
    const float *oth;
    float *own;
    const double *r64;
    double *partial;
    long pofs;
    const double *stop;
};
template <int PW>
__global__ __launch_bounds__(RB) void kb_rz_half(BTable<RzArg> tab, int color) {
    batch_for(tab, [&](const RzArg &a, const Blk &kb) {
        rz_half_body<PW>(kb, *cst(a.L), glb(a.oth), glb(a.own), color, glb(a.r64), glb(a.partial), a.pofs,
                         glb(a.stop));
    });
}

// a launch of a level in tiles (k_tile_down's and k_tile_up's arguments)
template <typename T>
struct TlArg {
    BGrid g;
    const LevelDev *L, *C;
    const T *b, *xin;
    T *x, *xb;
    bool more;   // k_tile_down's more, k_tile_up's two
    T *bc;
    const T *xc;
    double *partial;
    const double *stop;
};
template <typename T, int SRC>
__global__ __launch_bounds__(TileDown::NT) void kb_tile_down(BTable<TlArg<T>> tab) {
    batch_for(tab, [&](const TlArg<T> &a, const Blk &kb) {
        tile_down_body<T, SRC>(kb, *cst(a.L), glb(a.b), glb(a.xin), a.more, glb(a.x), *cst(a.C), glb(a.bc),
                               glb(a.stop));
    });
}
template <typename T, int SRC>
__global__ __launch_bounds__(TileUp::NT) void kb_tile_up(BTable<TlArg<T>> tab) {
    batch_for(tab, [&](const TlArg<T> &a, const Blk &kb) {
        tile_up_body<T, SRC>(kb, *cst(a.L), glb(a.b), glb(a.xin), glb(a.x), a.xb ? glb(a.xb) : (T *)nullptr, a.more,
                             *cst(a.C), glb(a.xc), a.partial ? glb(a.partial) : (double *)nullptr, glb(a.stop));
    });
}
template <typename T>
__global__ __launch_bounds__(TRZ_NT) void kb_tile_rz(BTable<TlArg<T>> tab) {
    batch_for(tab, [&](const TlArg<T> &a, const Blk &kb) {
        tile_rz_body<T>(kb, *cst(a.L), glb(a.b), glb(a.xin), glb(a.partial), glb(a.stop));
    });
}

template <typename T>
struct RsArg {
    BGrid g;
    const LevelDev *F, *C;
    const T *rf;
    T *bc;
    const double *stop;
};
template <typename T>
__global__ __launch_bounds__(RB) void kb_restrict(BTable<RsArg<T>> tab) {
    batch_for(tab, [&](const RsArg<T> &a, const Blk &kb) {
        restrict_body<T>(kb, *cst(a.F), glb(a.rf), *cst(a.C), glb(a.bc), glb(a.stop));
    });
}

template <typename T>
struct PrArg {
    BGrid g;
    const LevelDev *F, *C;
    const T *xin;
    T *xout;
    const T *xc;
    const double *stop;
};
template <typename T, int PW>
__global__ __launch_bounds__(RB) void kb_prolong(BTable<PrArg<T>> tab) {
    batch_for(tab, [&](const PrArg<T> &a, const Blk &kb) {
        prolong_red_body<T, PW>(kb, *cst(a.F), glb(a.xin), glb(a.xout), *cst(a.C), glb(a.xc), glb(a.stop));
    });
}

// the bottom of a case's V-cycle: the one-work-group tail (first < last),
// or the coarsest level alone from LDS tables or in global memory
template <typename T>
struct BtArg {
    BGrid g;
    const LevelDev *lev;
    int first, last, pre, post, sweeps;
    int s0, ns;   // the tile form's half sweeps
    bool all_out;
    T *x;
    const T *b;
    T *tmp;
    const double *stop;
};
template <typename T>
__global__ __launch_bounds__(TAIL_T) void kb_tail(BTable<BtArg<T>> tab) {
    batch_for(tab, [&](const BtArg<T> &a, const Blk &kb) {
        vcycle_tail_body<T>(kb, cst(a.lev), a.first, a.last, glb(a.b), glb(a.x), a.pre, a.post, a.sweeps,
                            glb(a.stop));
    });
}
template <typename T, int NT, int CP>
__global__ __launch_bounds__(NT) void kb_coarse_jac(BTable<BtArg<T>> tab) {
    batch_for(tab, [&](const BtArg<T> &a, const Blk &kb) {
        coarse_jac_body<T, NT, CP>(kb, *cst(a.lev + a.last), glb(a.x), glb(a.b), a.sweeps, glb(a.stop));
    });
}
template <typename T, int NT, int CP>
__global__ __launch_bounds__(NT) void kb_coarse_wg(BTable<BtArg<T>> tab) {
    batch_for(tab, [&](const BtArg<T> &a, const Blk &kb) {
        coarse_wg_body<T, NT, CP>(kb, *cst(a.lev + a.last), glb(a.x), glb(a.b), a.sweeps, glb(a.stop));
    });
}
// one launch of the tile form: half sweeps s0 .. s0 + ns - 1 from tmp to x
template <typename T, bool JAC>
__global__ __launch_bounds__(CT_T) void kb_coarse_tile(BTable<BtArg<T>> tab) {
    batch_for(tab, [&](const BtArg<T> &a, const Blk &kb) {
        coarse_tile_body<T, JAC>(kb, *cst(a.lev + a.last), glb(a.tmp), glb(a.x), glb(a.b), a.s0, a.ns, a.all_out,
                                 glb(a.stop));
    });
}

// the CG vector operations and the scalar step
struct CgArg {
    BGrid g;
    const LevelDev *L;
    long n;
    double *p, *x, *r, *Ap;
    const void *z;   // FP32 in the mixed form
    double *partial;
    double *scal;
    float *r32;
    int np;           // partial sums k_final adds
    double rtol;
    const double *rhs;   // the solve's right-hand side (field order)
};
__global__ __launch_bounds__(RB) void kb_matvec_dot(BTable<CgArg> tab) {
    batch_for(tab, [&](const CgArg &a, const Blk &kb) {
        matvec_dot_body(kb, *cst(a.L), glb(a.p), glb(a.Ap), glb(a.partial), glb(a.scal));
    });
}
__global__ __launch_bounds__(RB) void kb_matvec2_dot(BTable<CgArg> tab) {
    batch_for(tab, [&](const CgArg &a, const Blk &kb) {
        matvec2_dot_body(kb, *cst(a.L), glb(a.p), glb(a.Ap), glb(a.partial), glb(a.scal));
    });
}
template <typename T>
__global__ __launch_bounds__(RED_T) void kb_cg_px(BTable<CgArg> tab) {
    batch_for(tab, [&](const CgArg &a, const Blk &kb) {
        cg_px_body(kb, a.n, glb(a.p), glb((const T *)a.z), glb(a.x), glb(a.scal));
    });
}
__global__ __launch_bounds__(RED_T) void kb_cg_update_r(BTable<CgArg> tab) {
    batch_for(tab, [&](const CgArg &a, const Blk &kb) {
        cg_update_r_body(kb, a.n, glb(a.r), glb(a.Ap), glb(a.scal), glb(a.partial), glb(a.r32));
    });
}
template <typename T>
__global__ __launch_bounds__(RED_T) void kb_copy(BTable<CgArg> tab) {
    batch_for(tab, [&](const CgArg &a, const Blk &kb) { copy_body(kb, a.n, glb(a.p), glb((const T *)a.z)); });
}
__global__ __launch_bounds__(FIN_T) void kb_final(BTable<CgArg> tab, int slot, int op, int it) {
    batch_for(tab, [&](const CgArg &a, const Blk &kb) {
        final_body(kb, glb(a.partial), a.np, glb(a.scal), slot, op, it, a.rtol);
    });
}

// every case's solver scalars into one array (case q at q * SC_COUNT)
__global__ __launch_bounds__(64) void kb_gather_scalars(const double *const *__restrict__ scal, int ncase,
                                                        double *__restrict__ out) {
    const int q = blockIdx.x;
    if (q < ncase && threadIdx.x < SC_COUNT) out[(long)q * SC_COUNT + threadIdx.x] = glb(scal[q])[threadIdx.x];
}

// Profiling of the batched solve: while armed, run_ops records an event
// before the first launch and after every launch, so the elapsed time
// between two events is one launch's run time once the stream runs behind
// the host (the launches are queued far faster than they run).
constexpr int BK_COUNT = 9;
struct BProf {
    bool on = false, armed = false;
    std::vector<hipEvent_t> ev;
    std::vector<int> kind;
    std::vector<double> bytes;
    int n = 0;                          // launches recorded
};
template <typename T, int PW, int MODE, bool FROMB, bool PRO = false>
void launch_ma(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL((kb_march<T, PW, MODE, FROMB, PRO>), dim3(o.blocks), dim3(MT), 0, s, table<MaArg<T>>(o));
}
template <int PW>
void launch_rzb(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_rz_half<PW>, dim3(o.blocks), dim3(RB), 0, s, table<RzArg>(o), o.color);
}
template <typename T, int SRC>
void launch_down(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL((kb_tile_down<T, SRC>), dim3(o.blocks), dim3(TileDown::NT), 0, s, table<TlArg<T>>(o));
}
template <typename T>
void launch_tile_rz(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_tile_rz<T>, dim3(o.blocks), dim3(TRZ_NT), 0, s, table<TlArg<T>>(o));
}
template <typename T, int SRC>
void launch_up(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL((kb_tile_up<T, SRC>), dim3(o.blocks), dim3(TileUp::NT), 0, s, table<TlArg<T>>(o));
}
template <typename T>
void launch_restrict(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_restrict<T>, dim3(o.blocks), dim3(RB), 0, s, table<RsArg<T>>(o));
}
template <typename T, int PW>
void launch_prolong(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL((kb_prolong<T, PW>), dim3(o.blocks), dim3(RB), 0, s, table<PrArg<T>>(o));
}
template <typename T>
void launch_tail(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_tail<T>, dim3(o.blocks), dim3(TAIL_T), 0, s, table<BtArg<T>>(o));
}
template <typename T, int NT, int CP>
void launch_coarse_jac(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL((kb_coarse_jac<T, NT, CP>), dim3(o.blocks), dim3(NT), 0, s, table<BtArg<T>>(o));
}
template <typename T, int NT, int CP>
void launch_coarse_wg(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL((kb_coarse_wg<T, NT, CP>), dim3(o.blocks), dim3(NT), 0, s, table<BtArg<T>>(o));
}
template <typename T, bool JAC>
void launch_coarse_tile(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL((kb_coarse_tile<T, JAC>), dim3(o.blocks), dim3(CT_T), 0, s, table<BtArg<T>>(o));
}
void launch_matvec(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_matvec_dot, dim3(o.blocks), dim3(RB), 0, s, table<CgArg>(o));
}
void launch_matvec2(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_matvec2_dot, dim3(o.blocks), dim3(RB), 0, s, table<CgArg>(o));
}
template <typename T>
void launch_px(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_cg_px<T>, dim3(o.blocks), dim3(RED_T), 0, s, table<CgArg>(o));
}
void launch_update_r(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_cg_update_r, dim3(o.blocks), dim3(RED_T), 0, s, table<CgArg>(o));
}
template <typename T>
void launch_copy(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_copy<T>, dim3(o.blocks), dim3(RED_T), 0, s, table<CgArg>(o));
}
void launch_final(const BOp &o, hipStream_t s, int it) {
    hipLaunchKernelGGL(kb_final, dim3(o.blocks), dim3(FIN_T), 0, s, table<CgArg>(o), o.slot, o.op,
                       o.with_it ? it : 0);
}

template <typename T>
MGLevel<T> *levels(ibmdem_ctx *c);
template <>
MGLevel<double> *levels<double>(ibmdem_ctx *c) { return c->lev64; }
template <>
MGLevel<float> *levels<float>(ibmdem_ctx *c) { return c->lev32; }

// the level where a case's V-cycle turns: its tail's first level, else its coarsest
int bottom_level(const ibmdem_ctx *c) { return std::min(c->tail_first, c->nlev - 1); }

// z = M^-1 r for every case, with r.z into scal[slot] (k_final's op): the
// batched form of vcycle<T>(c, lev, 0, true) and precondition_dot
template <typename T>
int plan_precondition_dot(Arena &ar, std::vector<BOp> &ops, const std::vector<ibmdem_ctx *> &cs, int slot,
                          int op, std::string &err) {
    const bool mixed = !std::is_same<T, double>::value;
    const int pre = cs[0]->cs.mg_pre, post = cs[0]->cs.mg_post;
    int depth = 0;
    for (ibmdem_ctx *c : cs) depth = std::max(depth, bottom_level(c));
    int rc;
    // The cells that smooth on level l, over the cases. Tiles or passes (the
    // same values) are chosen by them, as for one level of that size: a batch
    // fills the chip, and the tiles' halo then costs time (40 uneven
    // cases of 96x80x64 cells on average in FP64: 104 ms a pass of four steps
    // and download with level 0 in tiles, 73 ms in passes). What the form
    // decides in a case's own run stays as it is there: the order of the r.z
    // sums (TlRz below) and whether the prolongation is part of a pass.
    auto cells_at = [&](int l) {
        double n = 0.0;
        for (ibmdem_ctx *c : cs)
            if (l < bottom_level(c)) n += (double)levels<T>(c)[l].n;
        return n;
    };
    auto tiled = [&](const ibmdem_ctx *c, int l) {
        return tile_level<T>(c, l) && cells_at(l) <= (double)tile_cells(pre, post);
    };
    // The pass of level l (vcycle's, MODE and FROMB by mode and fromb) of every
    // case whose V-cycle goes below l: one launch for the cases with two-pair
    // threads, one for the others. in and out: 0, 1 the halves of x, 2, 3 of r
    // (own_tile: 1 the cases whose own form is tiles alone, 0 the others alone)
    auto pass = [&](int l, int mode, bool fromb, int in, int to, int to2, int own_tile = -1, bool pro = false) {
        std::vector<MaArg<T>> args[2];
        std::vector<LevelDev> lev[2];
        BOp o[2];
        const double per = mode >= 2        ? 2.5 * sizeof(T)
                           : mode == 0 && fromb ? 1.5 * sizeof(T)
                           : mode == 1 && RES_BLACK<T> ? 2.5 * sizeof(T)
                                                       : 2.0 * sizeof(T);
        for (ibmdem_ctx *c : cs) {
            if (l >= bottom_level(c) || tiled(c, l)) continue;
            if (own_tile >= 0 && tile_level<T>(c, l) != (own_tile == 1)) continue;
            MGLevel<T> &L = levels<T>(c)[l];
            T *buf[4] = {L.x, L.x + L.d.half, L.r, L.r + L.d.half};
            const int pw = march_pw(L.d);
            const MarchShape sh = march_shape<T>(L.d, pw);
            MaArg<T> a{};
            a.g = bgrid(dim3(sh.ntx, sh.nty * sh.nzc), dim3(MT));
            a.nty = sh.nty;
            a.L = c->dlev + l;
            a.xin = in >= 0 ? buf[in] : nullptr;
            a.b = L.b;
            a.out = buf[to];
            a.out2 = to2 >= 0 ? buf[to2] : nullptr;
            a.partial = mode == 2 ? c->partial : nullptr;
            a.nzp = sh.nzp;
            a.xc = pro ? levels<T>(c)[l + 1].x : nullptr;
            a.stop = c->scal + SC_CONV;
            args[pw - 1].push_back(a);
            lev[pw - 1].push_back(L.d);
            if (l == 0) o[pw - 1].bytes += per * (double)c->n;
        }
        // chunks for the launch, except where the r.z sums follow the case's own
        for (int v = 0; v < (mode == 2 ? 0 : 2); ++v) {
            if (args[v].empty()) continue;
            const int planes = march_planes<T>(lev[v], v + 1, sizeof(T) == 4 && mode != 1 ? 2 : 1);
            for (size_t q = 0; q < args[v].size(); ++q) {
                MaArg<T> &a = args[v][q];
                const int nzc = div_up(lev[v][q].nz, planes);
                a.nzp = div_up(lev[v][q].nz, nzc);
                a.g = bgrid(dim3(a.g.gx, a.nty * nzc), dim3(MT));
            }
        }
        const BLaunch fp[2] = {launch_ma<double, 1, 0, false, true>, launch_ma<double, 2, 0, false, true>};
        const BLaunch fn[2][5] = {
            {launch_ma<T, 1, 0, false>, launch_ma<T, 1, 0, true>, launch_ma<T, 1, 1, false>, launch_ma<T, 1, 1, true>,
             mode == 2 ? launch_ma<double, 1, 2, false> : launch_ma<T, 1, 3, false>},
            {launch_ma<T, 2, 0, false>, launch_ma<T, 2, 0, true>, launch_ma<T, 2, 1, false>, launch_ma<T, 2, 1, true>,
             mode == 2 ? launch_ma<double, 2, 2, false> : launch_ma<T, 2, 3, false>}};
        for (int v = 1; v >= 0; --v) {
            o[v].kind = l == 0 ? IBMDEM_BK_SMOOTH0 : IBMDEM_BK_SMOOTH;
            const int r2 = add_op(ar, ops, pro ? fp[v] : fn[v][mode >= 2 ? 4 : 2 * mode + fromb], MT, args[v], o[v], err);
            if (r2) return r2;
        }
        return (int)IBMDEM_OK;
    };
    // launch_rz of every case (the mixed form's last sweeps at level 0), the
    // red cells' x in half `in` of r
    auto rz = [&](int in) {
        for (int q = 0; q < 2; ++q) {
            std::vector<RzArg> args[2];
            BOp o[2];
            for (ibmdem_ctx *c : cs) {
                MGLevel<float> &L = c->lev32[0];
                const SweepShape sw = sweep_shape(L.d);
                RzArg a{};
                a.g = bgrid(sw.grid, sw.block);
                a.L = c->dlev;
                a.oth = q ? L.x + L.d.half : L.r + (in - 2) * (long)L.d.half;
                a.own = L.x + (q ? 0 : L.d.half);
                a.r64 = c->cg_r;
                a.partial = c->partial;
                a.pofs = q * (long)sw.grid.x * sw.grid.y * sw.grid.z;
                a.stop = c->scal + SC_CONV;
                args[sw.x2].push_back(a);
                o[sw.x2].bytes += 8.0 * (double)c->n;
            }
            for (int v = 1; v >= 0; --v) {
                o[v].color = 1 - q;
                o[v].kind = IBMDEM_BK_SMOOTH0;
                const int r2 = add_op(ar, ops, v ? launch_rzb<2> : launch_rzb<1>, RB, args[v], o[v], err);
                if (r2) return r2;
            }
        }
        return (int)IBMDEM_OK;
    };
    // one launch in tiles on level l, of every case that takes them: in and
    // to as pass's, src and more the kernel's
    auto tile = [&](int l, bool up, TileSrc src, int in, int to, int to2, bool more, bool rzsum) {
        std::vector<TlArg<T>> args;
        BOp o;
        o.kind = l == 0 ? IBMDEM_BK_SMOOTH0 : IBMDEM_BK_SMOOTH;
        for (ibmdem_ctx *c : cs) {
            if (l >= bottom_level(c) || !tiled(c, l)) continue;
            MGLevel<T> &L = levels<T>(c)[l], &C = levels<T>(c)[l + 1];
            T *buf[4] = {L.x, L.x + L.d.half, L.r, L.r + L.d.half};
            TlArg<T> a{};
            a.g = bgrid(tile_grid(L.d), dim3(256, (up ? TileUp::NT : TileDown::NT) / 256));
            a.L = c->dlev + l;
            a.C = c->dlev + l + 1;
            a.b = L.b;
            a.xin = in >= 0 ? buf[in] : nullptr;
            a.x = buf[to];
            a.xb = to2 >= 0 ? buf[to2] : nullptr;
            a.more = more;
            a.bc = C.b;
            a.xc = C.x;
            a.partial = rzsum ? c->partial : nullptr;
            a.stop = c->scal + SC_CONV;
            args.push_back(a);
            if (l == 0) o.bytes += (src == TS_B ? 1.5 : to2 >= 0 ? 2.5 : 2.0) * sizeof(T) * (double)c->n;
        }
        const BLaunch fu[3] = {launch_up<T, TS_B>, launch_up<T, TS_X>, launch_up<T, TS_PROLONG>};
        const BLaunch fd[2] = {launch_down<T, TS_B>, launch_down<T, TS_X>};
        return add_op(ar, ops, up ? fu[src] : fd[src], up ? TileUp::NT : TileDown::NT, args, o, err);
    };
    // the halves of a visit in tiles, as vcycle's
    auto tile_down = [&](int l) {
        const int ns = tile_smooths(pre);
        int in = -1, r2;
        for (int q = 0; q < ns; ++q) {
            const int to = q & 1;
            if ((r2 = tile(l, true, q ? TS_X : TS_B, in, to, -1, tile_smooth_two(pre, q), false))) return r2;
            in = to;
        }
        return tile(l, false, ns ? TS_X : TS_B, in, 2, -1, pre > 1, false);
    };
    auto tile_up = [&](int l) {
        const int nu = tile_ups(post);
        for (int q = 0; q < nu; ++q) {
            const bool last = q == nu - 1;
            const int from = 2 + (q & 1);
            const int r2 = tile(l, true, q ? TS_X : TS_PROLONG, from, last ? 0 : 5 - from, last ? 1 : -1,
                                tile_up_two(post, q), l == 0 && last);
            if (r2) return r2;
        }
        return (int)IBMDEM_OK;
    };
    // r.z of the cases whose own level-0 form is tiles, after passes
    auto tile_rz = [&]() {
        std::vector<TlArg<T>> args;
        BOp o;
        o.kind = IBMDEM_BK_SMOOTH0;
        for (ibmdem_ctx *c : cs) {
            if (tiled(c, 0) || !tile_level<T>(c, 0)) continue;
            MGLevel<T> &L = levels<T>(c)[0];
            TlArg<T> a{};
            a.g = bgrid(tile_grid(L.d), dim3(128, TRZ_NT / 128));
            a.L = c->dlev;
            a.b = L.b;
            a.xin = L.x;
            a.partial = c->partial;
            a.stop = c->scal + SC_CONV;
            args.push_back(a);
            o.bytes += 2.0 * sizeof(T) * (double)c->n;
        }
        return add_op(ar, ops, launch_tile_rz<T>, TRZ_NT, args, o, err);
    };
    // the bottoms at level l
    auto bottoms = [&](int l) {
        // by form (coarse_form; the tails in the last list), and the tile
        // form's launches, each over the cases that still have one to do
        std::vector<BtArg<T>> by[CF_TILE + 1];
        std::vector<std::vector<BtArg<T>>> tiles[2];
        for (ibmdem_ctx *c : cs) {
            if (bottom_level(c) != l) continue;
            MGLevel<T> &L = levels<T>(c)[l];
            BtArg<T> a{};
            a.lev = c->dlev;
            a.first = l;
            a.last = c->nlev - 1;
            a.pre = c->cs.mg_pre;
            a.post = c->cs.mg_post;
            a.sweeps = c->cs.mg_coarse_sweeps;
            a.x = L.x;
            a.b = L.b;
            a.tmp = L.r;
            a.stop = c->scal + SC_CONV;
            if (l >= c->tail_first) {
                a.g = bgrid(dim3(1), dim3(TAIL_T));
                by[CF_TILE].push_back(a);
                continue;
            }
            const CoarseForm f = coarse_form(L.d);
            if (f < CF_TILE) {
                a.g = bgrid(dim3(1), dim3(coarse_threads(f)));
                by[f].push_back(a);
                continue;
            }
            const bool jac = f == CF_TILE_JAC;
            const int n = coarse_tile_launches(jac, a.sweeps);
            if ((int)tiles[jac].size() < n) tiles[jac].resize(n);
            a.g = bgrid(coarse_tile_grid(L.d), dim3(256, CT_T / 256));
            for (int q = 0; q < n; ++q) {
                const CoarseTileStep st = coarse_tile_step(jac, a.sweeps, q);
                a.s0 = st.s0;
                a.ns = st.ns;
                a.all_out = st.all_out;
                a.x = st.to_x ? L.x : L.r;
                a.tmp = st.to_x ? L.r : L.x;
                tiles[jac][q].push_back(a);
            }
        }
        int r;
        BOp o;
        o.kind = IBMDEM_BK_BOTTOM;
        const BLaunch fn[CF_TILE + 1] = {launch_coarse_wg<T, 256, 2>,   launch_coarse_wg<T, 1024, 1>,
                                         launch_coarse_wg<T, 1024, 2>,  launch_coarse_wg<T, 1024, 4>,
                                         launch_coarse_wg<T, 1024, 8>,  launch_coarse_jac<T, 512, 1>,
                                         launch_coarse_jac<T, 1024, 2>, launch_coarse_jac<T, 1024, 8>,
                                         launch_tail<T>};
        for (int f = 0; f <= CF_TILE; ++f)
            if ((r = add_op(ar, ops, fn[f], f == CF_TILE ? TAIL_T : coarse_threads((CoarseForm)f), by[f], o, err)))
                return r;
        for (int jac = 0; jac < 2; ++jac)
            for (const std::vector<BtArg<T>> &args : tiles[jac])
                if ((r = add_op(ar, ops, jac ? launch_coarse_tile<T, true> : launch_coarse_tile<T, false>, CT_T, args,
                                o, err)))
                    return r;
        return IBMDEM_OK;
    };
    int last_in = 0;   // the half of x the pre-smoothing leaves the red cells in
    for (int l = 0; l < depth; ++l) {
        int cur = -1;
        for (int q = 0; q < pre; ++q) {
            const int to = cur == 0 ? 1 : 0;
            if (q == pre - 1) {
                if ((rc = pass(l, 1, q == 0, cur, 2, q == 0 ? 0 : -1))) return rc;
                if (q == 0) cur = 0;
            } else {
                if ((rc = pass(l, 0, q == 0, cur, to, -1))) return rc;
                cur = to;
            }
        }
        last_in = cur;
        if ((rc = tile_down(l))) return rc;
        std::vector<RsArg<T>> rs;
        BOp ors;
        ors.kind = IBMDEM_BK_RESTRICT;
        for (ibmdem_ctx *c : cs) {
            if (l >= bottom_level(c) || tiled(c, l)) continue;
            MGLevel<T> &F = levels<T>(c)[l], &C = levels<T>(c)[l + 1];
            RsArg<T> a{};
            a.g = bgrid(dim3(div_up(C.d.nx, RS_CX), div_up(C.d.ny, RS_CY), C.d.nz), dim3(RB));
            a.F = c->dlev + l;
            a.C = c->dlev + l + 1;
            a.rf = F.r;
            a.bc = C.b;
            a.stop = c->scal + SC_CONV;
            rs.push_back(a);
            // the residual read (in FP64 its red half), the coarse right-hand
            // side written
            ors.bytes += sizeof(T) * ((RES_BLACK<T> ? 1.0 : 0.5) * (double)F.n + (double)C.n);
        }
        if ((rc = add_op(ar, ops, launch_restrict<T>, RB, rs, ors, err))) return rc;
        if ((rc = bottoms(l + 1))) return rc;
    }
    const bool fused = prolong_fused<T>(post);
    for (int l = depth - 1; l >= 0; --l) {
        std::vector<PrArg<T>> pr[2];
        BOp opr[2];
        for (ibmdem_ctx *c : cs) {
            if (l >= bottom_level(c) || tiled(c, l) || (fused && !tile_level<T>(c, l))) continue;
            MGLevel<T> &F = levels<T>(c)[l], &C = levels<T>(c)[l + 1];
            const int pw = march_pw(F.d);
            const LaunchShape sh = shape_for(F.d.nx / 2 / pw, F.d.ny, F.d.nz);
            PrArg<T> a{};
            a.g = bgrid(sh.grid, sh.block);
            a.F = c->dlev + l;
            a.C = c->dlev + l + 1;
            a.xin = F.x + last_in * (long)F.d.half;
            a.xout = F.r;
            a.xc = C.x;
            a.stop = c->scal + SC_CONV;
            pr[pw - 1].push_back(a);
            // the coarse solution and the red cells read, the latter written
            opr[pw - 1].bytes += sizeof(T) * (double)(F.n + C.n);
        }
        opr[0].kind = opr[1].kind = IBMDEM_BK_PROLONG;
        if ((rc = add_op(ar, ops, launch_prolong<T, 2>, RB, pr[1], opr[1], err))) return rc;
        if ((rc = add_op(ar, ops, launch_prolong<T, 1>, RB, pr[0], opr[0], err))) return rc;
        if ((rc = tile_up(l))) return rc;
        int cur = 2;
        for (int q = 0; q < post; ++q) {
            const bool last = q == post - 1;
            const int to = cur == 2 ? 3 : 2;
            if (last && l == 0 && mixed) {
                if ((rc = rz(cur))) return rc;
                break;
            }
            if (!last) {
                const bool pro = q == 0 && fused;
                if (pro && (rc = pass(l, 0, false, last_in, to, -1, 0, true))) return rc;
                if ((rc = pass(l, 0, false, cur, to, -1, pro ? 1 : -1))) return rc;
            } else if (l == 0) {
                if ((rc = pass(l, 2, false, cur, 0, 1, 0))) return rc;
                if ((rc = pass(l, 3, false, cur, 0, 1, 1))) return rc;
                if ((rc = tile_rz())) return rc;
            } else if ((rc = pass(l, 3, false, cur, 0, 1))) {
                return rc;
            }
            cur = to;
        }
    }
    std::vector<CgArg> fin;
    for (ibmdem_ctx *c : cs) {
        CgArg a{};
        a.g = bgrid(dim3(1), dim3(FIN_T));
        a.partial = c->partial;
        a.scal = c->scal;
        a.np = rz_blocks(c);
        a.rtol = c->cs.poisson_rtol;
        fin.push_back(a);
    }
    BOp o;
    o.slot = slot;
    o.op = op;
    o.kind = IBMDEM_BK_SCALAR;
    return add_op(ar, ops, launch_final, FIN_T, fin, o, err);
}

// the CG vectors of every case (the mixed form's FP32 copy of r with them)
CgArg cg_arg(ibmdem_ctx *c, dim3 grid, dim3 block, int np) {
    CgArg a{};
    a.g = bgrid(grid, block);
    a.L = c->dlev;
    a.n = c->n;
    a.z = c->cs.precision == IBMDEM_MIXED ? (const void *)c->lev32[0].x : c->cg_z;
    a.p = c->cg_p; a.x = c->cg_x; a.r = c->cg_r; a.Ap = c->cg_Ap;
    a.partial = c->partial;
    a.scal = c->scal;
    a.r32 = c->cs.precision == IBMDEM_MIXED ? c->lev32[0].b : nullptr;
    a.np = np;
    a.rtol = c->cs.poisson_rtol;
    return a;
}

template <typename T>
int plan_all(Arena &ar, std::vector<BOp> &begin, std::vector<BOp> &iter, const std::vector<ibmdem_ctx *> &cs,
             std::string &err) {
    int rc;
    // poisson_begin_precondition: z = M^-1 r with r.z, p = z
    if ((rc = plan_precondition_dot<T>(ar, begin, cs, SC_RZ, 0, err))) return rc;
    std::vector<CgArg> cp, px, mv[2], fpap, up, frr;
    double mv_cells[2] = {0.0, 0.0};
    for (ibmdem_ctx *c : cs) {
        const SweepShape sh = sweep_shape(c->lev64[0].d);
        const int mvb = (int)(sh.grid.x * sh.grid.y * sh.grid.z);
        cp.push_back(cg_arg(c, dim3(stream_blocks(c->n)), dim3(RED_T), 0));
        px.push_back(cg_arg(c, dim3(stream_blocks(c->n)), dim3(RED_T), 0));
        mv[sh.x2].push_back(cg_arg(c, sh.grid, sh.block, 0));
        mv_cells[sh.x2] += (double)c->n;
        fpap.push_back(cg_arg(c, dim3(1), dim3(FIN_T), mvb));
        up.push_back(cg_arg(c, dim3(RED_BLOCKS), dim3(RED_T), 0));
        frr.push_back(cg_arg(c, dim3(1), dim3(FIN_T), RED_BLOCKS));
    }
    double cells = 0.0;
    for (ibmdem_ctx *c : cs) cells += (double)c->n;
    const bool mixed = !std::is_same<T, double>::value;
    BOp o;
    o.kind = IBMDEM_BK_VECTOR;
    o.bytes = (8.0 + sizeof(T)) * cells;   // z read, p written
    if ((rc = add_op(ar, begin, launch_copy<T>, RED_T, cp, o, err))) return rc;
    // cg_iteration
    o.skip_first = true;
    o.bytes = (32.0 + sizeof(T)) * cells;   // p, x read and written, z read
    if ((rc = add_op(ar, iter, launch_px<T>, RED_T, px, o, err))) return rc;
    o = BOp();
    o.kind = IBMDEM_BK_MATVEC;
    o.bytes = 16.0 * mv_cells[1];   // p read, Ap written
    if ((rc = add_op(ar, iter, launch_matvec2, RB, mv[1], o, err))) return rc;
    o.bytes = 16.0 * mv_cells[0];
    if ((rc = add_op(ar, iter, launch_matvec, RB, mv[0], o, err))) return rc;
    o = BOp();
    o.kind = IBMDEM_BK_SCALAR;
    o.slot = SC_PAP; o.op = 1; o.with_it = true;
    if ((rc = add_op(ar, iter, launch_final, FIN_T, fpap, o, err))) return rc;
    BOp ou;
    ou.kind = IBMDEM_BK_VECTOR;
    ou.bytes = (24.0 + (mixed ? 4.0 : 0.0)) * cells;   // r read and written, Ap read (FP32 r written)
    if ((rc = add_op(ar, iter, launch_update_r, RED_T, up, ou, err))) return rc;
    o.slot = SC_RR; o.op = 3;
    if ((rc = add_op(ar, iter, launch_final, FIN_T, frr, o, err))) return rc;
    return plan_precondition_dot<T>(ar, iter, cs, SC_RZ_NEW, 2, err);
}

int prof_event(BProf &pr, int i, hipStream_t s, std::string &err) {
    while ((int)pr.ev.size() <= i) {
        hipEvent_t e = nullptr;
        if (hipEventCreate(&e) != hipSuccess) {
            err = "profiling event creation failed";
            return IBMDEM_ERR_HIP;
        }
        pr.ev.push_back(e);
    }
    if (hipEventRecord(pr.ev[i], s) != hipSuccess) {
        err = "profiling event record failed";
        return IBMDEM_ERR_HIP;
    }
    return IBMDEM_OK;
}

int run_ops(const std::vector<BOp> &ops, hipStream_t s, int it, BProf &pr, std::string &err) {
    const bool rec = pr.on && pr.armed;
    int rc;
    if (rec && pr.n == 0 && (rc = prof_event(pr, 0, s, err))) return rc;
    for (const BOp &o : ops) {
        if (o.skip_first && it == 1) continue;
        o.fn(o, s, it);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            err = std::string("batched solver launch: ") + hipGetErrorString(e);
            return IBMDEM_ERR_HIP;
        }
        if (rec) {
            if ((rc = prof_event(pr, pr.n + 1, s, err))) return rc;
            pr.kind.resize(pr.n + 1);
            pr.bytes.resize(pr.n + 1);
            pr.kind[pr.n] = o.kind;
            pr.bytes[pr.n] = o.bytes;
            pr.n++;
        }
    }
    return IBMDEM_OK;
}

}  // namespace

struct PoissonBatch {
    std::vector<ibmdem_ctx *> cs;
    std::vector<BOp> begin, iter;
    BProf prof;
    char *arena = nullptr;             // device copy of the tables
    const double **scal_ptrs = nullptr;   // in the arena
    double *gather_dev = nullptr;
    double *gather_host = nullptr;     // pinned
};

bool poisson_batchable(const ibmdem_ctx *c) {
    // the V-cycle must leave r.z with its last sweeps (precondition_dot)
    return c->nlev >= 2 && c->cs.mg_post >= 1;
}

void poisson_batch_destroy(PoissonBatch *pb) {
    if (!pb) return;
    for (hipEvent_t e : pb->prof.ev) (void)hipEventDestroy(e);
    if (pb->arena) (void)hipFree(pb->arena);
    if (pb->gather_dev) (void)hipFree(pb->gather_dev);
    if (pb->gather_host) (void)hipHostFree(pb->gather_host);
    delete pb;
}

int poisson_batch_create(const std::vector<ibmdem_ctx *> &cs, PoissonBatch **out, std::string &err) {
    *out = nullptr;
    if (cs.empty()) {
        err = "empty batch group";
        return IBMDEM_ERR_ARG;
    }
    const ibmdem_ctx *c0 = cs[0];
    for (const ibmdem_ctx *c : cs) {
        if (!poisson_batchable(c) || c->cs.precision != c0->cs.precision || c->cs.mg_pre != c0->cs.mg_pre ||
            c->cs.mg_post != c0->cs.mg_post || c->cs.poisson_max_iter != c0->cs.poisson_max_iter) {
            err = "cases of a batched solve must share precision, smoothing counts and iteration cap";
            return IBMDEM_ERR_ARG;
        }
    }
    PoissonBatch *pb = new (std::nothrow) PoissonBatch();
    if (!pb) return IBMDEM_ERR_ALLOC;
    pb->cs = cs;
    // the FP64 V-cycle's level 0 is the CG vectors (as precondition sets it)
    for (ibmdem_ctx *c : cs) {
        c->lev64[0].b = c->cg_r;
        c->lev64[0].x = c->cg_z;
    }
    Arena ar;
    int rc = c0->cs.precision == IBMDEM_MIXED ? plan_all<float>(ar, pb->begin, pb->iter, cs, err)
                                              : plan_all<double>(ar, pb->begin, pb->iter, cs, err);
    std::vector<const double *> sp;
    for (ibmdem_ctx *c : cs) sp.push_back(c->scal);
    const size_t sp_off = ar.put(sp.data(), sp.size() * sizeof(double *));
    hipError_t e = hipSuccess;
    if (!rc) {
        e = hipMalloc((void **)&pb->arena, ar.bytes.size());
        if (e == hipSuccess) e = hipMemcpy(pb->arena, ar.bytes.data(), ar.bytes.size(), hipMemcpyHostToDevice);
        if (e == hipSuccess) e = hipMalloc((void **)&pb->gather_dev, cs.size() * SC_COUNT * sizeof(double));
        if (e == hipSuccess)
            e = hipHostMalloc((void **)&pb->gather_host, cs.size() * SC_COUNT * sizeof(double), hipHostMallocDefault);
        if (e != hipSuccess) {
            err = std::string("batched solver set-up: ") + hipGetErrorString(e);
            rc = IBMDEM_ERR_HIP;
        }
    }
    if (rc) {
        poisson_batch_destroy(pb);
        return rc;
    }
    for (auto *ops : {&pb->begin, &pb->iter})
        for (BOp &o : *ops) {
            o.first = (const int *)(pb->arena + o.first_off);
            o.arg = pb->arena + o.arg_off;
        }
    pb->scal_ptrs = (const double **)(pb->arena + sp_off);
    *out = pb;
    return IBMDEM_OK;
}

int poisson_batch_begin(PoissonBatch *pb, hipStream_t s, std::string &err) {
    return run_ops(pb->begin, s, 0, pb->prof, err);
}

int poisson_batch_iteration(PoissonBatch *pb, hipStream_t s, int it, std::string &err) {
    return run_ops(pb->iter, s, it, pb->prof, err);
}

void poisson_batch_set_profile(PoissonBatch *pb, bool on) { pb->prof.on = on; }
bool poisson_batch_profiling(const PoissonBatch *pb) { return pb->prof.on; }

void poisson_batch_profile_arm(PoissonBatch *pb, bool armed) {
    pb->prof.armed = armed;
    if (armed) pb->prof.n = 0;
}

int poisson_batch_profile_collect(PoissonBatch *pb, double *ms, int64_t *launches, double *bytes) {
    const BProf &pr = pb->prof;
    if (!pr.on) return IBMDEM_OK;
    for (int i = 0; i < pr.n; ++i) {
        float t = 0.0f;
        if (hipEventElapsedTime(&t, pr.ev[i], pr.ev[i + 1]) != hipSuccess) return IBMDEM_ERR_HIP;
        const int k = pr.kind[i];
        if (k < 0 || k >= BK_COUNT) continue;
        ms[k] += t;
        launches[k] += 1;
        bytes[k] += pr.bytes[i];
    }
    return IBMDEM_OK;
}

int poisson_batch_gather(PoissonBatch *pb, hipStream_t s, std::string &err) {
    const int n = (int)pb->cs.size();
    hipLaunchKernelGGL(kb_gather_scalars, dim3(n), dim3(64), 0, s, pb->scal_ptrs, n, pb->gather_dev);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipMemcpyAsync(pb->gather_host, pb->gather_dev, (size_t)n * SC_COUNT * sizeof(double),
                           hipMemcpyDeviceToHost, s);
    if (e != hipSuccess) {
        err = std::string("batched solver scalars: ") + hipGetErrorString(e);
        return IBMDEM_ERR_HIP;
    }
    return IBMDEM_OK;
}

const double *poisson_batch_scalars(const PoissonBatch *pb, int q) { return pb->gather_host + (size_t)q * SC_COUNT; }

int poisson_batch_launches(const PoissonBatch *pb, int k) {
    int n = (int)pb->begin.size();
    for (int it = 1; it <= k; ++it)
        for (const BOp &o : pb->iter) n += !(o.skip_first && it == 1);
    return n;
}

// poisson_gauge of every context of a group as one launch
namespace {
struct GaugeArg {
    BGrid g;
    const LevelDev *L;
    const double *x, *p, *scal;
    double *pc;
};
__global__ __launch_bounds__(RB) void kb_gauge(BTable<GaugeArg> tab) {
    batch_for(tab, [&](const GaugeArg &a, const Blk &kb) {
        gauge_body(kb, *cst(a.L), glb(a.x), glb(a.p), glb(a.scal), glb(a.pc));
    });
}
void launch_gauge(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_gauge, dim3(o.blocks), dim3(RB), 0, s, table<GaugeArg>(o));
}
}  // namespace

int poisson_plan_gauge(bk::BatchPlan &P, const std::vector<ibmdem_ctx *> &cs, std::string &err) {
    std::vector<GaugeArg> args;
    for (ibmdem_ctx *c : cs) {
        const LevelDev &L0 = c->lev64[0].d;
        const LaunchShape fs = shape_for(div_up(L0.nx, 2), L0.ny, L0.nz);
        args.push_back(GaugeArg{bgrid(fs.grid, fs.block), c->dlev, c->cg_x, c->cg_p, c->scal, c->pcorr});
    }
    return add_op(P.ar, P.ops, launch_gauge, RB, args, BOp(), err);
}

// poisson_begin_rhs of every context of a group: the pinned row's sum (the
// contexts without a Dirichlet side), r = b and x = 0, then ||b||
namespace {
__global__ __launch_bounds__(RB) void kb_cg_init(BTable<CgArg> tab) {
    batch_for(tab, [&](const CgArg &a, const Blk &kb) {
        cg_init_body(kb, *cst(a.L), glb(a.rhs), glb(a.r), glb(a.x), glb(a.scal), glb(a.r32));
    });
}
__global__ __launch_bounds__(RED_T) void kb_dot_rr(BTable<CgArg> tab) {
    batch_for(tab, [&](const CgArg &a, const Blk &kb) {
        dot_body(kb, a.n, glb((const double *)a.r), glb((const double *)a.r), glb(a.partial), glb(a.scal));
    });
}
void launch_cg_init(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_cg_init, dim3(o.blocks), dim3(RB), 0, s, table<CgArg>(o));
}
void launch_dot_rr(const BOp &o, hipStream_t s, int) {
    hipLaunchKernelGGL(kb_dot_rr, dim3(o.blocks), dim3(RED_T), 0, s, table<CgArg>(o));
}
}  // namespace

int poisson_plan_rhs(bk::BatchPlan &P, const std::vector<ibmdem_ctx *> &cs, std::string &err) {
    std::vector<ReduceJob> pin;
    std::vector<CgArg> init, dot, fin;
    for (ibmdem_ctx *c : cs) {
        const LevelDev &L0 = c->lev64[0].d;
        if (!L0.dirichlet) pin.push_back(ReduceJob{c->rhs, nullptr, c->n, 1, c->partial, c->scal + SC_PIN});
        const LaunchShape fs = shape_for(div_up(L0.nx, 2), L0.ny, L0.nz);
        CgArg a = cg_arg(c, fs.grid, fs.block, 0);
        a.rhs = c->rhs;
        init.push_back(a);
        dot.push_back(cg_arg(c, dim3(RED_BLOCKS), dim3(RED_T), 0));
        fin.push_back(cg_arg(c, dim3(1), dim3(FIN_T), RED_BLOCKS));
    }
    int rc;
    if ((rc = plan_reduce_sum(P, pin, err))) return rc;
    if ((rc = add_op(P.ar, P.ops, launch_cg_init, RB, init, BOp(), err))) return rc;
    if ((rc = add_op(P.ar, P.ops, launch_dot_rr, RED_T, dot, BOp(), err))) return rc;
    BOp o;
    o.slot = SC_BNORM2;
    o.op = 4;
    return add_op(P.ar, P.ops, launch_final, FIN_T, fin, o, err);
}
