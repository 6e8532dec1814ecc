// mgtile.hpp — half a V-cycle visit of a small multigrid level in one launch.
//
// Included by poisson.hip inside its anonymous namespace, after mgmarch.hpp.
//
// Launches on a small level cost their start and latencies (4-5 us each), not
// their work: smoothing, residual and restriction of a level take five
// launches, correction and smoothing as many. Here each of the two halves is
// one launch over tiles of TL_X x TL_Y x TL_Z cells: a work-group loads its
// tile with a halo as deep as the half has half sweeps (up to two sweeps; a
// half of more is led by launches that smooth alone, tile_smooths), keeps it
// in LDS and registers, and sweeps the whole extended tile a barrier apart. A sweep's
// values are exact one layer further in than its input's, so the tile itself
// is exact at the end; halo cells are the neighbouring tiles' cells with the
// same arithmetic, so the result does not depend on the tiling and each
// cell's value is that of the passes of mgmarch.hpp. The halo makes a tile's
// work 6 to 9 times its cells', which small levels leave the chip room for.
// In FP64 the two launches take 8.0 and 7.4 us at 32^3, 9.7 and 8.2 us at
// 64^3 (one launch per operation: 42 and 44 us), bound by the chain of sweeps
// and the start.
//
// A thread owns the x-pair p of row y in M consecutive planes: the values and
// right-hand sides of its cells are in registers (by colour: a pair has one
// red and one black cell), so of a cell's neighbours the pair's other cell
// and most z neighbours are the thread's own, and only the outer x, the y and
// the z neighbours at the ends of its planes are read from LDS.
constexpr int TL_X = 16, TL_Y = 8, TL_Z = 8;
static_assert(TL_X % 2 == 0 && TL_Y % 2 == 0 && TL_Z % 2 == 0, "whole coarse cells");

template <int HX, int H, int M_>
struct TileGeoC {
    static constexpr int RL = (TL_X + 2 * HX) / 2, EY = TL_Y + 2 * H, EZ = TL_Z + 2 * H, M = M_;
    static constexpr int PL = RL * EY;                 // pairs of a plane
    static constexpr int GT = (PL + 63) / 64 * 64;     // threads of a group of M planes
    static constexpr int NG = (EZ + M - 1) / M, NT = GT * NG;
    // LDS slots of a colour: a plane before and after, read by the outermost
    // cells (whose values are not exact in any case)
    static constexpr int SLOTS = (NG * M + 2) * PL;
    static_assert(HX % 2 == 0 && NT <= 1024, "tile shape");
};
using TileDown = TileGeoC<6, 5, 5>;   // two sweeps, the residual, one layer for the restriction
using TileUp = TileGeoC<4, 4, 4>;     // two sweeps

// Where a launch's red cells come from: b / diag (the first red sweep from x =
// 0), a launch before it, or that and the correction from the coarse level.
enum TileSrc { TS_B, TS_X, TS_PROLONG };

// level index of an unwrapped one: wrapped across a periodic side (however
// often the halo goes round a small level), -1 beyond another. (ct_map's
// values; its step ahead of the remainder costs these kernels 2 % of a CG
// iteration at 96^3.)
__device__ __forceinline__ int tl_map(int v, int n, int lo) {
    if (v >= 0 && v < n) return v;
    if (lo != IBMDEM_BC_PERIODIC) return -1;
    v %= n;
    return v < 0 ? v + n : v;
}

// A thread's cells of an extended tile.
template <typename T, class G>
struct TileCells {
    int q;             // LDS slot of plane 0 of its group's planes
    int s0;            // LDS offset of a red cell's outer x neighbour in even planes (m = 0, 2, ...); -s0 in odd ones
    int y, p, z;       // row, pair, first plane in the extended tile
    bool act;          // the thread has a column
    int pos[G::M];     // storage position (in either half) of the pair in plane m, -1 beyond a side
    T r[G::M], b[G::M];        // values, red and black
    T fr[G::M], fb[G::M];      // right-hand sides
    T ir[G::M], ib[G::M];      // 1/diag
};

template <typename T, class G>
__device__ __forceinline__ void tile_init(TileCells<T, G> &c, const LevelDev &L, int ox, int oy, int oz) {
    const int t = threadIdx.x, g = __builtin_amdgcn_readfirstlane(t / G::GT), col = t - g * G::GT;
    c.act = col < G::PL;
    const int cc = c.act ? col : 0;
    c.y = cc / G::RL;
    c.p = cc - c.y * G::RL;
    c.z = g * G::M;
    c.q = G::PL + c.z * G::PL + cc;
    const int rl = L.nx >> 1;
    const int i = tl_map(ox + 2 * c.p, L.nx, L.bt[0]), j = tl_map(oy + c.y, L.ny, L.bt[2]);
    // red is the pair's even cell where (j + k) is even (unwrapped parities
    // are the wrapped ones: periodic extents are even)
    c.s0 = ((oy + c.y + oz + c.z) & 1) ? 1 : -1;
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        const int k = tl_map(oz + c.z + m, L.nz, L.bt[4]);
        c.pos[m] = c.act && i >= 0 && j >= 0 && k >= 0 ? (k * L.ny + j) * rl + (i >> 1) : -1;
    }
}
// 1/diag and diag of the thread's cells: the interior values unless the
// extended tile reaches a side that is not periodic
template <typename T, class G>
__device__ __forceinline__ int tile_diag(const TileCells<T, G> &c, const LevelDev &L, int ox, int oy, int oz, int m,
                                         bool odd) {
    const int i = tl_map(ox + 2 * c.p, L.nx, L.bt[0]), j = tl_map(oy + c.y, L.ny, L.bt[2]),
              k = tl_map(oz + c.z + m, L.nz, L.bt[4]);
    return c.pos[m] >= 0 ? diag_index(L, i + (odd ? 1 : 0), j, k) : DIAG_INTERIOR;
}
__device__ __forceinline__ bool tile_plain(const LevelDev &L, int ox, int oy, int oz, int ex, int ey, int ez) {
    const bool px = L.bt[0] == IBMDEM_BC_PERIODIC, py = L.bt[2] == IBMDEM_BC_PERIODIC,
               pz = L.bt[4] == IBMDEM_BC_PERIODIC;
    return (px || (ox > 0 && ox + ex < L.nx)) && (py || (oy > 0 && oy + ey < L.ny)) &&
           (pz || (oz > 0 && oz + ez < L.nz));
}
template <typename T, class G>
__device__ __forceinline__ void tile_ids(TileCells<T, G> &c, const LevelDev &L, int ox, int oy, int oz, bool plain,
                                         const T *s_id) {
    const T id_int = T(L.idiag[DIAG_INTERIOR]);
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        T a = id_int, b = id_int;
        if (!plain) {
            const bool odd = (c.s0 > 0) != ((m & 1) != 0);   // the red cell is the odd one
            a = s_id[tile_diag(c, L, ox, oy, oz, m, odd)];
            b = s_id[tile_diag(c, L, ox, oy, oz, m, !odd)];
        }
        c.ir[m] = c.pos[m] >= 0 ? a : T(0);
        c.ib[m] = c.pos[m] >= 0 ? b : T(0);
    }
}

// nbsum of the thread's cell of one colour in plane m; v: the thread's values
// of the other colour, lds: that colour's LDS slots, side: outer x offset
template <typename T, class G>
__device__ __forceinline__ T tile_nb(const T (&v)[G::M], const T *lds, int q, int side, int m, T ihx2, T ihy2, T ihz2) {
    const T *o = lds + q + m * G::PL;
    const T zb = m > 0 ? v[m > 0 ? m - 1 : 0] : o[-G::PL];
    const T zt = m < G::M - 1 ? v[m < G::M - 1 ? m + 1 : m] : o[G::PL];
    const T sx = (v[m] + o[side]) * ihx2;
    const T syy = (o[-G::RL] + o[G::RL]) * ihy2;
    const T szz = (zb + zt) * ihz2;
    return sx + syy + szz;
}

// a half sweep of one colour, the planes whose values are still exact
// (layer and further in); the caller's barrier follows
template <typename T, class G>
__device__ __forceinline__ void tile_sweep(TileCells<T, G> &c, bool red, int layer, T *sr, T *sb, T ihx2, T ihy2,
                                           T ihz2) {
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        if (c.z + m < layer || c.z + m >= G::EZ - layer) continue;   // the same on every lane
        const int side = red != ((m & 1) != 0) ? c.s0 : -c.s0;
        if (red) {
            c.r[m] = (c.fr[m] + tile_nb<T, G>(c.b, sb, c.q, side, m, ihx2, ihy2, ihz2)) * c.ir[m];
            if (c.act) sr[c.q + m * G::PL] = c.r[m];
        } else {
            c.b[m] = (c.fb[m] + tile_nb<T, G>(c.r, sr, c.q, side, m, ihx2, ihy2, ihz2)) * c.ib[m];
            if (c.act) sb[c.q + m * G::PL] = c.b[m];
        }
    }
}

// The last pre-smoothing sweeps, the residual and its restriction: b of the
// level (and, TS_X, the red cells' x) in, the red cells' x (xr, a half) and
// the coarse level's b out. From the first red sweep on (TS_B) or from xin:
// black and red once more if `more`, then black.
template <typename T, int SRC>
__device__ __forceinline__ void tile_down_body(const Blk &kb, const LevelDev &L, const T *__restrict__ bg,
                                               const T *__restrict__ xin, bool more, T *__restrict__ xr,
                                               const LevelDev &Cl, T *__restrict__ bc,
                                               const double *__restrict__ stop) {
    static_assert(SRC != TS_PROLONG, "the way down has no correction");
    using G = TileDown;
    const double stopped = *stop;   // waited for with the first loads
    __shared__ T sr[G::SLOTS], sb[G::SLOTS], s_id[64], s_dg[64];
    const int t = threadIdx.x;
    const int ox = kb.bx * TL_X - 6, oy = kb.by * TL_Y - 5, oz = kb.bz * TL_Z - 5;
    const T ihx2 = T(L.ihx2), ihy2 = T(L.ihy2), ihz2 = T(L.ihz2);
    if (t < 64) {
        s_id[t] = T(L.idiag[t]);
        s_dg[t] = T(L.diag[t]);
    }
    TileCells<T, G> c;
    tile_init(c, L, ox, oy, oz);
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        const int g = max(c.pos[m], 0);
        c.fr[m] = bg[g];
        c.fb[m] = bg[L.half + g];
        if (SRC == TS_X) c.r[m] = xin[g];
    }
    const bool plain = tile_plain(L, ox, oy, oz, 2 * G::RL, G::EY, G::EZ);
    __syncthreads();   // the tables
    if (stopped != 0.0) return;
    tile_ids(c, L, ox, oy, oz, plain, s_id);
    // cells beyond a side stay 0: (0 + nbsum) * 0 of the zeros and finite
    // values around them
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        c.fr[m] = c.pos[m] >= 0 ? c.fr[m] : T(0);
        c.fb[m] = c.pos[m] >= 0 ? c.fb[m] : T(0);
        if (SRC == TS_X) c.r[m] = c.pos[m] >= 0 ? c.r[m] : T(0);
        else c.r[m] = (c.fr[m] + T(0)) * c.ir[m];
        c.b[m] = T(0);
        if (c.act) {
            sr[c.q + m * G::PL] = c.r[m];
            sb[c.q + m * G::PL] = T(0);
        }
    }
    __syncthreads();
    if (more) {
        tile_sweep(c, false, 1, sr, sb, ihx2, ihy2, ihz2);
        __syncthreads();
        tile_sweep(c, true, 2, sr, sb, ihx2, ihy2, ihz2);
        __syncthreads();
    }
    T rb[G::M];   // the black cells' residual (FP32)
    const T dg_int = T(L.diag[DIAG_INTERIOR]);
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        rb[m] = T(0);
        if (c.z + m < 3 || c.z + m >= G::EZ - 3) continue;
        const int side = (m & 1) ? c.s0 : -c.s0;
        const T s = tile_nb<T, G>(c.r, sr, c.q, side, m, ihx2, ihy2, ihz2);
        c.b[m] = (c.fb[m] + s) * c.ib[m];
        if (c.act) sb[c.q + m * G::PL] = c.b[m];
        if (RES_BLACK<T>) {
            T dg = dg_int;
            if (!plain) dg = s_dg[tile_diag(c, L, ox, oy, oz, m, (c.s0 > 0) == ((m & 1) != 0))];
            rb[m] = c.pos[m] >= 0 ? c.fb[m] - (dg * c.b[m] - s) : T(0);
        }
    }
    __syncthreads();
    // the residual of the red cells takes their place in LDS (it reads black
    // cells alone), their x goes out
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        if (c.z + m < 4 || c.z + m >= G::EZ - 4) continue;
        const int side = (m & 1) ? -c.s0 : c.s0;
        T dg = dg_int;
        if (!plain) dg = s_dg[tile_diag(c, L, ox, oy, oz, m, (c.s0 > 0) != ((m & 1) != 0))];
        const T s = tile_nb<T, G>(c.b, sb, c.q, side, m, ihx2, ihy2, ihz2);
        if (c.act) sr[c.q + m * G::PL] = c.fr[m] - (dg * c.r[m] - s);
        const int j = oy + c.y, k = oz + c.z + m, i = ox + 2 * c.p;
        if (c.act && c.p >= 3 && c.p < 3 + TL_X / 2 && c.y >= 5 && c.y < 5 + TL_Y && c.z + m >= 5 &&
            c.z + m < 5 + TL_Z && i < L.nx && j < L.ny && k < L.nz)
            xr[c.pos[m]] = c.r[m];
    }
    if (RES_BLACK<T>) {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < G::M; ++m)
            if (c.act) sb[c.q + m * G::PL] = rb[m];
    }
    __syncthreads();
    constexpr int CX = TL_X / 2, CY = TL_Y / 2, CZ = TL_Z / 2;
    if (t >= CX * CY * CZ) return;
    const int I = kb.bx * CX + t % CX, J = kb.by * CY + t / CX % CY, K = kb.bz * CZ + t / (CX * CY);
    if (I >= Cl.nx || J >= Cl.ny || K >= Cl.nz) return;
    const bool px = L.bt[0] == IBMDEM_BC_PERIODIC, py = L.bt[2] == IBMDEM_BC_PERIODIC,
               pz = L.bt[4] == IBMDEM_BC_PERIODIC;
    const bool lo = I == 0 && !px, hi = I == Cl.nx - 1 && !px;
    const T wt[4] = {T(0.25), T(0.75), T(0.75), T(0.25)};
    T s = T(0);
#pragma unroll
    for (int c3 = 0; c3 < 4; ++c3) {
        int k = 2 * K - 1 + c3;
        if (!pz) k = min(max(k, 0), L.nz - 1);
#pragma unroll
        for (int c2 = 0; c2 < 4; ++c2) {
            int j = 2 * J - 1 + c2;
            if (!py) j = min(max(j, 0), L.ny - 1);
            const int o = G::PL + (k - oz) * G::PL + (j - oy) * G::RL + I - (ox >> 1);
            s = restrict_row(s, wt[c3] * wt[c2], ((j + k) & 1) == 0, lo, hi, [&](int d) { return sr[o + d]; },
                             [&](int d) { return sb[o + d]; });
        }
    }
    bc[lidx(Cl, I, J, K)] = T(0.125) * s;
}
template <typename T, int SRC>
__global__ __launch_bounds__(TileDown::NT) void k_tile_down(LevelDev L, const T *__restrict__ bg,
                                                            const T *__restrict__ xin, bool more, T *__restrict__ xr,
                                                            LevelDev Cl, T *__restrict__ bc,
                                                            const double *__restrict__ stop) {
    tile_down_body<T, SRC>(hw_blk(), L, bg, xin, more, xr, Cl, bc, stop);
}

// whether pair m of a thread lies in the tile itself (not its halo)
template <typename G, typename C>
__device__ __forceinline__ bool tile_owns(const C &c, const LevelDev &L, int ox, int oy, int oz, int m) {
    const int j = oy + c.y, k = oz + c.z + m, i = ox + 2 * c.p;
    return c.act && c.p >= 2 && c.p < 2 + TL_X / 2 && c.y >= 4 && c.y < 4 + TL_Y && c.z + m >= 4 &&
           c.z + m < 4 + TL_Z && i < L.nx && j < L.ny && k < L.nz;
}
// the block's partial sum: NW wavefronts by shuffles, then in order
template <int NW>
__device__ __forceinline__ void tile_partial(const Blk &kb, double dsum, double *__restrict__ partial) {
    const int t = threadIdx.x;
    __shared__ double red[NW];
    for (int st = 32; st > 0; st >>= 1) dsum += __shfl_down(dsum, st, 64);
    if ((t & 63) == 0) red[t >> 6] = dsum;
    __syncthreads();
    if (t == 0) {
        double a = 0.0;
        for (int w = 0; w < NW; ++w) a += red[w];
        partial[((long)kb.bz * kb.gy + kb.by) * kb.gx + kb.bx] = a;
    }
}

// One or two (`two`) sweeps, each black and then red: after the correction of
// the red cells (TS_PROLONG: the red cells' x of tile_down and the coarse
// level's x in), on a launch before this one (TS_X), or after the first red
// sweep from x = 0 (TS_B). The red cells' x out, and with xb the black ones';
// with partial, one partial sum of b.x per block (level 0: r.z).
template <typename T, int SRC>
__device__ __forceinline__ void tile_up_body(const Blk &kb, const LevelDev &L, const T *__restrict__ bg,
                                             const T *__restrict__ xr, T *__restrict__ x, T *__restrict__ xb, bool two,
                                             const LevelDev &Cl, const T *__restrict__ xc,
                                             double *__restrict__ partial, const double *__restrict__ stop) {
    using G = TileUp;
    const double stopped = *stop;
    __shared__ T sr[G::SLOTS], sb[G::SLOTS], s_id[64];
    // coarse parents of the extended tile: its coarse cells and one around
    constexpr int CX = G::RL + 2, CY = G::EY / 2 + 2, CZ = G::EZ / 2 + 2, CN = CX * CY * CZ;
    __shared__ T sc[CN];
    const int t = threadIdx.x;
    const int ox = kb.bx * TL_X - 4, oy = kb.by * TL_Y - 4, oz = kb.bz * TL_Z - 4;
    const T ihx2 = T(L.ihx2), ihy2 = T(L.ihy2), ihz2 = T(L.ihz2);
    if (t < 64) s_id[t] = T(L.idiag[t]);
    TileCells<T, G> c;
    tile_init(c, L, ox, oy, oz);
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        const int g = max(c.pos[m], 0);
        if (SRC != TS_B) c.r[m] = xr[g];
        c.fr[m] = bg[g];
        c.fb[m] = bg[L.half + g];
    }
    constexpr int CM = (CN + G::NT - 1) / G::NT;
    T cv[CM];   // (TS_PROLONG)
    // a coarse coordinate beyond the level: wrapped, or the edge cell again
    auto cmap = [](int v, int n, int lo) {
        if (v >= 0 && v < n) return v;
        if (lo != IBMDEM_BC_PERIODIC) return min(max(v, 0), n - 1);
        v %= n;
        return v < 0 ? v + n : v;
    };
#pragma unroll
    for (int u = 0; u < (SRC == TS_PROLONG ? CM : 0); ++u) {
        const int q = min(t + u * G::NT, CN - 1), zz = q / (CX * CY), yy = q / CX % CY, xx = q % CX;
        cv[u] = xc[lidx(Cl, cmap((ox >> 1) - 1 + xx, Cl.nx, Cl.bt[0]), cmap((oy >> 1) - 1 + yy, Cl.ny, Cl.bt[2]),
                        cmap((oz >> 1) - 1 + zz, Cl.nz, Cl.bt[4]))];
    }
    const bool plain = tile_plain(L, ox, oy, oz, 2 * G::RL, G::EY, G::EZ);
#pragma unroll
    for (int u = 0; u < (SRC == TS_PROLONG ? CM : 0); ++u)
        if (t + u * G::NT < CN) sc[t + u * G::NT] = cv[u];
    __syncthreads();
    if (stopped != 0.0) return;
    tile_ids(c, L, ox, oy, oz, plain, s_id);
    const T wt[2] = {T(0.75), T(0.25)};
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        c.fr[m] = c.pos[m] >= 0 ? c.fr[m] : T(0);
        c.fb[m] = c.pos[m] >= 0 ? c.fb[m] : T(0);
        c.b[m] = T(0);
        if (c.act) sb[c.q + m * G::PL] = T(0);
        if (SRC != TS_PROLONG) {
            if (SRC == TS_X) c.r[m] = c.pos[m] >= 0 ? c.r[m] : T(0);
            else c.r[m] = (c.fr[m] + T(0)) * c.ir[m];
            if (c.act) sr[c.q + m * G::PL] = c.r[m];
            continue;
        }
        // parents: the own coarse cell and the neighbour on the cell's side
        const int xx[2] = {c.p + 1, c.p + 1 + ((m & 1) ? -c.s0 : c.s0)};
        const int yo = oy + c.y, zo = oz + c.z + m;
        const int yy[2] = {c.y / 2 + 1, c.y / 2 + 1 + ((yo & 1) ? 1 : -1)};
        const int zz[2] = {(c.z + m) / 2 + 1, (c.z + m) / 2 + 1 + ((zo & 1) ? 1 : -1)};
        T s = T(0);
#pragma unroll
        for (int c3 = 0; c3 < 2; ++c3)
#pragma unroll
            for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
                for (int c1 = 0; c1 < 2; ++c1)
                    s = s + wt[c3] * wt[c2] * wt[c1] * sc[(zz[c3] * CY + yy[c2]) * CX + xx[c1]];
        c.r[m] = c.pos[m] >= 0 ? c.r[m] + s : T(0);
        if (c.act) sr[c.q + m * G::PL] = c.r[m];
    }
    __syncthreads();
    tile_sweep(c, false, 1, sr, sb, ihx2, ihy2, ihz2);
    __syncthreads();
    tile_sweep(c, true, 2, sr, sb, ihx2, ihy2, ihz2);
    if (two) {
        __syncthreads();
        tile_sweep(c, false, 3, sr, sb, ihx2, ihy2, ihz2);
        __syncthreads();
        tile_sweep(c, true, 4, sr, sb, ihx2, ihy2, ihz2);
    }
    double dsum = 0.0;
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        if (tile_owns<G>(c, L, ox, oy, oz, m)) {
            x[c.pos[m]] = c.r[m];
            if (xb) xb[c.pos[m]] = c.b[m];
            dsum += double(c.fr[m]) * double(c.r[m]);
            dsum += double(c.fb[m]) * double(c.b[m]);
        }
    }
    if (partial) tile_partial<G::NT / 64>(kb, dsum, partial);
}
template <typename T, int SRC>
__global__ __launch_bounds__(TileUp::NT) void k_tile_up(LevelDev L, const T *__restrict__ bg,
                                                        const T *__restrict__ xr, T *__restrict__ x,
                                                        T *__restrict__ xb, bool two, LevelDev Cl,
                                                        const T *__restrict__ xc, double *__restrict__ partial,
                                                        const double *__restrict__ stop) {
    tile_up_body<T, SRC>(hw_blk(), L, bg, xr, x, xb, two, Cl, xc, partial, stop);
}

// tile_up_body's partial sums of b.x from an x that is there already: a batch
// whose level 0 marches still sums r.z as each case's own launch does, so
// this is bound by memory. It runs the two groups of wavefronts that hold the
// tile's planes (the outer two's are halo and add 0), the loads ahead of the
// stop flag: a step of 20 cases of 64^3 takes 5.95 ms, 6.23 ms with all four
// groups, which left half of the CUs' wavefronts idle.
constexpr int TRZ_NT = 2 * TileUp::GT;
static_assert(TileUp::GT % 64 == 0 && TL_Z == 2 * TileUp::M && TileUp::NG == 4, "the tile is the middle two groups");
template <typename T>
__device__ __forceinline__ void tile_rz_body(const Blk &kb, const LevelDev &L, const T *__restrict__ bg,
                                             const T *__restrict__ x, double *__restrict__ partial,
                                             const double *__restrict__ stop) {
    using G = TileUp;
    const double stopped = *stop;   // waited for with the loads
    const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x / G::GT), col = threadIdx.x - g * G::GT;
    const int y = col / G::RL, p = col - y * G::RL;   // tile_init's column
    const int i = kb.bx * TL_X + 2 * (p - 2), j = kb.by * TL_Y + y - 4, k0 = kb.bz * TL_Z + g * G::M;
    const bool own = col < G::PL && p >= 2 && p < 2 + TL_X / 2 && y >= 4 && y < 4 + TL_Y && i < L.nx && j < L.ny;
    const int pl = (L.nx >> 1) * L.ny, pos = own ? k0 * pl + j * (L.nx >> 1) + (i >> 1) : 0;
    T v[G::M][4];
#pragma unroll
    for (int m = 0; m < G::M; ++m) {
        const int q = own && k0 + m < L.nz ? pos + m * pl : 0;
        v[m][0] = bg[q];
        v[m][1] = x[q];
        v[m][2] = bg[L.half + q];
        v[m][3] = x[L.half + q];
    }
    if (stopped != 0.0) return;
    double dsum = 0.0;
#pragma unroll
    for (int m = 0; m < G::M; ++m)
        if (own && k0 + m < L.nz) {
            dsum += double(v[m][0]) * double(v[m][1]);
            dsum += double(v[m][2]) * double(v[m][3]);
        }
    tile_partial<TRZ_NT / 64>(kb, dsum, partial);
}

// The launches of a visit. Before tile_down (q = 0 ..) and from tile_down's
// coarse level back up, each of one or two sweeps; the last one up writes x.
int tile_smooths(int pre) { return pre > 2 ? div_up(pre - 2, 2) : 0; }
bool tile_smooth_two(int pre, int q) { return pre - 2 - 2 * q >= 2; }
int tile_ups(int post) { return div_up(post, 2); }
bool tile_up_two(int post, int q) { return post - 2 * q >= 2; }

dim3 tile_grid(const LevelDev &d) { return dim3(div_up(d.nx, TL_X), div_up(d.ny, TL_Y), div_up(d.nz, TL_Z)); }
