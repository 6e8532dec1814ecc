// mgmarch.hpp — two fused half sweeps of a multigrid level, marching in z.
//
// Included by poisson.hip inside its anonymous namespace.
//
// A V-cycle visit of a level smooths red, black, red, black, ... from x = 0,
// takes the residual, and after the coarse correction smooths black, red,
// black, red, ... . A half sweep reads only the other colour, so
//   - the first red sweep is b / diag, which the black sweep after it can form
//     from b as it loads it;
//   - the black values a sweep leaves are read by the next red sweep (or the
//     residual) alone, so fused with it they need not be stored;
//   - the residual of the black cells, whose last update was made with the
//     same red values, is zero but for the rounding of that update, and is
//     left out in FP64. In FP32 that rounding (6e-8 of b) is kept: it is
//     part of the preconditioner the mixed form has had, and a change of it
//     moves the solution within the solve's tolerance, which the FP32
//     predictor's rounding of its input then amplifies to 1e-8;
//   - the correction of the black cells is overwritten by the first black
//     sweep after it, so only red cells are prolonged.
// Each pass here is therefore "black, then red" (stage A, stage B) on the red
// half of the level, out of place:
//   MODE 0  stage B relaxes, the red cells are written
//   MODE 1  stage B forms the residual of the red cells (last pre-smoothing
//           pass), that is written (in FP32 the black cells' too)
//   MODE 2  stage B relaxes and both colours are written, with the partial
//           sums of r.z (last post-smoothing pass at level 0 in FP64: x is z,
//           b is r); MODE 3 the same without the sums (other levels)
// FROMB passes take their red input from b (first pre-smoothing pass). PRO
// passes (FP64, the first post-smoothing pass) add the coarse correction to
// it as they load it: a thread interpolates each coarse plane in x and y once,
// to either side of its pairs, and two of those planes in z per fine plane,
// so the corrected red cells are neither written nor read again. (In FP32 the
// prolongation keeps its launch and with it its order of summation, for the
// reason above.)
// A level then moves 1.5 + 2 + 2 + 2.5 of its cells per V-cycle (pre = post
// = 2) where one launch per half sweep and one for the residual moved 14.5,
// in 4 launches instead of 9. At 256^3 in FP64 the four take 41, 44, 66
// (with the prolongation, 41 without) and 50 us (about 6 TB/s on those bytes
// but for the first, 4.9; the separate ones took 311 us), bound by HBM; on small levels by the steps (0.8 us each).
//
// A work-group owns a tile of rows (whole rows up to 64 x-pair groups, ranges
// of a row above) and marches up a chunk of planes, each thread with one
// group of PW adjacent x-pairs of one row. At step P it has loaded plane P of
// the red input, computes the black values of plane P - 1 and from them the
// red ones of plane P - 2: z neighbours are the thread's own registers, x and
// y neighbours come from LDS, where every step leaves the red plane P and the
// black plane P - 1 for the next (two buffers each, so one barrier a step).
// The next step's loads are issued before the step's arithmetic. The tile's
// outer two rows (and, in tiled rows, outer threads) are halo: their red
// input is loaded and the inner halo row's black values are computed again by
// each tile, with the same arithmetic, so a cell's value does not depend on
// the tiling.

struct MarchShape {
    int lx, ry;        // thread columns and rows of a tile (halo included)
    int ty;            // rows a tile owns
    int ntx, nty, nzc; // tiles per row, per plane, chunks
    int txl;           // groups a tile owns
    int nzp;           // planes a chunk owns
};
constexpr int MT = 1024;   // threads of a work-group
template <typename T>
constexpr bool RES_BLACK = std::is_same<T, float>::value;   // the black cells' residual is kept

// The shape a level's passes take, for PW pairs per thread. Whole rows where
// they are at most 64 groups (no x halo), else ranges with a halo group on
// each side; as many rows as the work-group holds, evenly spread; chunks so
// that the launch has about one work-group per CU (in FP64 a work-group fills
// a CU's registers; two in FP32), at least MARCH_MIN planes each (a chunk also
// loads four halo planes). A CG iteration with 2, 4 and 8 planes at least, us:
// 64^3 mixed 143, 148, 161; 128^3 222, 225, 247, mixed 234, 214, 228; 256^3 740,
// 739, 770, mixed 758, 734, 759.
constexpr int MARCH_MIN = 4;
template <typename T>
__host__ __device__ inline MarchShape march_shape(const LevelDev &d, int pw) {
    MarchShape s;
    const int groups = (d.nx >> 1) / pw;
    s.ntx = groups <= 64 ? 1 : (groups + 63) / 64;
    s.txl = (groups + s.ntx - 1) / s.ntx;
    s.lx = s.ntx == 1 ? groups : s.txl + 2;
    const int most = MT / s.lx - 4;   // lx <= 66: at least 11 rows
    s.nty = (d.ny + most - 1) / most;
    s.ty = (d.ny + s.nty - 1) / s.nty;
    s.ry = s.ty + 4;
    const int tiles = s.ntx * s.nty, slots = sizeof(T) == 8 ? 256 : 512, want = tiles < slots ? slots / tiles : 1;
    int per = (d.nz + want - 1) / want;
    per = per < MARCH_MIN ? MARCH_MIN : per;
    s.nzc = (d.nz + per - 1) / per;
    s.nzp = (d.nz + s.nzc - 1) / s.nzc;
    return s;
}
// The chunk length of a launch over a batch of cases (their levels d, all of
// pw pairs): the one whose work-groups are through in the fewest steps. A chunk
// of `per` planes is per + 4 steps, and an XCD, whose 32 CUs hold `wgs`
// work-groups each, takes the case's chunks in batch_for's ranges. Chunks that
// gave each case its share of one or two rounds left some XCDs a round behind:
// a step of 20 cases of 64^3 in FP64 took 5.90 ms with them and takes 5.47, two
// of 128^3 4.59 and 4.22, 64 uneven settling cases 28.5 and 25.8 (mixed 26.2
// and 23.8).
template <typename T>
int march_planes(const std::vector<LevelDev> &d, int pw, int wgs) {
    int best = MARCH_MIN, most = MARCH_MIN;
    long cost = LONG_MAX;
    std::vector<int> plane;
    for (const LevelDev &l : d) {
        const MarchShape s = march_shape<T>(l, pw);
        plane.push_back(s.ntx * s.nty);
        most = std::max(most, l.nz);
    }
    for (int per = MARCH_MIN; per <= most; ++per) {
        double n[8] = {};
        for (size_t q = 0; q < d.size(); ++q) {
            const int nb = plane[q] * div_up(d[q].nz, per);
            for (int x = 0; x < 8; ++x) {
                int lo, hi;
                xcd_range(nb, 1, x, lo, hi);
                n[x] += nb >= 8 ? hi - lo : nb / 8.0;
            }
        }
        const long c = (long)std::ceil(*std::max_element(n, n + 8) / (32 * wgs)) * (per + 4);
        if (c < cost) {
            cost = c;
            best = per;
        }
        if (c <= per + 4) break;   // one round: longer chunks take longer
    }
    return best;
}

// wavefronts per SIMD the registers are held to: two work-groups per CU for
// the FP32 passes that fit (65 registers without it)
template <typename T, int MODE>
constexpr int MARCH_WAVES = sizeof(T) == 4 && (MODE == 0 || MODE == 3) ? 8 : 4;

// PW values of a colour half
template <typename T, int PW>
__device__ __forceinline__ void ldp(const T *p, T (&v)[PW]) {
    if constexpr (PW == 2) ld2(p, v[0], v[1]);
    else v[0] = p[0];
}
template <typename T, int PW>
__device__ __forceinline__ void stp(T *p, const T (&v)[PW]) {
    if constexpr (PW == 2) st2(p, v[0], v[1]);
    else p[0] = v[0];
}

template <typename T, int PW, int MODE, bool FROMB, bool PRO>
__device__ __forceinline__ void march_body(const Blk &kb, const LevelDev &L, const T *__restrict__ xin,
                                           const T *__restrict__ b, T *__restrict__ out, T *__restrict__ out2,
                                           double *__restrict__ partial, int nzp, const T *__restrict__ xc,
                                           const double *__restrict__ stop) {
    const double stopped = *stop;   // waited for with the first loads
    __shared__ T s_r[2][MT * PW], s_b[2][MT * PW], s_id[64], s_dg[64];
    const MarchShape sh = march_shape<T>(L, PW);
    const int t = threadIdx.x, ty = t / sh.lx, tx = t - ty * sh.lx;
    if (t < 64) {
        s_id[t] = T(L.idiag[t]);
        s_dg[t] = T(L.diag[t]);
    }
    const T ihx2 = T(L.ihx2), ihy2 = T(L.ihy2), ihz2 = T(L.ihz2);
    const bool px = L.bt[0] == IBMDEM_BC_PERIODIC, py = L.bt[2] == IBMDEM_BC_PERIODIC,
               pz = L.bt[4] == IBMDEM_BC_PERIODIC;
    const int rl = L.nx >> 1, pl = rl * L.ny;
    // the thread's group and row: inside the level, wrapped across a periodic
    // side, or (beyond another side) a column of zeros
    const int y0 = kb.by * sh.ty, z0 = kb.bz * nzp, z1 = min(z0 + nzp, L.nz);
    const int j = y0 - 2 + ty;
    int p = (kb.bx * sh.txl + tx - (sh.ntx > 1 ? 1 : 0)) * PW, jr = j;
    bool valid = ty < sh.ry;
    if (p < 0 || p >= rl) {
        valid = valid && px;
        p = p < 0 ? p + rl : p - rl;   // a tile reaches at most one group (and its ragged end) beyond the row
        if (p < 0 || p >= rl) p = 0, valid = false;
    }
    if (jr < 0 || jr >= L.ny) {
        valid = valid && py;
        jr %= L.ny;
        jr = jr < 0 ? jr + L.ny : jr;
    }
    const int pos = jr * rl + p;
    const bool inA = valid && ty >= 1 && ty < sh.ry - 1;
    const bool own = valid && ty >= 2 && ty < sh.ry - 2 && j < L.ny && j < y0 + sh.ty &&
                     (sh.ntx == 1 || (tx >= 1 && tx <= sh.txl && (kb.bx * sh.txl + tx - 1) * PW < rl));
    // LDS positions of the x neighbours outside the group: -1 none (0)
    const int me = t * PW, row0 = ty * sh.lx * PW, rw = sh.lx * PW;
    const bool wrap = sh.ntx == 1 && px;
    const int iw = tx > 0 ? me - 1 : (wrap ? row0 + rw - 1 : -1);
    const int ie = tx < sh.lx - 1 ? me + PW : (wrap ? row0 : -1);
    int cxe[PW], cxo[PW];
#pragma unroll
    for (int c = 0; c < PW; ++c) {
        cxe[c] = diag_count(2 * (p + c), L.nx, L.bt[0], L.bt[1]) * 16;
        cxo[c] = diag_count(2 * (p + c) + 1, L.nx, L.bt[0], L.bt[1]) * 16;
    }
    const int cy = diag_count(jr, L.ny, L.bt[2], L.bt[3]) * 4;
    // plane k (-2 .. nz + 1) wrapped across a periodic side; absent beyond others
    auto zwrap = [&](int k) { return k < 0 ? (pz ? k + L.nz : 0) : (k < L.nz ? k : (pz ? k - L.nz : 0)); };
    auto zhere = [&](int k) { return pz || (k >= 0 && k < L.nz); };
    auto zcount = [&](int kr) { return diag_count(kr, L.nz, L.bt[4], L.bt[5]); };
    // In step P the cells of one row that are loaded (red of plane P), updated
    // in stage A (black of plane P - 1) and in stage B (red of plane P - 2)
    // are all the even ones of their pairs, or all the odd ones, and the
    // other way round in the next step: w[0] holds what the even steps
    // use, w[1] what the odd ones do: whether the cells are odd (their outer
    // x neighbour lies east), that neighbour's LDS position, 1/diag and diag
    // of the cells in planes with both z neighbours.
    struct Way {
        bool odd, has;
        int q;
        T id[PW], dg[PW];
        int di[PW];
    } w[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        w[e].odd = ((j + z0 + e) & 1) != 0;
        const int q = w[e].odd ? ie : iw;
        w[e].has = q >= 0;
        w[e].q = max(q, 0);
#pragma unroll
        for (int c = 0; c < PW; ++c) {
            w[e].di[c] = (w[e].odd ? cxo[c] : cxe[c]) + cy;
            w[e].id[c] = T(L.idiag[w[e].di[c] + 2]);
            w[e].dg[c] = MODE == 1 ? T(L.diag[w[e].di[c] + 2]) : T(0);
        }
    }
    const T *bb = b + L.half;
    // x neighbour of each cell of the group outside its own pair
    auto side = [&](const T (&v)[PW], const T *lds, const Way &y, T (&o)[PW]) {
        const T l = lds[y.q], out1 = y.has ? l : T(0);
        if constexpr (PW == 2) {
            o[0] = y.odd ? v[1] : out1;
            o[1] = y.odd ? out1 : v[0];
        } else {
            o[0] = out1;
        }
    };
    auto sum = [&](const T (&v)[PW], const T (&o)[PW], const T *lds, const T (&zb)[PW], const T (&zt)[PW], T (&s)[PW]) {
        T ys[PW], yn[PW];
        ldp<T, PW>(lds + me - rw, ys);
        ldp<T, PW>(lds + me + rw, yn);
#pragma unroll
        for (int c = 0; c < PW; ++c) {
            const T sx = (v[c] + o[c]) * ihx2;
            const T syy = (ys[c] + yn[c]) * ihy2;
            const T szz = (zb[c] + zt[c]) * ihz2;
            s[c] = sx + syy + szz;
        }
    };
    // 1/diag (diag) of the cells in plane kr
    auto ids = [&](const Way &y, int kr, const T (&in)[PW], const T *tab, T (&o)[PW]) {
        const int cz = zcount(kr);
#pragma unroll
        for (int c = 0; c < PW; ++c) o[c] = in[c];
        if (cz != 2) {
#pragma unroll
            for (int c = 0; c < PW; ++c) o[c] = tab[y.di[c] + cz];
        }
    };
    // r*: red input of planes P-2, P-1, P; k*: black values of planes P-3,
    // P-2, P-1; with FROMB the right-hand sides of the red planes stay
    // alongside
    T r0[PW], r1[PW], r2[PW], k0[PW], k1[PW], k2[PW], q0[PW], q1[PW], q2[PW], cb[PW];
    struct Next {   // a step's loads
        T r[PW], b[PW], q[PW];
    } n0, n1;
#pragma unroll
    for (int c = 0; c < PW; ++c) {
        r0[c] = r1[c] = r2[c] = k0[c] = k1[c] = k2[c] = q0[c] = q1[c] = q2[c] = cb[c] = T(0);
        n0.r[c] = n0.b[c] = n0.q[c] = n1.r[c] = n1.b[c] = n1.q[c] = T(0);
    }
    // loads of step P: red plane P, black right-hand side of plane P - 1, red
    // one of plane P - 2 (of absent planes: some plane's, not used)
    auto fetch = [&](int P, Next &n) {
        const long pr = (long)zwrap(P) * pl + pos, pa = (long)zwrap(max(P - 1, z0 - 1)) * pl + pos;
        const long pb = (long)max(P - 2, z0) * pl + pos;
        if (valid) ldp<T, PW>((FROMB ? b : xin) + pr, n.r);
        if (inA) ldp<T, PW>(bb + pa, n.b);
        if (!FROMB && own) ldp<T, PW>(b + pb, n.q);
    };
    // PRO: the coarse correction of the thread's red cells. The coarse level
    // has half the cells per dimension; columns p - 1 .. p + PW of rows J[0]
    // (the parent) and J[1] (the neighbour on the row's side), a missing one
    // beyond a side the parent's (parents()). In an even plane the red cell of
    // a pair lies to side A (east where j is odd), in an odd one to side B.
    struct Coarse {
        int nx, ny, nz, rl, half;   // (two pairs per thread: a split coarse row, one: an odd one)
        int ic[PW + 2], J[2];
        T raw[2][PW + 2], a[PW], ap[PW], b[PW];   // interpolated: side A of planes K, K - 1, side B of K
    } cg;
    if constexpr (PRO) {
        cg.nx = L.nx >> 1;
        cg.ny = L.ny >> 1;
        cg.nz = L.nz >> 1;
        cg.rl = PW == 2 ? cg.nx >> 1 : cg.nx;
        cg.half = PW == 2 ? cg.rl * cg.ny * cg.nz : 0;
        for (int c = 0; c < PW + 2; ++c) {
            const int i = p + c - 1;
            cg.ic[c] = i < 0 ? (px ? i + cg.nx : 0) : (i < cg.nx ? i : (px ? i - cg.nx : cg.nx - 1));
        }
        cg.J[0] = jr >> 1;
        const int jn = cg.J[0] + ((jr & 1) ? 1 : -1);
        cg.J[1] = jn < 0 ? (py ? jn + cg.ny : 0) : (jn < cg.ny ? jn : (py ? jn - cg.ny : cg.ny - 1));
    }
    auto coarse_load = [&](int K, T (&raw)[2][PW + 2]) {
        K = K < 0 ? (pz ? K + cg.nz : 0) : (K < cg.nz ? K : (pz ? K - cg.nz : cg.nz - 1));
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int o = (K * cg.ny + cg.J[q]) * cg.rl;
            if constexpr (PW == 2) {
                // p is even (and the coarse row split): columns p and p + 2 lie
                // in one colour half, p - 1 and p + 1 in the other
                const int h = ((cg.J[q] + K) & 1) ? cg.half : 0, even = o + h, odd = o + cg.half - h;
                raw[q][1] = xc[even + (p >> 1)];
                raw[q][2] = xc[odd + (p >> 1)];
                const T w = xc[odd + (cg.ic[0] >> 1)], e = xc[even + (cg.ic[PW + 1] >> 1)];
                raw[q][0] = cg.ic[0] == p ? raw[q][1] : w;
                raw[q][PW + 1] = cg.ic[PW + 1] == p + 1 ? raw[q][2] : e;
            } else {
#pragma unroll
                for (int c = 0; c < PW + 2; ++c) raw[q][c] = xc[o + cg.ic[c]];
            }
        }
    };
    // plane K interpolated in x and y, to side A and side B of each pair
    auto coarse_xy = [&](const T (&raw)[2][PW + 2], T (&a)[PW], T (&bs)[PW]) {
        const T w0 = T(0.75), w1 = T(0.25);
        const bool east = (j & 1) != 0;
#pragma unroll
        for (int c = 0; c < PW; ++c) {
            T lo[2], hi[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const T m = w0 * raw[q][c + 1];
                lo[q] = m + w1 * raw[q][c];
                hi[q] = m + w1 * raw[q][c + 2];
            }
            const T vw = w0 * lo[0] + w1 * lo[1], ve = w0 * hi[0] + w1 * hi[1];
            a[c] = east ? ve : vw;
            bs[c] = east ? vw : ve;
        }
    };
    // two steps' loads are in flight (each step reuses its own registers for
    // the step after the next), so a step does not wait for the memory latency
    fetch(z0 - 2, n0);
    fetch(z0 - 1, n1);
    if constexpr (PRO) {
        const int K = (z0 - 2) >> 1;
        T before[2][PW + 2];
#pragma unroll
        for (int c = 0; c < PW; ++c) cg.a[c] = cg.ap[c] = cg.b[c] = T(0);
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int c = 0; c < PW + 2; ++c) before[q][c] = cg.raw[q][c] = T(0);
        if (valid) {
            coarse_load(K - 1, before);
            coarse_load(K, cg.raw);
            coarse_xy(before, cg.ap, cg.b);
            coarse_xy(cg.raw, cg.a, cg.b);
            if (z0 & 1) coarse_load(K + 1, cg.raw);
        }
    }
    if (stopped != 0.0) return;
    double dsum = 0.0;
    if (ty < sh.ry && !inA) {   // black values beyond a side stay 0
        const T zero[PW] = {};
        stp<T, PW>(s_b[0] + me, zero);
        stp<T, PW>(s_b[1] + me, zero);
    }
    __syncthreads();   // the tables
    // The first two steps only load: their stages work on planes before the
    // chunk's and what they compute reaches nothing that is stored.
    auto step = [&](int P, Next &n, const Way &y, T *sr, const T *srp, const T *sb, T *sbw) {
        const bool vr = valid && zhere(P), va = inA && zhere(P - 1);
        const int kr = zwrap(P), ka = zwrap(P - 1);
        T idv[PW];
#pragma unroll
        for (int c = 0; c < PW; ++c) {
            r0[c] = r1[c];
            r1[c] = r2[c];
            k0[c] = k1[c];
            k1[c] = k2[c];
            if (FROMB) {
                q0[c] = q1[c];
                q1[c] = q2[c];
                q2[c] = n.r[c];
            } else {
                q0[c] = n.q[c];
            }
            cb[c] = n.b[c];
            r2[c] = n.r[c];
        }
        if constexpr (PRO) {
            // s = 3/4 of the parent plane K = P / 2 and 1/4 of K - 1 (P even)
            // or K + 1, whose values were loaded in the step before
            const T w0 = T(0.75), w1 = T(0.25);
            if (P & 1) {
                T a[PW], bs[PW];
                coarse_xy(cg.raw, a, bs);
#pragma unroll
                for (int c = 0; c < PW; ++c) {
                    r2[c] = r2[c] + (w0 * cg.b[c] + w1 * bs[c]);
                    cg.ap[c] = cg.a[c];
                    cg.a[c] = a[c];
                    cg.b[c] = bs[c];
                }
            } else {
#pragma unroll
                for (int c = 0; c < PW; ++c) r2[c] = r2[c] + (w0 * cg.a[c] + w1 * cg.ap[c]);
                if (valid && P + 1 < z1 + 2) coarse_load((P >> 1) + 1, cg.raw);
            }
        }
        if (FROMB) {
            ids(y, kr, y.id, s_id, idv);
#pragma unroll
            for (int c = 0; c < PW; ++c) r2[c] = (r2[c] + T(0)) * idv[c];
        }
#pragma unroll
        for (int c = 0; c < PW; ++c) r2[c] = vr ? r2[c] : T(0);
        if (P + 2 < z1 + 2) fetch(P + 2, n);
        if (ty < sh.ry) stp<T, PW>(sr + me, r2);
        // stage A: black of plane P - 1
        T s[PW], o[PW];
        if (inA) {
            side(r1, srp, y, o);
            sum(r1, o, srp, r0, r2, s);
            ids(y, ka, y.id, s_id, idv);
#pragma unroll
            for (int c = 0; c < PW; ++c) k2[c] = va ? (cb[c] + s[c]) * idv[c] : T(0);
            if ((MODE >= 2 || (MODE == 1 && RES_BLACK<T>)) && P - 1 >= z0 && P - 1 < z1 && own) {
                const long g = (long)ka * pl + pos;
                if constexpr (MODE == 1) {
                    T v[PW], dgv[PW];
                    ids(y, ka, y.dg, s_dg, dgv);
#pragma unroll
                    for (int c = 0; c < PW; ++c) v[c] = cb[c] - (dgv[c] * k2[c] - s[c]);
                    stp<T, PW>(out + L.half + g, v);
                } else {
                    stp<T, PW>(out2 + g, k2);
                    if (MODE == 2) {
#pragma unroll
                        for (int c = 0; c < PW; ++c) dsum += double(cb[c]) * double(k2[c]);
                    }
                }
            }
            stp<T, PW>(sbw + me, k2);   // black plane P - 1
        }
        // stage B: red of plane P - 2
        if (P - 2 >= z0 && own) {
            side(k1, sb, y, o);
            sum(k1, o, sb, k0, k2, s);
            const long g = (long)(P - 2) * pl + pos;
            T v[PW];
            ids(y, P - 2, MODE == 1 ? y.dg : y.id, MODE == 1 ? s_dg : s_id, idv);
            if (MODE == 1) {
#pragma unroll
                for (int c = 0; c < PW; ++c) v[c] = q0[c] - (idv[c] * r0[c] - s[c]);
                if (FROMB) stp<T, PW>(out2 + g, r0);
            } else {
#pragma unroll
                for (int c = 0; c < PW; ++c) v[c] = (q0[c] + s[c]) * idv[c];
            }
            stp<T, PW>(out + g, v);
            if (MODE == 2) {
#pragma unroll
                for (int c = 0; c < PW; ++c) dsum += double(q0[c]) * double(v[c]);
            }
        }
        __syncthreads();
    };
    // at an even step red plane P goes to buffer 0 (plane P - 1 is in 1) and
    // black plane P - 1 to buffer 1 (plane P - 2 is in 0), at an odd step the
    // other way round
    for (int P = z0 - 2; P < z1 + 2; P += 2) {
        step(P, n0, w[0], s_r[0], s_r[1], s_b[0], s_b[1]);
        if (P + 1 < z1 + 2) step(P + 1, n1, w[1], s_r[1], s_r[0], s_b[1], s_b[0]);
    }
    if (MODE == 2) {
        // the block's partial sum: wavefronts by shuffles, then in order
        __shared__ double red[MT / 64];
        for (int st = 32; st > 0; st >>= 1) dsum += __shfl_down(dsum, st, 64);
        if ((t & 63) == 0) red[t >> 6] = dsum;
        __syncthreads();
        if (t == 0) {
            double a = 0.0;
            for (int w = 0; w < MT / 64; ++w) a += red[w];
            partial[((long)kb.bz * sh.nty + kb.by) * sh.ntx + kb.bx] = a;
        }
    }
}

// Tiles that share halo rows on one XCD: XCD x (block b runs on XCD b % 8)
// takes the x-th contiguous eighth of the tiles.
__device__ __forceinline__ Blk march_blk(const MarchShape &sh) {
    const int nb = sh.ntx * sh.nty * sh.nzc, per = (nb + 7) >> 3;
    const int q = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    Blk kb = hw_blk();
    kb.bx = q % sh.ntx;
    kb.by = (q / sh.ntx) % sh.nty;
    kb.bz = (int)blockIdx.x >> 3 < per && q < nb ? q / (sh.ntx * sh.nty) : -1;
    return kb;
}
template <typename T, int PW, int MODE, bool FROMB, bool PRO>
__global__ __launch_bounds__(MT, (MARCH_WAVES<T, MODE>)) void k_march(LevelDev L, const T *__restrict__ xin,
                                                                      const T *__restrict__ b, T *__restrict__ out,
                                                                      T *__restrict__ out2,
                                                                      double *__restrict__ partial,
                                                                      const T *__restrict__ xc,
                                                                      const double *__restrict__ stop) {
    const MarchShape sh = march_shape<T>(L, PW);
    const Blk kb = march_blk(sh);
    if (kb.bz < 0) return;
    march_body<T, PW, MODE, FROMB, PRO>(kb, L, xin, b, out, out2, partial, sh.nzp, xc, stop);
}

// The last black and red sweeps at level 0 of the mixed form, one launch each:
// x of the other colour in, the x of the cells of `color` out, with one partial
// sum of r.z, z = double(x), per block over its cells. Each thread has PW pairs of two adjacent rows. These two are not
// fused: their partial sums keep one association (this block shape, a tree
// over its threads), since a change in the last bit of r.z reaches r's
// conversion to FP32 and from there the solution at the solve's tolerance.
// Bound by memory: 30 us a launch at 256^3 (35 us when an FP64 copy of z was
// written as well).
template <int PW>
__device__ __forceinline__ void rz_half_body(const Blk &kb, const LevelDev &L, const float *__restrict__ oth,
                                             float *__restrict__ own, int color, const double *__restrict__ r64,
                                             double *__restrict__ partial, long pofs,
                                             const double *__restrict__ stop) {
    const double stopped = *stop;   // waited for with the first loads
    const int rl = L.nx >> 1, pl = rl * L.ny;
    const int p0 = PW * (kb.bx * kb.dx + kb.tx), k = kb.bz, j0 = (kb.by * kb.dy + kb.ty) * 2;
    const bool px = L.bt[0] == IBMDEM_BC_PERIODIC, py = L.bt[2] == IBMDEM_BC_PERIODIC,
               pz = L.bt[4] == IBMDEM_BC_PERIODIC;
    const float ihx2 = float(L.ihx2), ihy2 = float(L.ihy2), ihz2 = float(L.ihz2);
    const float id_int = float(L.idiag[DIAG_INTERIOR]);
    const int pc = min(p0, rl - PW);   // pairs past the row load its last ones and are dropped
    const bool hb = k > 0 || pz, ht = k < L.nz - 1 || pz;
    const int db = hb ? (k > 0 ? -pl : (L.nz - 1) * pl) : 0, dt = ht ? (k < L.nz - 1 ? pl : -(L.nz - 1) * pl) : 0;
    const int cz = diag_count(k, L.nz, L.bt[4], L.bt[5]);
    int pos[2], h[2];
    float a[2][PW], xo[2], ys[2][PW], yn[2][PW], zb[2][PW], zt[2][PW];
    double r[2][PW];
    bool side[2], hs[2], hn[2];
#pragma unroll
    for (int rr = 0; rr < 2; ++rr) {
        const int j = min(j0 + rr, L.ny - 1);
        pos[rr] = (k * L.ny + j) * rl + pc;
        h[rr] = ((j + k) & 1) == color ? 0 : 1;   // the colour's cell of a pair: even or odd
        hs[rr] = j > 0 || py;
        hn[rr] = j < L.ny - 1 || py;
        const float *q = oth + pos[rr];
        ldp<double, PW>(r64 + (long)color * L.half + pos[rr], r[rr]);
        ldp<float, PW>(q, a[rr]);
        // the outer x neighbour: west of the first pair's even cell, east of
        // the last one's odd cell
        const bool w = pc > 0 || px, e = pc + PW < rl || px;
        side[rr] = h[rr] ? e : w;
        xo[rr] = q[h[rr] ? (e ? (pc + PW < rl ? PW : PW - rl) : 0) : (w ? (pc > 0 ? -1 : rl - 1) : 0)];
        ldp<float, PW>(q + db, zb[rr]);
        ldp<float, PW>(q + dt, zt[rr]);
        ldp<float, PW>(q + (hs[rr] ? (j > 0 ? -rl : (L.ny - 1) * rl) : 0), ys[rr]);
        ldp<float, PW>(q + (hn[rr] ? (j < L.ny - 1 ? rl : -(L.ny - 1) * rl) : 0), yn[rr]);
    }
    if (stopped != 0.0) return;
    double dsum = 0.0;
#pragma unroll
    for (int rr = 0; rr < 2; ++rr) {
        const int j = j0 + rr;
        if (j >= L.ny || p0 >= rl) continue;
        const int cyz = diag_count(j, L.ny, L.bt[2], L.bt[3]) * 4 + cz;
        float x[PW];
#pragma unroll
        for (int c = 0; c < PW; ++c) {
            const bool outer = h[rr] ? c == PW - 1 : c == 0;
            const float l = outer ? (side[rr] ? xo[rr] : 0.0f) : a[rr][h[rr] ? (c < PW - 1 ? c + 1 : c) : (c > 0 ? c - 1 : c)];
            const float sx = (a[rr][c] + l) * ihx2;
            const float syy = ((hs[rr] ? ys[rr][c] : 0.0f) + (hn[rr] ? yn[rr][c] : 0.0f)) * ihy2;
            const float szz = ((hb ? zb[rr][c] : 0.0f) + (ht ? zt[rr][c] : 0.0f)) * ihz2;
            const int di = diag_count(2 * (pc + c) + h[rr], L.nx, L.bt[0], L.bt[1]) * 16 + cyz;
            float id = id_int;
            if (di != DIAG_INTERIOR) id = float(L.idiag[di]);
            x[c] = (float(r[rr][c]) + (sx + syy + szz)) * id;
            dsum += r[rr][c] * double(x[c]);
        }
        stp<float, PW>(own + pos[rr], x);
    }
    __shared__ double red[RB];
    const int t = kb.ty * kb.dx + kb.tx;
    dsum = tree_sum<RB>(dsum, t, red);
    if (t == 0) partial[pofs + ((long)kb.bz * kb.gy + kb.by) * kb.gx + kb.bx] = dsum;
}
template <int PW>
__global__ __launch_bounds__(RB) void k_rz_half(LevelDev L, const float *__restrict__ oth, float *__restrict__ own,
                                                int color, const double *__restrict__ r64,
                                                double *__restrict__ partial, long pofs,
                                                const double *__restrict__ stop) {
    rz_half_body<PW>(hw_blk(), L, oth, own, color, r64, partial, pofs, stop);
}

// b_c = (1/8) sum w r_f over the 4x4x4 fine cells of a coarse cell, w =
// wz*wy*wx from (1/4,3/4,3/4,1/4), summed in (z, y, x) order; in FP64 over
// the red cells alone (the black cells' residual is zero). A block owns RS_CX
// x RS_CY coarse cells of one coarse plane and stages the pairs they weigh
// (2 RS_CY + 2 rows of RS_CX + 2 pairs of 4 fine planes, mapped by tile_coord)
// in LDS (33 us from 256^3 in FP64; 51 us over both colours). A row's taps 2I-1 .. 2I+2 are the odd cell of pair I - 1, both
// cells of pair I and the even cell of pair I + 1; at a side that is not
// periodic the tap beyond it is the edge cell again.
constexpr int RS_CX = 32, RS_CY = 8;
constexpr int RS_RX = RS_CX + 2, RS_RY = 2 * RS_CY + 2, RS_ROWS = RS_RY * 4;
static_assert(RS_CX * RS_CY == RB, "one coarse cell per thread");
// the taps of one fine row, in x order. even: the row's red cells are the
// even ones; red(q), black(q): the values of the coarse cell's pair I + q;
// lo, hi: the coarse cell lies at an edge beyond which a tap is clamped
template <typename T, typename V, typename W>
__device__ __forceinline__ T restrict_row(T s, T w, bool even, bool lo, bool hi, const V &red, const W &black) {
    const T w1 = w * T(0.75), w0 = w * T(0.25);
    if (RES_BLACK<T>) {
        const T a = even ? (lo ? red(0) : black(-1)) : (lo ? black(0) : red(-1));
        const T b = even ? red(0) : black(0), c = even ? black(0) : red(0);
        const T d = even ? (hi ? black(0) : red(1)) : (hi ? red(0) : black(1));
        s = s + w0 * a;
        s = s + w1 * b;
        s = s + w1 * c;
        s = s + w0 * d;
    } else if (even) {
        if (lo) s = s + w0 * red(0);             // tap 2I - 1 is cell 0
        s = s + w1 * red(0);
        if (!hi) s = s + w0 * red(1);            // tap 2I + 2
    } else {
        if (!lo) s = s + w0 * red(-1);           // tap 2I - 1
        s = s + w1 * red(0);
        if (hi) s = s + w0 * red(0);             // tap 2I + 2 is the last cell
    }
    return s;
}
template <typename T>
__device__ __forceinline__ void restrict_body(const Blk &kb, const LevelDev &F, const T *__restrict__ rf,
                                              const LevelDev &Cl, T *__restrict__ bc,
                                              const double *__restrict__ stop) {
    const double stopped = *stop;   // waited for with the first loads
    constexpr int NC = RES_BLACK<T> ? 2 : 1;   // colours staged
    __shared__ T tile[NC][RS_ROWS * RS_RX];
    const int t = kb.tx;
    const int I0 = kb.bx * RS_CX, J0 = kb.by * RS_CY, K = kb.bz;
    const int rl = F.nx >> 1;
    const bool px = F.bt[0] == IBMDEM_BC_PERIODIC;
    // half-wavefront h loads pairs I0 .. I0 + 31 of rows h, h + 8, ...; the
    // outer two pairs of every row are one more load of the first threads
    constexpr int NH = RB / 32, RPH = RS_ROWS / NH;
    static_assert(RS_ROWS % NH == 0 && 2 * RS_ROWS <= RB, "row split of the restriction tile");
    auto rowpos = [&](int r) {
        const int k = tile_coord(2 * K - 1 + r / RS_RY, F.nz, F.bt[4], F.bt[5]);
        const int j = tile_coord(2 * J0 - 1 + r % RS_RY, F.ny, F.bt[2], F.bt[3]);
        return (k * F.ny + j) * rl;
    };
    auto pair = [&](int q) {   // a pair beyond the row: wrapped, or unused
        if (q < 0) q = px ? q + rl : 0;
        if (q >= rl) q = px ? q - rl : rl - 1;
        return min(max(q, 0), rl - 1);
    };
    const int lane = t & 31, h = t >> 5;
    T v[NC][RPH], ve[NC];
    const int pc = pair(I0 + lane);
#pragma unroll
    for (int u = 0; u < RPH; ++u) {
        const int o = rowpos(h + NH * u) + pc;
#pragma unroll
        for (int a = 0; a < NC; ++a) v[a][u] = rf[(long)a * F.half + o];
    }
    {
        const int e = min(t, 2 * RS_ROWS - 1), o = rowpos(e >> 1) + pair(e & 1 ? I0 + RS_CX : I0 - 1);
#pragma unroll
        for (int a = 0; a < NC; ++a) ve[a] = rf[(long)a * F.half + o];
    }
    if (stopped != 0.0) return;
#pragma unroll
    for (int a = 0; a < NC; ++a) {
#pragma unroll
        for (int u = 0; u < RPH; ++u) tile[a][(h + NH * u) * RS_RX + 1 + lane] = v[a][u];
        if (t < 2 * RS_ROWS) tile[a][(t >> 1) * RS_RX + (t & 1 ? RS_RX - 1 : 0)] = ve[a];
    }
    __syncthreads();
    const int I = I0 + lane, J = J0 + h;
    if (I >= Cl.nx || J >= Cl.ny) return;
    const T wt[4] = {T(0.25), T(0.75), T(0.75), T(0.25)};
    const bool lo = I == 0 && !px, hi = I == Cl.nx - 1 && !px;
    int par[4];
#pragma unroll
    for (int c2 = 0; c2 < 4; ++c2) par[c2] = tile_coord(2 * J - 1 + c2, F.ny, F.bt[2], F.bt[3]);
    T s = T(0);
#pragma unroll
    for (int c3 = 0; c3 < 4; ++c3) {
        const int k = tile_coord(2 * K - 1 + c3, F.nz, F.bt[4], F.bt[5]);
#pragma unroll
        for (int c2 = 0; c2 < 4; ++c2) {
            const int o = (c3 * RS_RY + 2 * h + c2) * RS_RX + 1 + lane;
            s = restrict_row(s, wt[c3] * wt[c2], ((par[c2] + k) & 1) == 0, lo, hi,
                             [&](int q) { return tile[0][o + q]; }, [&](int q) { return tile[NC - 1][o + q]; });
        }
    }
    bc[lidx(Cl, I, J, K)] = T(0.125) * s;
}
template <typename T>
__global__ __launch_bounds__(RB) void k_restrict(LevelDev F, const T *__restrict__ rf, LevelDev Cl,
                                                 T *__restrict__ bc, const double *__restrict__ stop) {
    restrict_body<T>(hw_blk(), F, rf, Cl, bc, stop);
}

// xout = xin + P x_c on the red cells: 8 parents, weights (3/4 own, 1/4
// neighbour) per dimension. A thread has PW adjacent pairs of one row; the
// block's coarse parents (its pairs' coarse columns +-1, rows +-1, the
// plane's two parent planes) are staged in LDS, column x of a row at (x & 1) *
// (TX / 2) + x / 2: a row's red cells are two apart, so the summing loop's
// lanes read consecutive words. 41 us onto 256^3 in FP64 (51 us for both
// colours, in place).
constexpr int PR_TILE = 1056;   // 2 (by / 2 + 2) (PW bx + 2) for the shapes of shape_for
template <typename T, int PW>
__device__ __forceinline__ void prolong_red_body(const Blk &kb, const LevelDev &F, const T *__restrict__ xin,
                                                 T *__restrict__ xout, const LevelDev &Cl,
                                                 const T *__restrict__ xc, const double *__restrict__ stop) {
    const double stopped = *stop;   // waited for with the first loads
    __shared__ T tile[PR_TILE];
    const int bx = kb.dx, by = kb.dy;
    const int TX = PW * bx + 2, TY = by / 2 + 2, TXH = (TX + 1) / 2;
    const int I0 = PW * kb.bx * bx - 1, J0 = (kb.by * by) / 2 - 1;
    const int k = kb.bz;
    int pk[2];
    parents(k, Cl.nz, Cl.bt[4], Cl.bt[5], pk[0], pk[1]);
    const int t = kb.ty * bx + kb.tx, rl = F.nx >> 1;
    const int p0 = PW * (kb.bx * bx + kb.tx), pc = min(p0, rl - PW);
    const int j = kb.by * by + kb.ty, jc = min(j, F.ny - 1);
    const long pos = (long)(k * F.ny + jc) * rl + pc;
    T x[PW];
    ldp<T, PW>(xin + pos, x);   // in flight while the coarse tile is staged
    const int NROW = 2 * TY, NW = bx * by / 64;
    if (TX >= 64) {
        // wavefront w stages rows w, w + NW, ...: a row's (J, K) are the same
        // on every lane, and a lane maps its columns once
        const int lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
        int Ic[3];
#pragma unroll
        for (int u = 0; u < 3; ++u) Ic[u] = tile_coord(I0 + lane + 64 * u, Cl.nx, Cl.bt[0], Cl.bt[1]);
        for (int r = w; r < NROW; r += NW) {
            const int y = r % TY, c = r / TY;
            const int J = tile_coord(J0 + y, Cl.ny, Cl.bt[2], Cl.bt[3]), K = pk[c];
            T v[3];
#pragma unroll
            for (int u = 0; u < 3; ++u)
                if (lane + 64 * u < TX) v[u] = xc[lidx(Cl, Ic[u], J, K)];
#pragma unroll
            for (int u = 0; u < 3; ++u) {
                const int q = lane + 64 * u;
                if (q < TX) tile[r * 2 * TXH + (q & 1) * TXH + (q >> 1)] = v[u];
            }
        }
    } else {
        const int NT = NROW * TX;
        for (int q0 = t; q0 < NT; q0 += 4 * bx * by) {
            T v[4];
            int dst[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int q = q0 + u * bx * by;
                dst[u] = -1;
                if (q < NT) {
                    const int r = q / TX, xx = q - r * TX, y = r % TY, c = r / TY;
                    const int I = tile_coord(I0 + xx, Cl.nx, Cl.bt[0], Cl.bt[1]);
                    const int J = tile_coord(J0 + y, Cl.ny, Cl.bt[2], Cl.bt[3]);
                    v[u] = xc[lidx(Cl, I, J, pk[c])];
                    dst[u] = r * 2 * TXH + (xx & 1) * TXH + (xx >> 1);
                }
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (dst[u] >= 0) tile[dst[u]] = v[u];
        }
    }
    __syncthreads();
    if (j >= F.ny || p0 >= rl || stopped != 0.0) return;
    const T wt[2] = {T(0.75), T(0.25)};
    const int ty[2] = {j / 2 - J0, j / 2 + ((j & 1) ? 1 : -1) - J0};
    const int odd = (j + k) & 1;   // the row's red cells are the odd ones
#pragma unroll
    for (int c = 0; c < PW; ++c) {
        // pair pc + c is coarse column pc + c; the other parent lies on the
        // red cell's side
        const int a = pc + c - I0, tx[2] = {a, odd ? a + 1 : a - 1};
        const int sx[2] = {(tx[0] & 1) * TXH + (tx[0] >> 1), (tx[1] & 1) * TXH + (tx[1] >> 1)};
        T s = T(0);
#pragma unroll
        for (int c3 = 0; c3 < 2; ++c3)
#pragma unroll
            for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
                for (int c1 = 0; c1 < 2; ++c1)
                    s = s + wt[c3] * wt[c2] * wt[c1] * tile[(c3 * TY + ty[c2]) * 2 * TXH + sx[c1]];
        x[c] = x[c] + s;
    }
    stp<T, PW>(xout + pos, x);
}
template <typename T, int PW>
__global__ __launch_bounds__(RB) void k_prolong_red(LevelDev F, const T *__restrict__ xin, T *__restrict__ xout,
                                                    LevelDev Cl, const T *__restrict__ xc,
                                                    const double *__restrict__ stop) {
    prolong_red_body<T, PW>(hw_blk(), F, xin, xout, Cl, xc, stop);
}
