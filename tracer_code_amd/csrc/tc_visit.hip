// Jacobi-Richardson sweeps of a level visit (iterate_stream,
// iterative_solver.f90:871-912), several per launch, with the correction
// held in registers.
//
// A launch of one sweep reads and writes every plane of the level for 13
// taps of arithmetic, and on all levels but the finest it is nothing but
// latency: k_sweep takes 4.0 us on 16x16 and on 512x256 cells alike.  Here a
// workgroup holds a region of LW columns by NW*(64/LW)*R rows: a wavefront's
// lanes are LW columns of 64/LW row groups, and a lane keeps R rows of its
// column, with their coefficients, in registers for the whole launch.  A
// sweep takes the neighbours along x by DPP wave shifts, those along z from
// the lane's own rows and, past them, from a copy of the region in LDS
// (two copies, alternating, so that a sweep has one barrier).
//
// Tiles: a workgroup owns tx by ty cells of its region; the rest is a halo
// of 2 cells per sweep, which it recomputes.  Where a level fits one region
// (a small level), a workgroup holds all of it, needs no halo, and runs the
// visit's sweeps in one launch.
//
// Walls and ghosts: the correction is zero on the walls (only interior
// points and ghosts are ever written), so cells outside the interior are
// held as zeros with zero coefficients.  A sweep at an interior point reads
// past a wall only at its second neighbour along one axis, which is the
// mirror of the point itself: -S (or zsg*S at the bottom and the top).  The
// 3x3 neighbourhood reaches the walls at most.
#include <algorithm>

#include "tc_kernels.h"

namespace tc {

namespace {

// ---- lane shifts -------------------------------------------------------------
// the value of the previous lane (wave_shr:1) or the next (wave_shl:1); the
// first (last) lane gets 0.  Between the row groups of a wavefront the
// shifts cross from one group's last column to the next group's first: both
// are cells of the halo or a wall (or beyond it), see the tile rule below.
__device__ __forceinline__ double from_left(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(__builtin_amdgcn_mov_dpp(hi, 0x138, 0xF, 0xF, true),
                            __builtin_amdgcn_mov_dpp(lo, 0x138, 0xF, 0xF, true));
}
__device__ __forceinline__ double from_right(double v)
{
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(__builtin_amdgcn_mov_dpp(hi, 0x130, 0xF, 0xF, true),
                            __builtin_amdgcn_mov_dpp(lo, 0x130, 0xF, 0xF, true));
}

// ---- geometry ------------------------------------------------------------------
// The region of tile (X, Y) starts at column 1 + X*tx - hx, row 1 + Y*ty - hz.
// With tiles, hx and hz are at least 2 per sweep, the same beyond the own
// cells on the far side.  hx = 0 (hz = 0): one tile spans the interior along
// that axis; the region then ends at or behind the far wall (LW >= nx), so
// that a shift across the end of a row group meets a wall's zero.
struct VisitTile {
    int tx, ty, hx, hz;
};
struct VisitFactors {
    double v[VISIT_KMAX];  // the sweep's factor; on the ratio level the cosine that its per-point factor takes
};

// The 13 values a sweep at one point reads.
template <typename T>
struct Taps {
    T c, xm1, xp1, xm2, xp2, zm1, zp1, zm2, zp2, mm, pm, mp, pp;
};

// ---- the reference's operator in FP64 ----------------------------------------
// stream_space_g with the second-order tables D1 = (-1/2, 0, 1/2),
// D2 = (1, -2, 1), D3 = (-1/2, 1, 0, -1, 1/2), D4 = (1, -4, 6, -4, 1) put in
// (visit_tables tests for them): the sums run in the same order, products by
// powers of two are exact and become FMAs, those by zero are left out.  The
// results are the same bits (a finite x + 0*S is x), in 64 FP64 instructions
// a point instead of 148.
struct RefCell {
    double vis, vd, vx2, vz2, vxz4, vis2, rhs, dts;
};

// a/d as the division rounds it, from y = 1/d rounded: two corrections by
// the FMA remainder (Markstein's theorem: with y correctly rounded and the
// quotient within an ulp, one more correction rounds correctly).  5
// instructions instead of the division sequence.
__device__ __forceinline__ double div_by(double a, double d, double y)
{
    double q = a * y;
    q = __builtin_fma(__builtin_fma(-d, q, a), y, q);
    return __builtin_fma(__builtin_fma(-d, q, a), y, q);
}
// With spacings that are powers of two (POW2) the quotients are exact
// scalings: they go into the FMA that follows (fma(x, s, y) rounds once, as
// the sum of the scaled x does) or, where the quotient is only multiplied by a
// coefficient, into the coefficient (vxz4, vis2).
template <bool POW2>
struct RefScale;
template <>
struct RefScale<true> {
    static __device__ __forceinline__ double sum(double a, double, double ya, double b, double, double yb)
    {
        return fma(a, ya, b * yb);
    }
    static __device__ __forceinline__ double diff(double a, double, double ya, double b, double, double yb)
    {
        return fma(a, ya, -(b * yb));
    }
    static __device__ __forceinline__ double one(double a, double, double) { return a; }
    static __device__ __forceinline__ double coef(double c, double y) { return c * y; }
};
template <>
struct RefScale<false> {
    static __device__ __forceinline__ double sum(double a, double da, double ya, double b, double db, double yb)
    {
        return div_by(a, da, ya) + div_by(b, db, yb);
    }
    static __device__ __forceinline__ double diff(double a, double da, double ya, double b, double db, double yb)
    {
        return div_by(a, da, ya) - div_by(b, db, yb);
    }
    static __device__ __forceinline__ double one(double a, double d, double y) { return div_by(a, d, y); }
    static __device__ __forceinline__ double coef(double c, double) { return c; }
};

template <bool POW2>
__device__ __forceinline__ double ref_residual(const Taps<double>& t, const RefCell& q, const Spacing& h)
{
    using Sc = RefScale<POW2>;
    const double Srr = fma(-2.0, t.c, t.xm1) + t.xp1;
    const double Sss = fma(-2.0, t.c, t.zm1) + t.zp1;
    const double Srrr = fma(0.5, t.xp2, fma(-0.5, t.xm2, t.xm1) - t.xp1);
    const double Ssss = fma(0.5, t.zp2, fma(-0.5, t.zm2, t.zm1) - t.zp1);
    const double c6 = 6.0 * t.c;
    const double Srrrr = fma(-4.0, t.xp1, fma(-4.0, t.xm1, t.xm2) + c6) + t.xp2;
    const double Sssss = fma(-4.0, t.zp1, fma(-4.0, t.zm1, t.zm2) + c6) + t.zp2;
    const double Srs = fma(0.25, t.pp, fma(-0.25, t.mp, fma(-0.25, t.pm, 0.25 * t.mm)));
    const double Srss = fma(0.5, t.pp, fma(-0.5, t.mp, (fma(0.5, t.pm, -0.5 * t.mm) + t.xm1) - t.xp1));
    const double Srrs = fma(0.5, t.pp, fma(0.5, t.mp, fma(-0.5, t.pm, fma(-0.5, t.mm, t.zm1))) - t.zp1);
    const double Srrss =
        fma(-2.0, t.zp1, fma(-2.0, t.xp1, fma(4.0, t.c, fma(-2.0, t.xm1, fma(-2.0, t.zm1, t.mm) + t.pm))) + t.mp) + t.pp;
    const double t1 = q.vd * Sc::diff(Srr, h.dr2, h.idr2, Sss, h.ds2, h.ids2);
    const double t2 = q.vis * Sc::sum(Srrrr, h.dr4, h.idr4, Sssss, h.ds4, h.ids4);
    const double t3 = q.vis2 * Sc::one(Srrss, h.dr2ds2, h.idr2ds2);
    const double t4 = q.vxz4 * Sc::one(Srs, h.drds, h.idrds);
    const double t5 = q.vx2 * Sc::sum(Srrr, h.dr3, h.idr3, Srss, h.drds2, h.idrds2);
    const double t6 = q.vz2 * Sc::sum(Ssss, h.ds3, h.ids3, Srrs, h.dr2ds, h.idr2ds);
    const double ss = t1 + t2 + t3 + t4 + t5 + t6 - q.rhs;
    return -ss;
}

struct RefArgs {
    const double *vis, *vx, *vz, *vxx, *vzz, *vxz, *rhs, *dts, *ratio;
};

// Bound: FP64 arithmetic and one barrier a sweep (a region of 32x32 cells: 4
// rows of 64 cells per SIMD, about 85 instructions of 4 cycles each, 0.65 us
// with the barrier), plus 2.5 to 3 us for the launch and the loads of 9
// planes, which the launch's sweeps share.  On the levels that do not fit
// the L2s (1024x512 and up) the loads: 72 B per staged cell.
// RES (one tile holds the level): the residual of the result goes to R.
template <bool POW2, bool RATIO, int LW, int R, int NW, bool RES>
__global__ __launch_bounds__(NW * 64) void k_visit_ref(const double* __restrict__ Ein, double* __restrict__ Eout,
                                                       RefArgs A, Grid g, Spacing h, VisitTile vt, VisitFactors sf,
                                                       int nk, double zsg, double* __restrict__ Rout)
{
    constexpr int GR = 64 / LW, ROWS = NW * GR * R;
    __shared__ double buf[2][ROWS * LW];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane % LW, row0 = (wv * GR + lane / LW) * R;  // this lane's column and first row in the region
    const int2 tile = xcd_tile();
    const int i = 1 + tile.x * vt.tx - vt.hx + li, k0 = 1 + tile.y * vt.ty - vt.hz + row0;
    const bool col = i >= 1 && i <= g.nx - 1;
    double S[R];
    RefCell q[R];
    double lb[RATIO ? R : 1];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool in = col && k0 + r >= 1 && k0 + r <= g.nz - 1;
        const size_t c = g.at(in ? i : 1, in ? k0 + r : 1);
        S[r] = Ein ? Ein[c] : 0.0;
        const double vis = A.vis[c], vx = A.vx[c], vz = A.vz[c], vxx = A.vxx[c], vzz = A.vzz[c], vxz = A.vxz[c];
        const double rhs = A.rhs[c], dts = A.dts[c];
        if (!in) S[r] = 0.0;
        q[r].vis = in ? vis : 0.0;
        q[r].vd = in ? vxx - vzz : 0.0;
        q[r].vx2 = in ? 2.0 * vx : 0.0;
        q[r].vz2 = in ? 2.0 * vz : 0.0;
        q[r].vxz4 = in ? RefScale<POW2>::coef(4.0 * vxz, h.idrds) : 0.0;
        q[r].vis2 = in ? RefScale<POW2>::coef(2.0 * vis, h.idr2ds2) : 0.0;
        q[r].rhs = in ? rhs : 0.0;
        q[r].dts = in ? dts : 0.0;
        if constexpr (RATIO) {
            const double a = A.ratio[c];
            lb[r] = (!in || a > 1e99) ? -2.0 : -2.0 * (a * a) / (1.0 + a * a);
        }
    }
    const bool wl = i == 1, wr = i == g.nx - 1;
    // the region holds a side wall's neighbours (uniform)
    const int i0 = 1 + tile.x * vt.tx - vt.hx;
    const bool sides = i0 <= 1 || i0 + LW > g.nx - 1;
    // the rows of the wavefront, and those whose result counts after the last sweep
    const int w0 = wv * GR * R, w1 = w0 + GR * R - 1;
    const int kg = 1 + tile.y * vt.ty - vt.hz;
    const int own0 = vt.hz, own1 = vt.hz + vt.ty - 1;
    auto taps = [&](const double* __restrict__ b, int r, const double (&v)[R + 4], const double (&lf)[R + 2],
                    const double (&rt)[R + 2]) {
        Taps<double> t;
        t.c = v[r + 2];
        t.zm1 = v[r + 1]; t.zp1 = v[r + 3]; t.zm2 = v[r]; t.zp2 = v[r + 4];
        t.xm1 = lf[r + 1]; t.xp1 = rt[r + 1];
        t.mm = lf[r]; t.pm = rt[r]; t.mp = lf[r + 2]; t.pp = rt[r + 2];
        t.xm2 = from_left(t.xm1); t.xp2 = from_right(t.xp1);
        if (sides) {
            t.xm2 = wl ? -t.c : t.xm2;
            t.xp2 = wr ? -t.c : t.xp2;
        }
        if (k0 + r == 1) t.zm2 = zsg * t.c;
        if (k0 + r == g.nz - 1) t.zp2 = zsg * t.c;
        (void)b;
        return t;
    };
    // the rows -2..R+1 around the lane's own, and their neighbours along x
    auto gather = [&](const double* __restrict__ b, double (&v)[R + 4], double (&lf)[R + 2], double (&rt)[R + 2]) {
        const int up = row0 * LW + li;
        v[0] = row0 >= 2 ? b[up - 2 * LW] : 0.0;
        v[1] = row0 >= 1 ? b[up - LW] : 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r + 2] = S[r];
        v[R + 2] = row0 + R < ROWS ? b[up + R * LW] : 0.0;
        v[R + 3] = row0 + R + 1 < ROWS ? b[up + (R + 1) * LW] : 0.0;
#pragma unroll
        for (int r = 0; r < R + 2; ++r) {
            lf[r] = from_left(v[r + 1]);
            rt[r] = from_right(v[r + 1]);
        }
    };
#pragma unroll 1
    for (int s = 0; s < nk; ++s) {
        double* __restrict__ b = buf[s & 1];
#pragma unroll
        for (int r = 0; r < R; ++r) b[(row0 + r) * LW + li] = S[r];
        __syncthreads();
        // rows that the own cells still depend on, inside the interior (the
        // whole wavefront skips the sweep otherwise)
        const int ext = 2 * (nk - 1 - s) + (RES ? 2 : 0);
        const int lo = max(own0 - ext, 1 - kg), hi = min(own1 + ext, g.nz - 1 - kg);
        if (w1 < lo || w0 > hi) continue;
        double v[R + 4], lf[R + 2], rt[R + 2], n[R];
        gather(b, v, lf, rt);
        const double f = sf.v[s];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const Taps<double> t = taps(b, r, v, lf, rt);
            double cc = f;
            if constexpr (RATIO) cc = 2.0 / (-lb[r] + 1.0 + (lb[r] + 1.0) * f);
            n[r] = S[r] + cc * q[r].dts * ref_residual<POW2>(t, q[r], h);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) S[r] = n[r];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int rr = row0 + r, k = k0 + r;
        if (li >= vt.hx && li < vt.hx + vt.tx && rr >= vt.hz && rr < vt.hz + vt.ty && col && k >= 1 && k <= g.nz - 1) {
            Eout[g.at(i, k)] = S[r];
            stream_ghosts(Eout, g, i, k, S[r], zsg);
        }
    }
    if constexpr (RES) {
        double* __restrict__ b = buf[nk & 1];
#pragma unroll
        for (int r = 0; r < R; ++r) b[(row0 + r) * LW + li] = S[r];
        __syncthreads();
        double v[R + 4], lf[R + 2], rt[R + 2];
        gather(b, v, lf, rt);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const Taps<double> t = taps(b, r, v, lf, rt);
            const double res = ref_residual<POW2>(t, q[r], h);
            if (col && k0 + r >= 1 && k0 + r <= g.nz - 1) Rout[g.at(i, k0 + r)] = res;
        }
    }
}

template <bool POW2, int LW, int R, int NW, bool RES>
void visit_ref_launch(hipStream_t st, bool ratio, dim3 gr, const double* in, double* out, const RefArgs& A,
                      const Grid& g, const Spacing& h, const VisitTile& vt, const VisitFactors& sf, int nk, double zsg,
                      double* res)
{
    if (ratio)
        hipLaunchKernelGGL((k_visit_ref<POW2, true, LW, R, NW, RES>), gr, dim3(NW * 64), 0, st, in, out, A, g, h, vt, sf,
                           nk, zsg, res);
    else
        hipLaunchKernelGGL((k_visit_ref<POW2, false, LW, R, NW, RES>), gr, dim3(NW * 64), 0, st, in, out, A, g, h, vt,
                           sf, nk, zsg, res);
}

// one tile holds the interior: no halo
VisitTile whole_tile(const Grid& g) { return VisitTile{g.nx - 1, g.nz - 1, 0, 0}; }

// tiles of a region of w by r cells for nk sweeps; an axis that the region
// spans needs no halo
VisitTile tiles_for(const Grid& g, int w, int r, int nk)
{
    VisitTile t = whole_tile(g);
    if (g.nx > w) { t.hx = 2 * nk; t.tx = w - 4 * nk; }
    if (g.nz - 1 > r) { t.hz = 2 * nk; t.ty = r - 4 * nk; }
    return t;
}
dim3 tile_grid(const Grid& g, const VisitTile& t)
{
    return dim3((unsigned)((g.nx - 1 + t.tx - 1) / t.tx), (unsigned)((g.nz - 1 + t.ty - 1) / t.ty));
}

}  // namespace

// Whether the FD tables are the second-order ones that the kernels of this
// file have built in (config.fd_coefficients(2), main.f90:350-469).
bool visit_tables(const FD& F)
{
    static const double d1[3] = {-0.5, 0.0, 0.5}, d2[3] = {1.0, -2.0, 1.0};
    static const double d3[5] = {-0.5, 1.0, 0.0, -1.0, 0.5}, d4[5] = {1.0, -4.0, 6.0, -4.0, 1.0};
    for (int j = 0; j < 3; ++j)
        if (F.D1[j + 1] != d1[j] || F.D2[j + 1] != d2[j]) return false;
    for (int j = 0; j < 5; ++j)
        if (F.D3[j] != d3[j] || F.D4[j] != d4[j]) return false;
    return true;
}

// The regions of visit_plan_ref: columns, rows.
//   0: 16x16 (4 waves of 4 row groups, 1 row a lane)
//   1: 32x32 (8 waves of 2 row groups, 2 rows)
//   2: 32x32 (16 waves of 2 row groups, 1 row)
//   3: 64x32 (8 waves, 4 rows)
struct VisitRegion {
    int w, r;
};
static constexpr VisitRegion VISIT_REGIONS[4] = {{16, 16}, {32, 32}, {32, 32}, {64, 32}};

// Measured, us a sweep (one sweep per launch: 4.0 up to 512x256 cells, 8.9 at
// 1024x512, 25.0 at 2048x1024; spacings that are powers of two, then others):
//   a level that region 0 or 1 holds runs all its sweeps in one launch:
//     16x16 0.41 / 0.46, 32x32 0.84 / 1.17 (tiles of region 0: 1.27 / 1.34);
//     one workgroup for 64x32 cells would take 1.40, tiles take 1.33;
//   else tiles of region 2 with as many sweeps a launch as leave at most one
//     tile per CU: 64x64 1.06 (7 sweeps, 256 tiles; 6: 1.13, 4: 1.5),
//     128x64 1.14 (6), 256x128 1.35 (5; region 1: 1.50), 304x176 - / 1.77
//     (4); up to two tiles per CU with 4 sweeps: 512x256 2.16 (region 3: 2.6);
//   else region 3, 4 sweeps: less halo, two workgroups per CU whose loads and
//     arithmetic overlap: 1024x512 5.5 (64x64 regions, one per CU: 5.9),
//     2048x1024 16.4 (19.0).
VisitPlan visit_plan_ref(const Grid& g, int cus)
{
    VisitPlan p;
    for (int c = 0; c < 2; ++c)
        if (g.nx <= VISIT_REGIONS[c].w && g.nz - 1 <= VISIT_REGIONS[c].r) {
            p.cfg = c;
            p.k = VISIT_KMAX;
            p.whole = true;
            return p;
        }
    auto tiles = [&](int k) {
        const dim3 t = tile_grid(g, tiles_for(g, VISIT_REGIONS[2].w, VISIT_REGIONS[2].r, k));
        return (long)t.x * t.y;
    };
    p.cfg = 2;
    for (p.k = 7; p.k > 4; --p.k)
        if (tiles(p.k) <= cus) return p;
    if (tiles(4) > 2L * cus) p.cfg = 3;
    return p;
}

void launch_visit_ref(hipStream_t st, const VisitPlan& p, bool pow2, bool use_ratio, const Level& L, const double* rhs,
                      const double* in, double* out, const Spacing& h, const double* fac, int nk, double zsg,
                      double* res)
{
    const RefArgs A{L.vis, L.visx, L.visz, L.visxx, L.viszz, L.visxz, rhs, L.dtstream, L.ratio};
    VisitFactors sf;
    for (int s = 0; s < nk; ++s) sf.v[s] = fac[s];
    const VisitRegion rg = VISIT_REGIONS[p.cfg];
    const VisitTile vt = p.whole ? whole_tile(L.g) : tiles_for(L.g, rg.w, rg.r, nk);
    const dim3 gr = tile_grid(L.g, vt);
    auto go = [&](auto pw) {
        constexpr bool P = decltype(pw)::value;
        if (res) {
            if (p.cfg == 0) visit_ref_launch<P, 16, 1, 4, true>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, res);
            else visit_ref_launch<P, 32, 2, 8, true>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, res);
            return;
        }
        switch (p.cfg) {
        case 0: visit_ref_launch<P, 16, 1, 4, false>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, nullptr); break;
        case 1: visit_ref_launch<P, 32, 2, 8, false>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, nullptr); break;
        case 2: visit_ref_launch<P, 32, 1, 16, false>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, nullptr); break;
        default: visit_ref_launch<P, 64, 4, 8, false>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, nullptr); break;
        }
    };
    if (pow2) go(std::integral_constant<bool, true>{});
    else go(std::integral_constant<bool, false>{});
}

}  // namespace tc
