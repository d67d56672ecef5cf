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
#include "tc_stencil32.h"

namespace tc {

namespace {

// ---- lane shifts -------------------------------------------------------------
// Between the row groups of a wavefront from_left and from_right cross from one
// group's last column to the next group's first: both are cells of the halo or
// a wall (or beyond it), see the tile rule below.

// ---- geometry ------------------------------------------------------------------
// The region of tile (X, Y) starts at column 1 + X*tx - hx, row 1 + Y*ty - hz.
// With tiles, hx and hz are at least 2 per sweep, the same beyond the own
// cells on the far side.  hx = 0 (hz = 0): one tile spans the interior along
// that axis; the region then ends at or behind the far wall (LW >= nx), so
// that a shift across the end of a row group meets a wall's zero.
struct VisitTile {
    int tx, ty, hx, hz;
};
template <typename T>
struct VisitFac {
    T v[VISIT_KMAX];  // the sweep's factor; on the ratio level the cosine that its per-point factor takes
};
using VisitFactors = VisitFac<double>;

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
    const double *vis, *vx, *vz, *vxx, *vzz, *vxz;
    double* rhs;
    const double *dts, *ratio;
};

// Bound: VALU issue and one barrier a sweep (a region of 32x32 cells: 4
// rows of 64 cells per SIMD, about 85 instructions of 4 cycles each, 0.65 us
// with the barrier), plus 2.5 to 3 us for the launch and the loads of 9
// planes, which the launch's sweeps share.  By counters, issue fills 71% of a
// launch that holds 32x32 cells (35% at 16x16, one wave a SIMD: there the chain
// of LDS round trip, barrier and FMAs is longer), 29 to 48% of the tiles of
// region 2 and 46 to 58% of region 3's, which move 2.1 to 3.0 TB/s beside it
// (72 B per staged cell).
// RES (one tile holds the level): the residual of the result goes to R.
template <bool POW2, bool RATIO, int LW, int R, int NW, bool RES>
__global__ __launch_bounds__(NW * 64) void k_visit_ref(const double* __restrict__ Ein, double* __restrict__ Eout,
                                                       RefArgs A, Grid g, Spacing h, VisitTile vt, VisitFactors sf,
                                                       int nk, double zsg, double* __restrict__ Rout, VisitStart vs)
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
        const double dts = A.dts[c];
        double rhs;
        if (vs.resf) {
            rhs = restrict_at(vs.resf, vs.gf, in ? i : 1, in ? k0 + r : 1);
            const int rr = row0 + r;
            if (in && li >= vt.hx && li < vt.hx + vt.tx && rr >= vt.hz && rr < vt.hz + vt.ty) A.rhs[c] = rhs;
        } else {
            rhs = A.rhs[c];
        }
        if (vs.Ec) S[r] = S[r] + prolong_at(vs.Ec, vs.gc, in ? i : 1, in ? k0 + r : 1);
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
    auto taps = [&](int r, const double (&v)[R + 4], const double (&lf)[R + 2], const double (&rt)[R + 2]) {
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
            const Taps<double> t = taps(r, v, lf, rt);
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
            const Taps<double> t = taps(r, v, lf, rt);
            const double res = ref_residual<POW2>(t, q[r], h);
            if (col && k0 + r >= 1 && k0 + r <= g.nz - 1) Rout[g.at(i, k0 + r)] = res;
        }
    }
}

template <bool POW2, int LW, int R, int NW, bool RES>
void visit_ref_launch(hipStream_t st, bool ratio, dim3 gr, const double* in, double* out, const RefArgs& A,
                      const Grid& g, const Spacing& h, const VisitTile& vt, const VisitFactors& sf, int nk, double zsg,
                      double* res, const VisitStart& vs)
{
    if (ratio)
        hipLaunchKernelGGL((k_visit_ref<POW2, true, LW, R, NW, RES>), gr, dim3(NW * 64), 0, st, in, out, A, g, h, vt, sf,
                           nk, zsg, res, vs);
    else
        hipLaunchKernelGGL((k_visit_ref<POW2, false, LW, R, NW, RES>), gr, dim3(NW * 64), 0, st, in, out, A, g, h, vt,
                           sf, nk, zsg, res, vs);
}

// ---- the 13-tap operator of the defect-correction cycles ---------------------
// The dt-scaled weights of the 13 taps of one point with the second-order
// tables put in, from the five coefficients (42 operations, once per launch),
// and the scaled right-hand side.
template <typename T>
struct Cell13 {
    T c, xm1, xp1, xm2, xp2, zm1, zp1, zm2, zp2, mm, pm, mp, pp, rd;
};
template <typename T>
struct H13 {
    T idr2, ids2, idr3, ids3, idr4, ids4, idrds, idrds2, idr2ds, idr2ds2;
};
template <typename T>
struct Args13 {
    const T *vis, *vx, *vz, *a1, *vxx, *vzz, *vxz;
    T* rhs;
    const T *dts, *lb;  // FP32: a1, lb; FP64: vxx, vzz, lb = the ratio
};
// the next level's right-hand side, formed after the last sweep (FP32); RowB
// and bout: for the coarsest level, the coarse solve's equilibrated
// right-hand side too
struct End13 {
    float* out;
    Grid go;
    const double* RowB;
    double* bout;
    H32 h;
};
struct Prolong13 {
    const float* Ec;
    Grid gc;
};
// what the first launch of a visit does before its sweeps: FP32 the
// prolongation, FP64 that or the restriction (VisitStart)
template <typename T>
using Start13 = std::conditional_t<sizeof(T) == 4, Prolong13, VisitStart>;

template <typename T>
__device__ __forceinline__ Cell13<T> weights13(T vis, T vx, T vz, T a1, T vxz, T dts, T rhs, const H13<T>& h)
{
    const T e = dts * vis, b = T(2) * dts * vx, c = T(2) * dts * vz, a = dts * a1, xq = dts * vxz * h.idrds;
    const T e4x = e * h.idr4, e4z = e * h.ids4, et = T(2) * e * h.idr2ds2;
    const T b3 = b * h.idr3, bp = b * h.idrds2, c3 = c * h.ids3, cr = c * h.idr2ds;
    const T ax = a * h.idr2, az = a * h.ids2;
    Cell13<T> w;
    w.xm2 = fma(T(-0.5), b3, e4x);
    w.xp2 = fma(T(0.5), b3, e4x);
    w.zm2 = fma(T(-0.5), c3, e4z);
    w.zp2 = fma(T(0.5), c3, e4z);
    const T mx = fma(T(-2), et, fma(T(-4), e4x, ax)), bx = b3 + bp;
    w.xm1 = mx + bx;
    w.xp1 = mx - bx;
    const T mz = fma(T(-2), et, fma(T(-4), e4z, -az)), cz = c3 + cr;
    w.zm1 = mz + cz;
    w.zp1 = mz - cz;
    w.c = fma(T(4), et, fma(T(6), e4x + e4z, T(2) * (az - ax)));
    const T d1 = et + xq, d2 = et - xq, s1 = T(0.5) * (bp + cr), s2 = T(0.5) * (bp - cr);
    w.mm = d1 - s1;
    w.pp = d1 + s1;
    w.pm = d2 + s2;
    w.mp = d2 - s2;
    w.rd = dts * rhs;
    return w;
}

// the same for any tables
template <typename T>
struct Tables13 {
    T D1[5], D2[5], D3[5], D4[5];
};
struct NoTables {};
template <typename T>
__device__ __forceinline__ Cell13<T> weights13_any(const Tables13<T>& F, T vis, T vx, T vz, T a1, T vxz, T dts, T rhs,
                                                   const H13<T>& h)
{
    T v[13];
    tap_weights<T>(F, h, vis, vx, vz, a1, vxz, v);
    return Cell13<T>{dts * v[0], dts * v[1], dts * v[2], dts * v[3],  dts * v[4],  dts * v[5],  dts * v[6],
                     dts * v[7], dts * v[8], dts * v[9], dts * v[10], dts * v[11], dts * v[12], dts * rhs};
}

// 1/x of the per-point factor (1 <= x <= 5): the hardware's reciprocal with a
// Newton step, which rounds to within an ulp of the quotient
__device__ __forceinline__ float recip(float x)
{
    const float r = __builtin_amdgcn_rcpf(x);
    return fma(fma(-x, r, 1.0f), r, r);
}
__device__ __forceinline__ double recip(double x) { return 1.0 / x; }

// dts (rhs - L(S)): three chains of FMAs
template <typename T>
__device__ __forceinline__ T step13(const Taps<T>& t, const Cell13<T>& w)
{
    T a = fma(-w.c, t.c, w.rd);
    T b = -w.xm1 * t.xm1;
    T d = -w.mm * t.mm;
    a = fma(-w.zm1, t.zm1, a);
    b = fma(-w.xp1, t.xp1, b);
    d = fma(-w.pm, t.pm, d);
    a = fma(-w.zp1, t.zp1, a);
    b = fma(-w.xm2, t.xm2, b);
    d = fma(-w.mp, t.mp, d);
    a = fma(-w.zm2, t.zm2, a);
    b = fma(-w.xp2, t.xp2, b);
    d = fma(-w.pp, t.pp, d);
    a = fma(-w.zp2, t.zp2, a);
    return a + (b + d);
}

// Bound: the launch and the loads (3.4 us with a 32x32 region of one row a
// lane, of which 256 fit the chip), then 0.2 us a sweep (about 25
// instructions a point and the barrier).  By counters, VALU issue fills 25 to
// 34% of such launches and 63 to 75% of those that hold a level of 64 columns;
// on the levels of more tiles 52 to 71%, beside loads of 32 B per staged cell
// (FP32, 1.9 to 3.4 TB/s).
// END: after the last sweep, FP32: the residual in FP64 of the held cells and
// its restriction to the next level (residual32_std, restrict_fw32: the
// values of k_residual_restrict32), for which the region reaches 2 cells
// before and 3 behind the own ones.
// TAB: NoTables for the second-order tables, else the tables.
template <typename T, bool RATIO, int LW, int R, int NW, bool END, typename TAB = NoTables>
__global__ __launch_bounds__(NW * 64) void k_visit13(const T* __restrict__ Ein, T* __restrict__ Eout, Args13<T> A,
                                                     Grid g, H13<T> h, VisitTile vt, VisitFac<T> sf, int nk, T zsg,
                                                     Start13<T> pr, End13 en, TAB tab)
{
    constexpr int GR = 64 / LW, ROWS = NW * GR * R;
    __shared__ T buf[2][ROWS * LW];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane % LW, row0 = (wv * GR + lane / LW) * R;
    const int2 tile = xcd_tile();
    const int i0 = 1 + tile.x * vt.tx - vt.hx, kg = 1 + tile.y * vt.ty - vt.hz;  // the region's origin
    const int i = i0 + li, k0 = kg + row0;
    const bool col = i >= 1 && i <= g.nx - 1;
    T S[R];
    Cell13<T> q[R];
    T lb[RATIO ? R : 1];
    float rc[END ? R : 1][6];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int k = k0 + r;
        const bool in = col && k >= 1 && k <= g.nz - 1;
        const size_t c = g.at(in ? i : 1, in ? k : 1);
        S[r] = Ein ? Ein[c] : T(0);
        const T vis = A.vis[c], vx = A.vx[c], vz = A.vz[c], vxz = A.vxz[c], dts = A.dts[c];
        T rhs;
        if constexpr (sizeof(T) == 8) {
            if (pr.resf) {
                rhs = restrict_at(pr.resf, pr.gf, in ? i : 1, in ? k : 1);
                const int rr = row0 + r;
                if (in && li >= vt.hx && li < vt.hx + vt.tx && rr >= vt.hz && rr < vt.hz + vt.ty) A.rhs[c] = rhs;
            } else {
                rhs = A.rhs[c];
            }
            if (pr.Ec) S[r] = S[r] + prolong_at(pr.Ec, pr.gc, in ? i : 1, in ? k : 1);
        } else {
            rhs = A.rhs[c];
        }
        T a1;
        if constexpr (sizeof(T) == 4) a1 = A.a1[c];
        else a1 = A.vxx[c] - A.vzz[c];
        if constexpr (sizeof(T) == 4) {
            // the coarse correction prolonged into this level (prolong_add32, its
            // four sources loaded by every thread and the parity's value selected)
            if (pr.Ec) {
                const int pi = in ? i : 1, pk = in ? k : 1;
                const int c0 = pi >> 1, c1 = (pi + 1) >> 1, d0 = pk >> 1, d1 = (pk + 1) >> 1;
                const float e00 = pr.Ec[pr.gc.at(c0, d0)], e10 = pr.Ec[pr.gc.at(c1, d0)];
                const float e11 = pr.Ec[pr.gc.at(c1, d1)], e01 = pr.Ec[pr.gc.at(c0, d1)];
                const bool ie = (pi & 1) == 0, ke = (pk & 1) == 0;
                const float two = __fmul_rn(__fadd_rn(e00, ie ? e01 : e10), 0.5f);
                const float four = __fmul_rn(__fadd_rn(__fadd_rn(__fadd_rn(e00, e10), e11), e01), 0.25f);
                S[r] = __fadd_rn(S[r], (ie && ke) ? e00 : ((ie || ke) ? two : four));
            }
        }
        if (!in) S[r] = T(0);
        if constexpr (std::is_same_v<TAB, NoTables>) q[r] = weights13<T>(vis, vx, vz, a1, vxz, in ? dts : T(0), rhs, h);
        else q[r] = weights13_any<T>(tab, vis, vx, vz, a1, vxz, in ? dts : T(0), rhs, h);
        if constexpr (END) { rc[r][0] = vis; rc[r][1] = vx; rc[r][2] = vz; rc[r][3] = a1; rc[r][4] = vxz; rc[r][5] = rhs; }
        if constexpr (RATIO) {
            if constexpr (sizeof(T) == 4) {
                lb[r] = in ? A.lb[c] : T(-2);
            } else {
                const T a = A.lb[c];
                lb[r] = (!in || a > T(1e99)) ? T(-2) : T(-2) * (a * a) / (T(1) + a * a);
            }
        }
    }
    const bool wl = i == 1, wr = i == g.nx - 1;
    const bool sides = i0 <= 1 || i0 + LW > g.nx - 1;
    const int w0 = wv * GR * R, w1 = w0 + GR * R - 1;
    auto gather = [&](const T* __restrict__ b, T (&v)[R + 4], T (&lf)[R + 2], T (&rt)[R + 2]) {
        const int up = row0 * LW + li;
        v[0] = row0 >= 2 ? b[up - 2 * LW] : T(0);
        v[1] = row0 >= 1 ? b[up - LW] : T(0);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r + 2] = S[r];
        v[R + 2] = row0 + R < ROWS ? b[up + R * LW] : T(0);
        v[R + 3] = row0 + R + 1 < ROWS ? b[up + (R + 1) * LW] : T(0);
#pragma unroll
        for (int r = 0; r < R + 2; ++r) {
            lf[r] = from_left(v[r + 1]);
            rt[r] = from_right(v[r + 1]);
        }
    };
    auto taps = [&](int r, const T (&v)[R + 4], const T (&lf)[R + 2], const T (&rt)[R + 2]) {
        Taps<T> t;
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
        return t;
    };
#pragma unroll 1
    for (int s = 0; s < nk; ++s) {
        T* __restrict__ b = buf[s & 1];
#pragma unroll
        for (int r = 0; r < R; ++r) b[(row0 + r) * LW + li] = S[r];
        __syncthreads();
        const int ext = 2 * (nk - 1 - s);
        const int lo = max(vt.hz - ext - (END ? 2 : 0), 1 - kg);
        const int hi = min(vt.hz + vt.ty - 1 + ext + (END ? 3 : 0), g.nz - 1 - kg);
        if (w1 < lo || w0 > hi) continue;
        T v[R + 4], lf[R + 2], rt[R + 2];
        gather(b, v, lf, rt);
        const T f = sf.v[s];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            T cc = f;
            if constexpr (RATIO) cc = T(2) * recip(-lb[r] + T(1) + (lb[r] + T(1)) * f);
            S[r] = fma(cc, step13(taps(r, v, lf, rt), q[r]), S[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int rr = row0 + r, k = k0 + r;
        if (li >= vt.hx && li < vt.hx + vt.tx && rr >= vt.hz && rr < vt.hz + vt.ty && col && k >= 1 && k <= g.nz - 1) {
            Eout[g.at(i, k)] = S[r];
            stream_ghosts(Eout, g, i, k, S[r], zsg);
        }
    }
    if constexpr (END) {
        T* __restrict__ b = buf[nk & 1];
#pragma unroll
        for (int r = 0; r < R; ++r) b[(row0 + r) * LW + li] = S[r];
        __syncthreads();
        T v[R + 4], lf[R + 2], rt[R + 2];
        gather(b, v, lf, rt);
        float* __restrict__ res = reinterpret_cast<float*>(buf[1 - (nk & 1)]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const Taps<T> t = taps(r, v, lf, rt);
            const Tap13d d{t.c, t.xm1, t.xp1, t.xm2, t.xp2, t.zm1, t.zp1, t.zm2, t.zp2, t.mm, t.pm, t.mp, t.pp};
            res[(row0 + r) * LW + li] =
                residual32_std(d, en.h, rc[r][0], rc[r][1], rc[r][2], rc[r][3], rc[r][4], rc[r][5]);
        }
        __syncthreads();
        const int ncx = vt.tx / 2, ncz = vt.ty / 2;
        for (int e = threadIdx.x; e < ncx * ncz; e += NW * 64) {
            const int ic = tile.x * ncx + 1 + e % ncx, kc = tile.y * ncz + 1 + e / ncx;
            if (ic > en.go.nx - 1 || kc > en.go.nz - 1) continue;
            const int p = (2 * kc - kg) * LW + 2 * ic - i0;  // the fine centre
            const float x = restrict_fw32(res[p - LW - 1], res[p + LW - 1], res[p + LW + 1], res[p - 1], res[p - LW],
                                          res[p + 1], res[p + LW], res[p]);
            en.out[en.go.at(ic, kc)] = x;
            if (en.bout) {
                const int u = ic * (en.go.nz + 1) + kc;
                en.bout[u] = (double)x * en.RowB[u];
            }
        }
    }
}

// one tile holds the interior: no halo
VisitTile whole_tile(const Grid& g) { return VisitTile{g.nx - 1, g.nz - 1, 0, 0}; }

// tiles of a region of w by r cells for nk sweeps; an axis that the region
// spans needs no halo.  end: room for the residual and its restriction (an
// even number of own cells, so that a coarse point's centre is its tile's)
VisitTile tiles_for(const Grid& g, int w, int r, int nk, bool end = false)
{
    VisitTile t = whole_tile(g);
    const int lo = 2 * nk + (end ? 2 : 0), hi = 2 * nk + (end ? 3 : 0);
    if (g.nx > w) { t.hx = lo; t.tx = w - lo - hi; if (end) t.tx &= ~1; }
    if (g.nz - 1 > r) { t.hz = lo; t.ty = r - lo - hi; if (end) t.ty &= ~1; }
    return t;
}
dim3 tile_grid(const Grid& g, const VisitTile& t)
{
    return dim3((unsigned)((g.nx - 1 + t.tx - 1) / t.tx), (unsigned)((g.nz - 1 + t.ty - 1) / t.ty));
}

}  // namespace

// Whether the FD tables are the second-order ones that k_visit_ref and
// k_visit13's weights have built in (config.fd_coefficients(2), main.f90:350-469).
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
                      double* res, const VisitStart& vs)
{
    // (the plane is written only where vs asks for the restriction)
    const RefArgs A{L.vis, L.visx, L.visz, L.visxx, L.viszz, L.visxz, const_cast<double*>(rhs), L.dtstream, L.ratio};
    VisitFactors sf;
    for (int s = 0; s < nk; ++s) sf.v[s] = fac[s];
    const VisitRegion rg = VISIT_REGIONS[p.cfg];
    const VisitTile vt = p.whole ? whole_tile(L.g) : tiles_for(L.g, rg.w, rg.r, nk);
    const dim3 gr = tile_grid(L.g, vt);
    auto go = [&](auto pw) {
        constexpr bool P = decltype(pw)::value;
        if (res) {
            if (p.cfg == 0) visit_ref_launch<P, 16, 1, 4, true>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, res, vs);
            else visit_ref_launch<P, 32, 2, 8, true>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, res, vs);
            return;
        }
        switch (p.cfg) {
        case 0: visit_ref_launch<P, 16, 1, 4, false>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, nullptr, vs); break;
        case 1: visit_ref_launch<P, 32, 2, 8, false>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, nullptr, vs); break;
        case 2: visit_ref_launch<P, 32, 1, 16, false>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, nullptr, vs); break;
        default: visit_ref_launch<P, 64, 4, 8, false>(st, use_ratio, gr, in, out, A, L.g, h, vt, sf, nk, zsg, nullptr, vs); break;
        }
    };
    if (pow2) go(std::integral_constant<bool, true>{});
    else go(std::integral_constant<bool, false>{});
}

// ---- plans of the 13-tap sweeps ---------------------------------------------------
// The regions: columns, rows; the last three take tiles.
//   0: 16x16 (4 waves of 4 row groups, 1 row a lane)     whole levels
//   4: 64x16 (16 waves, 1 row)                            whole levels
//   1: 64x32 (16 waves, 2 rows)                           whole levels, tiles
//   2: 32x32 (16 waves of 2 row groups, 1 row)            whole levels, tiles
//   3: 64x32 (8 waves, 4 rows), FP32; 64x48 (16 waves, 3 rows), FP64     tiles
static VisitRegion region13(int cfg, bool f32)
{
    switch (cfg) {
    case 0: return {16, 16};
    case 1: return {64, 32};
    case 2: return {32, 32};
    case 3: return f32 ? VisitRegion{64, 32} : VisitRegion{64, 48};
    default: return {64, 16};
    }
}

// The time of a launch as measured on 16x16 to 2048x1024 cells, within about
// 10%: a part for the launch and its loads, one per sweep, and one per 256
// tiles beyond the first 256.  us, FP32 (FP64):
//   32x32 regions   3.4 + 0.2 k, then 1.8      (3.4 + 0.38 k, then 1.9)
//   64x32, 16 waves 4.0 + 0.35 k, then 2.9     (4.6 + 0.5 k, then 7)
//   region 3        4.6 + 0.35 k, then 2.2     (5.5 + 0.8 k, then 7)
// The residual and restriction after the last sweep add 1.4 us, 1.9 in the
// 64-column regions, and (a second round of their larger state) 5 per 256
// further tiles; apart (k_residual_restrict32) they take 4.4 us and 5.4 us
// per million points.
static double cost13(int cfg, bool f32, int k, double tiles, int cus, bool end)
{
    const double more = std::max(0.0, tiles / cus - 1.0);
    double c;
    if (cfg == 2) c = f32 ? 3.4 + 0.2 * k + 1.8 * more : 3.4 + 0.38 * k + 1.9 * more;
    else if (cfg == 1) c = f32 ? 4.0 + 0.35 * k + 2.9 * more : 4.6 + 0.5 * k + 7.0 * more;
    else c = f32 ? 4.6 + 0.35 * k + 2.2 * more : 5.5 + 0.8 * k + 7.0 * more;
    if (end) c += (cfg == 2 ? 1.4 : 1.9) + 5.0 * more;
    return c;
}

// The launches of a visit of n sweeps.  A level that a region holds runs them
// (and the residual, with end) in one launch, 8 sweeps (with end): 16x16 4.2
// us (4.8), 32x32 5.7 (6.8), 64x16 5.6 (6.7), 64x32 7.6 (9.7; as tiles 8.7 and
// 10.2).  Else the cheapest, by cost13, of launches that share the sweeps
// evenly and, with end, a last one of 1 to 4 that forms the next right-hand
// side too.  us a visit of 8 sweeps (before: k_sweep_tb, 4 sweeps a launch),
// with the residual and restriction: 128x64 9.7 (15.0), 256x128 10.3 (14.6),
// 512x256 14.7 (21.3); 16 sweeps of 1024x512 44 (85); 10 of 2048x1024, none:
// 69 (127 as ten launches of one sweep).  only: 0, or the region that
// tc_set_tb_tile asks for (it too runs a level that it holds whole), or the
// one that other tables than the second-order ones take.
Visit13Plan visit_plan13(const Grid& g, bool f32, int n, bool end, int cus, int only)
{
    Visit13Plan p;
    for (int c : {0, 4, 2, 1, 3}) {
        if (only ? c != only : c == 3) continue;
        const VisitRegion rg = region13(c, f32);
        if (g.nx <= rg.w && g.nz - 1 <= rg.r && (only || c != 1 || n >= 8)) {
            p.cfg = p.end_cfg = c;
            p.whole = true;
            p.launches = (n + VISIT_KMAX - 1) / VISIT_KMAX;
            p.end = end;
            return p;
        }
    }
    auto cost = [&](int c, int k, bool e) {
        const VisitRegion rg = region13(c, f32);
        const VisitTile t = tiles_for(g, rg.w, rg.r, k, e);
        if (t.tx < 2 || t.ty < 2) return 1e30;
        const dim3 gr = tile_grid(g, t);
        return cost13(c, f32, k, (double)gr.x * gr.y, cus, e);
    };
    // n sweeps shared by m launches of region c
    auto shared = [&](int c, int sweeps, int m) {
        if (m == 0) return 0.0;
        const int k = sweeps / m, more = sweeps - k * m;  // `more` launches of k + 1, the others of k
        return more * (more ? cost(c, k + 1, false) : 0.0) + (m - more) * cost(c, k, false);
    };
    double best = 1e30;
    const double apart = end ? 4.4 + 5.4e-6 * (double)g.nx * g.nz : 0.0;
    for (int c = 1; c < 4; ++c) {
        if (only && c != only) continue;
        for (int k = 1; k <= 7; ++k) {
            if (cost(c, k, false) > 1e29) continue;
            const int m = (n + k - 1) / k;
            const double all = shared(c, n, m) + apart;
            if (all < best) {
                best = all;
                p.cfg = c;
                p.launches = m;
                p.end = false;
            }
            if (!end) continue;
            for (int ke = 1; ke <= 4 && ke <= n; ++ke) {
                const int me = (n - ke + k - 1) / k;
                const double body = shared(c, n - ke, me);
                for (int ce = 1; ce < 4; ++ce) {
                    const double t = body + cost(ce, ke, true);
                    if (t < best) {
                        best = t;
                        p.cfg = c;
                        p.launches = me;
                        p.end = true;
                        p.end_cfg = ce;
                        p.end_k = ke;
                    }
                }
            }
        }
    }
    return p;
}

namespace {

template <typename T>
H13<T> h13_from(const Spacing& h)
{
    return H13<T>{(T)h.idr2, (T)h.ids2, (T)h.idr3, (T)h.ids3, (T)h.idr4,
                  (T)h.ids4, (T)h.idrds, (T)h.idrds2, (T)h.idr2ds, (T)h.idr2ds2};
}

template <typename T, int LW, int R, int NW>
void visit13_go(hipStream_t st, dim3 gr, bool ratio, bool end, const T* in, T* out, const Args13<T>& A, const Grid& g,
                const H13<T>& h, const VisitTile& vt, const VisitFac<T>& sf, int nk, T zsg, const Start13<T>& pr,
                const End13& en)
{
    const dim3 b(NW * 64);
    if constexpr (sizeof(T) == 4) {
        if (end) {
            if (ratio) hipLaunchKernelGGL((k_visit13<T, true, LW, R, NW, true>), gr, b, 0, st, in, out, A, g, h, vt, sf, nk, zsg, pr, en, NoTables{});
            else hipLaunchKernelGGL((k_visit13<T, false, LW, R, NW, true>), gr, b, 0, st, in, out, A, g, h, vt, sf, nk, zsg, pr, en, NoTables{});
            return;
        }
    }
    if (ratio) hipLaunchKernelGGL((k_visit13<T, true, LW, R, NW, false>), gr, b, 0, st, in, out, A, g, h, vt, sf, nk, zsg, pr, en, NoTables{});
    else hipLaunchKernelGGL((k_visit13<T, false, LW, R, NW, false>), gr, b, 0, st, in, out, A, g, h, vt, sf, nk, zsg, pr, en, NoTables{});
}

template <typename T>
void launch13(hipStream_t st, int cfg, bool whole, bool ratio, bool end, const Args13<T>& A, const Grid& g,
              const Spacing& h, const T* in, T* out, const double* fac, int nk, double zsg, const Start13<T>& pr,
              const End13& en, const FD* tables)
{
    VisitFac<T> sf;
    for (int s = 0; s < nk; ++s) sf.v[s] = (T)fac[s];
    const VisitRegion rg = region13(cfg, sizeof(T) == 4);
    const VisitTile vt = whole ? whole_tile(g) : tiles_for(g, rg.w, rg.r, nk, end);
    const dim3 gr = tile_grid(g, vt);
    const H13<T> hh = h13_from<T>(h);
    const T z = (T)zsg;
    if (tables) {
        // (cfg is OTHER_TABLES_CFG)
        Tables13<T> tb;
        for (int j = 0; j < 5; ++j) {
            tb.D1[j] = (T)tables->D1[j];
            tb.D2[j] = (T)tables->D2[j];
            tb.D3[j] = (T)tables->D3[j];
            tb.D4[j] = (T)tables->D4[j];
        }
        if (ratio) hipLaunchKernelGGL((k_visit13<T, true, 32, 1, 16, false, Tables13<T>>), gr, dim3(1024), 0, st, in, out, A, g, hh, vt, sf, nk, z, pr, en, tb);
        else hipLaunchKernelGGL((k_visit13<T, false, 32, 1, 16, false, Tables13<T>>), gr, dim3(1024), 0, st, in, out, A, g, hh, vt, sf, nk, z, pr, en, tb);
        return;
    }
    switch (cfg) {
    case 0: visit13_go<T, 16, 1, 4>(st, gr, ratio, end, in, out, A, g, hh, vt, sf, nk, z, pr, en); break;
    case 1: visit13_go<T, 64, 2, 16>(st, gr, ratio, end, in, out, A, g, hh, vt, sf, nk, z, pr, en); break;
    case 2: visit13_go<T, 32, 1, 16>(st, gr, ratio, end, in, out, A, g, hh, vt, sf, nk, z, pr, en); break;
    case 4: visit13_go<T, 64, 1, 16>(st, gr, ratio, end, in, out, A, g, hh, vt, sf, nk, z, pr, en); break;
    default:
        if constexpr (sizeof(T) == 4) visit13_go<T, 64, 4, 8>(st, gr, ratio, end, in, out, A, g, hh, vt, sf, nk, z, pr, en);
        else visit13_go<T, 64, 3, 16>(st, gr, ratio, end, in, out, A, g, hh, vt, sf, nk, z, pr, en);
        break;
    }
}

}  // namespace

void launch_visit13_32(hipStream_t st, int cfg, bool whole, bool use_ratio, const Level& L, const float* rhs,
                       const float* in, float* out, const Spacing& h, const double* fac, int nk, double zsg,
                       const float* Pc, const Grid* gc, const RRTarget* rr, const FD* tables)
{
    const Args13<float> A{L.vis32, L.visx32, L.visz32, L.a132, nullptr, nullptr, L.visxz32,
                         const_cast<float*>(rhs), L.dts32, L.lb32};
    Prolong13 pr{nullptr, L.g};
    if (Pc) { pr.Ec = Pc; pr.gc = *gc; }
    End13 en{};
    if (rr) { en.out = rr->out; en.go = rr->go; en.RowB = rr->RowB; en.bout = rr->bout; en.h = h32_from(h); }
    launch13<float>(st, cfg, whole, use_ratio, rr != nullptr, A, L.g, h, in, out, fac, nk, zsg, pr, en, tables);
}

void launch_visit13_64(hipStream_t st, int cfg, bool whole, bool use_ratio, const Level& L, const double* rhs,
                       const double* in, double* out, const Spacing& h, const double* fac, int nk, double zsg,
                       const VisitStart& vs, const FD* tables)
{
    const Args13<double> A{L.vis, L.visx, L.visz, nullptr, L.visxx, L.viszz, L.visxz, const_cast<double*>(rhs),
                           L.dtstream, L.ratio};
    launch13<double>(st, cfg, whole, use_ratio, false, A, L.g, h, in, out, fac, nk, zsg, vs, End13{}, tables);
}

}  // namespace tc
