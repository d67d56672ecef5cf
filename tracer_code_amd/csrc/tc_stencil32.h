// FP32 form of the stream_space stencil (the mixed-precision cycle).
#pragma once
#include "tc_stencil.h"

namespace tc {

struct FD32 {
    float D1[5], D2[5], D3[5], D4[5];
    float Drs[9], Drss[9], Drrs[9], Drrss[9];
};
struct H32 {
    float idr, ids, idr2, ids2, idr3, ids3, idr4, ids4, idrds, idrds2, idr2ds, idr2ds2;
};

inline FD32 fd32_from(const FD& F)
{
    FD32 o;
    for (int j = 0; j < 5; ++j) { o.D1[j] = (float)F.D1[j]; o.D2[j] = (float)F.D2[j]; o.D3[j] = (float)F.D3[j]; o.D4[j] = (float)F.D4[j]; }
    for (int j = 0; j < 9; ++j) { o.Drs[j] = (float)F.Drs[j]; o.Drss[j] = (float)F.Drss[j]; o.Drrs[j] = (float)F.Drrs[j]; o.Drrss[j] = (float)F.Drrss[j]; }
    return o;
}
inline H32 h32_from(const Spacing& h)
{
    return H32{(float)h.idr, (float)h.ids, (float)h.idr2, (float)h.ids2, (float)h.idr3, (float)h.ids3,
               (float)h.idr4, (float)h.ids4, (float)h.idrds, (float)h.idrds2, (float)h.idr2ds, (float)h.idr2ds2};
}

#pragma clang fp contract(fast)
// FP32 fields and weights; A is the arithmetic type.  With A = double every
// product of two FP32 values is exact and only the sums round, which keeps
// the residual passed to the next level accurate relative to the (small)
// defect even where rhs and L(S) nearly cancel.
template <typename A, int AX, typename G>
__device__ __forceinline__ A dot3gf(const float* D, const G& S)
{
    return A(D[1]) * A(S(AX == 0 ? -1 : 0, AX == 0 ? 0 : -1)) + A(D[2]) * A(S(0, 0)) +
           A(D[3]) * A(S(AX == 0 ? 1 : 0, AX == 0 ? 0 : 1));
}
template <typename A, int AX, typename G>
__device__ __forceinline__ A dot5gf(const float* D, const G& S)
{
    return A(D[0]) * A(S(AX == 0 ? -2 : 0, AX == 0 ? 0 : -2)) + A(D[1]) * A(S(AX == 0 ? -1 : 0, AX == 0 ? 0 : -1)) +
           A(D[2]) * A(S(0, 0)) + A(D[3]) * A(S(AX == 0 ? 1 : 0, AX == 0 ? 0 : 1)) +
           A(D[4]) * A(S(AX == 0 ? 2 : 0, AX == 0 ? 0 : 2));
}
template <typename A, typename G>
__device__ __forceinline__ A sum9gf(const float* M, const G& S)
{
    return A(M[0]) * A(S(-1, -1)) + A(M[1]) * A(S(0, -1)) + A(M[2]) * A(S(1, -1)) + A(M[3]) * A(S(-1, 0)) +
           A(M[4]) * A(S(0, 0)) + A(M[5]) * A(S(1, 0)) + A(M[6]) * A(S(-1, 1)) + A(M[7]) * A(S(0, 1)) +
           A(M[8]) * A(S(1, 1));
}
// rhs - L(S); a1 = vis_xx - vis_zz
template <typename A, typename G>
__device__ __forceinline__ A stream_space32_g(const FD32& F, const H32& h, const G& S, float vis, float vx, float vz,
                                              float a1, float vxz, float rhs)
{
    A Srr = dot3gf<A, 0>(F.D2, S) * A(h.idr2);
    A Sss = dot3gf<A, 1>(F.D2, S) * A(h.ids2);
    A Srrr = dot5gf<A, 0>(F.D3, S) * A(h.idr3);
    A Ssss = dot5gf<A, 1>(F.D3, S) * A(h.ids3);
    A Srrrr = dot5gf<A, 0>(F.D4, S) * A(h.idr4);
    A Sssss = dot5gf<A, 1>(F.D4, S) * A(h.ids4);
    A Srs = sum9gf<A>(F.Drs, S) * A(h.idrds);
    A Srss = sum9gf<A>(F.Drss, S) * A(h.idrds2);
    A Srrs = sum9gf<A>(F.Drrs, S) * A(h.idr2ds);
    A Srrss = sum9gf<A>(F.Drrss, S) * A(h.idr2ds2);
    A L = A(a1) * (Srr - Sss) + A(vis) * (Srrrr + Sssss) + A(2) * A(vis) * Srrss + A(4) * A(vxz) * Srs +
          A(2) * A(vx) * (Srrr + Srss) + A(2) * A(vz) * (Ssss + Srrs);
    return A(rhs) - L;
}
template <typename A>
__device__ __forceinline__ A stream_space32(const FD32& F, const H32& h, const float* __restrict__ S, size_t c,
                                            ptrdiff_t ld, float vis, float vx, float vz, float a1, float vxz,
                                            float rhs)
{
    return stream_space32_g<A>(F, h, PlaneAt<float>{S, c, ld}, vis, vx, vz, a1, vxz, rhs);
}

// S(i+di, k+dk) of a 7x7 neighbourhood held in registers (row-major, centre
// at index 24) for the point (a, b) cells from its centre
struct Patch7At {
    const float* p;
    int a, b;
    __device__ __forceinline__ float operator()(int di, int dk) const { return p[(b + dk + 3) * 7 + a + di + 3]; }
};

// The weights of the 13 taps of one point for any tables F (D1..D4 at
// offsets -2..2) and reciprocal spacings h: c, xm1, xp1, xm2, xp2, zm1, zp1,
// zm2, zp2, mm, pm, mp, pp
template <typename T, typename TAB, typename H>
__device__ __forceinline__ void tap_weights(const TAB& F, const H& h, T vis, T vx, T vz, T a1, T vxz, T (&v)[13])
{
    // axis parts: a1 (S_rr - S_ss) + 2 vx S_rrr + 2 vz S_sss + vis (S_rrrr + S_ssss)
    auto wx = [&](int d) { return a1 * F.D2[d + 2] * h.idr2 + T(2) * vx * F.D3[d + 2] * h.idr3 + vis * F.D4[d + 2] * h.idr4; };
    auto wz = [&](int d) { return -a1 * F.D2[d + 2] * h.ids2 + T(2) * vz * F.D3[d + 2] * h.ids3 + vis * F.D4[d + 2] * h.ids4; };
    // 3x3 part: 4 vxz S_rs + 2 vx S_rss + 2 vz S_rrs + 2 vis S_rrss
    auto wb = [&](int di, int dk) {
        return T(4) * vxz * F.D1[dk + 2] * F.D1[di + 2] * h.idrds + T(2) * vx * F.D2[dk + 2] * F.D1[di + 2] * h.idrds2 +
               T(2) * vz * F.D1[dk + 2] * F.D2[di + 2] * h.idr2ds + T(2) * vis * F.D2[dk + 2] * F.D2[di + 2] * h.idr2ds2;
    };
    const T w[13] = {wx(0) + wz(0) + wb(0, 0), wx(-1) + wb(-1, 0), wx(1) + wb(1, 0), wx(-2), wx(2),
                     wz(-1) + wb(0, -1), wz(1) + wb(0, 1), wz(-2), wz(2), wb(-1, -1), wb(1, -1), wb(-1, 1), wb(1, 1)};
#pragma unroll
    for (int q = 0; q < 13; ++q) v[q] = w[q];
}

// restrict (iterative_solver.f90:596-626) at one coarse point from the fine
// residuals around its fine centre: the reference's weights, whose corner sum
// counts (ii-1,kk+1) twice and (ii+1,kk-1) not at all
__device__ __forceinline__ float restrict_fw32(float rmm, float rmp, float rpp, float rm0, float r0m, float rp0,
                                               float r0p, float r00)
{
    const float corners = (rmm + rmp + rpp + rmp) * (1.0f / 16.0f);
    const float sides = (rm0 + r0m + rp0 + r0p) * (1.0f / 8.0f);
    return corners + sides + r00 * 0.25f;
}
#pragma clang fp contract(off)

// rhs - L(S) of FP32 fields in FP64 with the second-order tables put in
// (stream_space32_g; the products of FP32 values are exact, the sums round):
// explicit operations, so that every kernel gets the same bits
struct Tap13d {
    double c, xm1, xp1, xm2, xp2, zm1, zp1, zm2, zp2, mm, pm, mp, pp;
};
__device__ __forceinline__ float residual32_std(const Tap13d& t, const H32& h, float vis, float vx, float vz, float a1,
                                                float vxz, float rhs)
{
    const double Srr = fma(-2.0, t.c, t.xm1) + t.xp1, Sss = fma(-2.0, t.c, t.zm1) + t.zp1;
    const double Srrr = fma(0.5, t.xp2, fma(-0.5, t.xm2, t.xm1) - t.xp1);
    const double Ssss = fma(0.5, t.zp2, fma(-0.5, t.zm2, t.zm1) - t.zp1);
    const double Srrrr = fma(6.0, t.c, fma(-4.0, t.xm1, t.xm2) + fma(-4.0, t.xp1, t.xp2));
    const double Sssss = fma(6.0, t.c, fma(-4.0, t.zm1, t.zm2) + fma(-4.0, t.zp1, t.zp2));
    const double dm = t.mm - t.pm, dp = t.pp - t.mp, sm = t.mm + t.pm, sp = t.pp + t.mp;
    const double Srs = 0.25 * (dm + dp);
    const double Srss = fma(0.5, dp - dm, t.xm1 - t.xp1);
    const double Srrs = fma(0.5, sp - sm, t.zm1 - t.zp1);
    const double Srrss = fma(-2.0, (t.xm1 + t.xp1) + (t.zm1 + t.zp1), fma(4.0, t.c, sm + sp));
    double L = (double)a1 * fma(Srr, (double)h.idr2, -(Sss * (double)h.ids2));
    L = fma((double)vis, fma(Srrrr, (double)h.idr4, Sssss * (double)h.ids4), L);
    L = fma(2.0 * (double)vis, Srrss * (double)h.idr2ds2, L);
    L = fma(4.0 * (double)vxz, Srs * (double)h.idrds, L);
    L = fma(2.0 * (double)vx, fma(Srrr, (double)h.idr3, Srss * (double)h.idrds2), L);
    L = fma(2.0 * (double)vz, fma(Ssss, (double)h.ids3, Srrs * (double)h.idr2ds), L);
    return (float)((double)rhs - L);
}
template <typename G>
__device__ __forceinline__ Tap13d taps13(const G& S)
{
    return Tap13d{S(0, 0),  S(-1, 0),  S(1, 0),  S(-2, 0), S(2, 0),  S(0, -1), S(0, 1),
                  S(0, -2), S(0, 2),   S(-1, -1), S(1, -1), S(-1, 1), S(1, 1)};
}

}  // namespace tc
