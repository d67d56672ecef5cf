// Coarsest-grid direct solve of the multigrid W-cycle
// (Compute_Matrix_coarse iterative_solver.f90:1026-1179, DGBEQU/DGBTRF at
// :1165/:97, Compute_coarse_vector/DGBTRS/Stream_grid_coarse :139-142,
// :1181-1204).
//
// The reference factors the row-equilibrated banded matrix with MKL and
// back-substitutes 8 times per 6-level W-cycle.  Sequential banded
// substitution is latency-bound on a GPU, so here the matrix is factored
// once per solve (LAPACK DGBTF2 semantics, one workgroup, by panels), its
// explicit inverse is formed column-parallel from those factors (DGBTRS
// applied to the unit vectors, by blocks), and every coarse visit becomes one
// dense GEMV that streams the inverse from HBM / Infinity Cache.
#include "tc_kernels.h"

namespace tc {

// Band storage: A(p,q) (1-based) at ab[(kl+ku+p-q) + (q-1)*ldab] (0-based row).
#define ABx(r, q) ab[(size_t)(r) + (size_t)(q) * (size_t)ldab]

// stream_space with build=1 (iterative_solver.f90:487-560), uniform grid:
// coefficient of S(iq,kq)*Sval in the row of interior point (i,k).
__device__ double stream_coeff(const FD& F, const Spacing& h, int ivis, double vis, double vx, double vz, double vxx,
                               double vzz, double vxz, int i, int k, int iq, int kq, double Sval)
{
    const int di = iq - i, dk = kq - k;
    double Sr = 0, Srr = 0, Srrr = 0, Srrrr = 0, Ss = 0, Sss = 0, Ssss = 0, Sssss = 0;
    if (k == kq) {
        Sr = F.D1[di + 2] * Sval / h.dr;
        Srr = F.D2[di + 2] * Sval / h.dr2;
        Srrr = F.D3[di + 2] * Sval / h.dr3;
        Srrrr = F.D4[di + 2] * Sval / h.dr4;
    }
    if (i == iq) {
        Ss = F.D1[dk + 2] * Sval / h.ds;
        Sss = F.D2[dk + 2] * Sval / h.ds2;
        Ssss = F.D3[dk + 2] * Sval / h.ds3;
        Sssss = F.D4[dk + 2] * Sval / h.ds4;
    }
    double m9 = 0.0, m9s = 0.0, m9r = 0.0, m9rs = 0.0;
    if (di >= -1 && di <= 1 && dk >= -1 && dk <= 1) {
        const int t = (dk + 1) * 3 + (di + 1);
        m9 = F.Drs[t]; m9s = F.Drss[t]; m9r = F.Drrs[t]; m9rs = F.Drrss[t];
    }
    double Srs = m9 * Sval / h.drds;
    double Srss = m9s * Sval / h.drds2;
    double Srrs = m9r * Sval / h.dr2ds;
    double Srrss = m9rs * Sval / h.dr2ds2;
    (void)Sr; (void)Ss;
    double t1, t2, t3, t4, t5, t6;
    if (ivis == 0) {
        t1 = 0.0; t2 = vis * (Srrrr + Sssss); t3 = 2.0 * vis * Srrss; t4 = 0.0; t5 = 0.0; t6 = 0.0;
    } else {
        t1 = (vxx - vzz) * (Srr - Sss);
        t2 = vis * (Srrrr + Sssss);
        t3 = 2.0 * vis * Srrss;
        t4 = 4.0 * vxz * Srs;
        t5 = 2.0 * vx * (Srrr + Srss);
        t6 = 2.0 * vz * (Ssss + Srrs);
    }
    return t1 + t2 + t3 + t4 + t5 + t6;
}

// One thread per matrix row p (Database=2 ordering p = (nz_c+1)*ip + kp + 1):
// set the in-domain stencil entries, add the folded ghost entries, identity
// rows on the walls, then DGBEQU's row factor R(p) = 1/max|A(p,:)| and the
// row scaling.  The band must be zero on entry.
__global__ __launch_bounds__(256) void k_coarse_assemble(double* __restrict__ ab, double* __restrict__ RowB,
                                                         const double* __restrict__ V, const double* __restrict__ vx,
                                                         const double* __restrict__ vz, const double* __restrict__ vxx,
                                                         const double* __restrict__ vzz, const double* __restrict__ vxz,
                                                         Grid g, FD F, Spacing h, int ivis, int Vbc, int kl, int ku, int n)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x + 1;
    if (p > n) return;
    const int ldab = 2 * kl + ku + 1, kl_ku_1 = kl + ku + 1;
    const int nxc = g.nx, nzc = g.nz, N = nzc + 1;
    const int kp = p - N * ((p - 1) / N) - 1, ip = (p - 1) / N;
    const int limit[5] = {0, 1, 2, 1, 0};
    if (ip > 0 && ip < nxc && kp > 0 && kp < nzc) {
        const size_t c = g.at(ip, kp);
        const double vis = V[c], gx = vx[c], gz = vz[c], gxx = vxx[c], gzz = vzz[c], gxz = vxz[c];
        for (int j = -2; j <= 2; ++j) {
            int iq = j + ip;
            if (iq >= 0 && iq <= nxc)
                for (int kq = -limit[j + 2] + kp; kq <= kp + limit[j + 2]; ++kq)
                    if (kq >= 0 && kq <= nzc) {
                        int q = N * iq + kq + 1;
                        ABx(kl_ku_1 + p - q - 1, q - 1) = stream_coeff(F, h, ivis, vis, gx, gz, gxx, gzz, gxz, ip, kp, iq, kq, 1.0);
                    }
        }
        for (int j = -2; j <= 2; ++j) {
            int iq = j + ip;
            for (int kq = -limit[j + 2] + kp; kq <= kp + limit[j + 2]; ++kq) {
                if (iq < 0 || iq > nxc || kq < 0 || kq > nzc) {
                    int iiq, kkq;
                    double xval, zval;
                    if (iq < 0) { iiq = -iq; xval = -1.0; }
                    else if (iq > nxc) { iiq = 2 * nxc - iq; xval = -1.0; }
                    else { iiq = iq; xval = 1.0; }
                    if (kq < 0) { kkq = -kq; zval = (Vbc == 0) ? -1.0 : 1.0; }
                    else if (kq > nzc) { kkq = 2 * nzc - kq; zval = (Vbc == 0) ? -1.0 : 1.0; }
                    else { kkq = kq; zval = 1.0; }
                    double Sval = xval * zval;
                    int q = N * iiq + kkq + 1;
                    double& a = ABx(kl_ku_1 + p - q - 1, q - 1);
                    a = a + stream_coeff(F, h, ivis, vis, gx, gz, gxx, gzz, gxz, ip, kp, iq, kq, Sval);
                }
            }
        }
    } else {
        ABx(kl_ku_1 - 1, p - 1) = 1.0;
    }
    // DGBEQU row factor over the band of row p, then the row scaling.
    const double smlnum = 2.2250738585072014e-308, bignum = 1.0 / smlnum;
    double rmax = 0.0;
    int q0 = p - kl > 1 ? p - kl : 1, q1 = p + ku < n ? p + ku : n;
    for (int q = q0; q <= q1; ++q) {
        double v = fabs(ABx(kl_ku_1 + p - q - 1, q - 1));
        if (v > rmax) rmax = v;
    }
    double rv = rmax > smlnum ? rmax : smlnum;
    rv = rv < bignum ? rv : bignum;
    double R = 1.0 / rv;
    RowB[p - 1] = R;
    // rows p with p-q in [-kl, ku] are scaled (iterative_solver.f90:1168-1172)
    int s0 = p - ku > 1 ? p - ku : 1, s1 = p + kl < n ? p + kl : n;
    for (int q = s0; q <= s1; ++q) {
        double& a = ABx(kl_ku_1 + p - q - 1, q - 1);
        a = R * a;
    }
}

// DGBTF2 (LAPACK, unblocked banded LU with partial pivoting) by one
// workgroup; same operations per element as the reference algorithm.
__global__ __launch_bounds__(256) void k_dgbtf2(double* __restrict__ ab, int ldab, int n, int kl, int ku,
                                                int32_t* __restrict__ ipiv, int32_t* __restrict__ info_out)
{
    const int kv = ku + kl;
    const int tid = threadIdx.x, nt = blockDim.x;
    __shared__ int sh_jp;
    __shared__ int sh_ju;
    __shared__ double sh_piv, sh_old;
    __shared__ int sh_info;
    for (int j = ku + 1; j < (kv < n ? kv : n); ++j)
        for (int i = kv - j + tid; i < kl; i += nt) ABx(i, j) = 0.0;
    if (tid == 0) { sh_ju = 0; sh_info = 0; }
    __syncthreads();
    for (int j = 0; j < n; ++j) {
        if (j + kv < n)
            for (int i = tid; i < kl; i += nt) ABx(i, j + kv) = 0.0;
        const int km = kl < n - 1 - j ? kl : n - 1 - j;
        // IDAMAX over rows kv..kv+km of column j (first maximum wins), wave 0
        if (tid < 64) {
            double best = -1.0;
            int bi = 1 << 30;
            for (int t = tid; t <= km; t += 64) {
                double v = fabs(ABx(kv + t, j));
                if (v > best) { best = v; bi = t; }
            }
            for (int off = 32; off > 0; off >>= 1) {
                double ob = __shfl_down(best, off, 64);
                int oi = __shfl_down(bi, off, 64);
                if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
            }
            if (tid == 0) {
                sh_jp = bi;
                sh_piv = ABx(kv + bi, j);
                sh_old = ABx(kv, j);
            }
        }
        __syncthreads();
        const int jp = sh_jp;
        const double piv = sh_piv;
        if (tid == 0) ipiv[j] = jp + j + 1;
        if (piv != 0.0) {
            int jt = j + ku + jp;
            if (jt > n - 1) jt = n - 1;
            const int ju = sh_ju > jt ? sh_ju : jt;
            // column j: swap + DSCAL by the reciprocal pivot; columns j+1..ju: swap
            const double rp = 1.0 / piv;
            if (tid == 0) ABx(kv, j) = piv;
            for (int t = 1 + tid; t <= km; t += nt) {
                double v = (t == jp) ? sh_old : ABx(kv + t, j);
                ABx(kv + t, j) = v * rp;
            }
            if (jp != 0)
                for (int t = 1 + tid; t <= ju - j; t += nt) {
                    double a = ABx(kv + jp - t, j + t);
                    ABx(kv + jp - t, j + t) = ABx(kv - t, j + t);
                    ABx(kv - t, j + t) = a;
                }
            __syncthreads();
            if (tid == 0) sh_ju = ju;
            // DGER rank-1 update of the trailing band
            if (km > 0 && ju > j) {
                const int ncol = ju - j;
                const int tot = ncol * km;
                for (int e = tid; e < tot; e += nt) {
                    int jj = e / km + 1, t = e % km + 1;
                    double y = ABx(kv - jj, j + jj);
                    if (y != 0.0) {
                        double temp = -1.0 * y;
                        ABx(kv + t - jj, j + jj) += ABx(kv + t, j) * temp;
                    }
                }
            }
        } else if (tid == 0 && sh_info == 0) {
            sh_info = j + 1;
        }
        __syncthreads();
    }
    if (tid == 0) *info_out = sh_info;
}

// ---------------------------------------------------------------------------
// DGBTF2 by panels of CB columns, one workgroup, the active part of the band
// in LDS.
//
// Bound: the chain of n pivots (search, reciprocal, update of the next
// column).  One barrier-separated step per column took 2.4 to 4.1 us; here one
// wavefront factors a panel in registers (a lane per row, two rows a lane
// where there are more than 64; pivot search by lane shifts, the pivot row by
// lane reads), and the other columns take the panel's CB steps at once: their
// row swaps and the unit-lower solve with a thread per column, then the update
// of the rows below as 16x16 FP64 matrix products, which read each element of
// the window once per panel instead of once per column.
//
// Element (r, c) of the window, rows 16J..16J+95 of columns 16J..16J+159 at
// panel J, lives at W[(c % LU_CS) * LU_RS + r % LU_RW]: blocks of 16 never
// wrap, and the odd column stride keeps both a lane per row and a lane per
// column free of bank conflicts.  The pivots are DGBTF2's (largest magnitude,
// first row wins), the stored factors have its form (multipliers of a column
// not moved by later swaps), and each update is a fused multiply-add.
// Measured, by columns and bandwidth: 2145, 66 8.7 -> 2.35 ms; 897, 46 2.76 ->
// 0.77; 280, 28 0.67 -> 0.25; 81, 18 0.17 -> 0.09 (1.1 and 0.9 us a column
// with two rows a lane and with one).
// ---------------------------------------------------------------------------
constexpr int CB = 16;          // panel and block size
constexpr int LU_CS = 10 * CB;  // column slots: 15 + kl + ku + 1 of them at most
constexpr int LU_RW = 6 * CB;   // row slots: 15 + kl + 1 at most
constexpr int LU_RS = LU_RW + 1;
constexpr int LU_THREADS = 512;
// Bands that the blocked kernels take (kl = ku = 72 at most, by the window's 16
// columns and rows beyond the band).  At 289 columns, kl 72: 3.2 + 5.4 ms by the
// general kernels, 0.35 + 0.09 here; wider windows do not fit the LDS.
bool coarse_blocked(int kl, int ku) { return CB + kl + ku <= LU_CS && CB + kl <= LU_RW; }

typedef double v4d __attribute__((ext_vector_type(4)));
// D = A B + C of 16x16x4: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and
// D[4 v + l / 16][l % 16] in component v
__device__ __forceinline__ v4d mfma4(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ double lane_read(double v, int l)
{
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned dpp_max(unsigned v)
{
    return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, ROWS == 0xf));
}
// largest of a wavefront's 64 values, in every lane
__device__ __forceinline__ unsigned wave_max(unsigned v)
{
    v = dpp_max<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
    v = dpp_max<0x112, 0xf>(v);
    v = dpp_max<0x114, 0xf>(v);
    v = dpp_max<0x118, 0xf>(v);
    v = dpp_max<0x142, 0xa>(v);  // row_bcast 15, 31
    v = dpp_max<0x143, 0xc>(v);
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
// order of a magnitude's high word; 0 for what is not a candidate or not a number
__device__ __forceinline__ unsigned pivot_key(double v, bool valid)
{
    const unsigned hi = (unsigned)__double2hiint(v) & 0x7fffffffu;
    return valid && !(v != v) ? hi + 1 : 0;
}

// H: rows a lane of the panel's wavefront (1 where all its rows fit in 64)
template <int H>
__global__ __launch_bounds__(LU_THREADS) void k_lu_panels(double* __restrict__ ab, int ldab, int n, int kl, int ku,
                                                         int32_t* __restrict__ ipiv, int32_t* __restrict__ info_out)
{
    extern __shared__ double W[];  // LU_CS * LU_RS
    __shared__ int piv_s[CB];
    const int kv = ku + kl;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    auto slot = [&](int r, int c) { return (c % LU_CS) * LU_RS + r % LU_RW; };
    auto band = [&](int r, int c) -> double {
        return (r < n && c < n && c - r <= ku && r - c <= kl) ? ab[(size_t)(kv + r - c) + (size_t)c * ldab] : 0.0;
    };
    for (int e = tid; e < LU_CS * LU_RW; e += LU_THREADS) {
        const int r = e % LU_RW, c = e / LU_RW;
        W[slot(r, c)] = band(r, c);
    }
    int info = 0;
    __syncthreads();
    // entering at the next panel: 16 rows of its 160 columns, 16 columns of
    // its other 80 rows
    constexpr int NROW = CB * LU_CS, NIN = NROW + CB * (LU_RW - CB), PER = (NIN + LU_THREADS - 1) / LU_THREADS;
    for (int j0 = 0; j0 < n; j0 += CB) {
        auto entering = [&](int e, int& r, int& c) {
            if (e < NROW) { r = j0 + LU_RW + e % CB; c = j0 + CB + e / CB; }
            else { r = j0 + CB + (e - NROW) % (LU_RW - CB); c = j0 + LU_CS + (e - NROW) / (LU_RW - CB); }
        };
        double vin[PER];
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int e = tid + u * LU_THREADS;
            int r, c;
            entering(e < NIN ? e : 0, r, c);
            vin[u] = band(r, c);
        }
        if (wv == 0) {
            // A row stays in its lane; pos is where DGBTF2 would have it, so an
            // interchange is two lanes' pos.
            double v[H][CB];
            int pos[H];
#pragma unroll
            for (int h = 0; h < H; ++h) {
                pos[h] = lane + 64 * h;
#pragma unroll
                for (int c = 0; c < CB; ++c)
                    v[h][c] = pos[h] < LU_RW ? W[slot(j0 + pos[h], j0 + c)] : 0.0;
            }
#pragma unroll
            for (int q = 0; q < CB; ++q) {
                const int j = j0 + q;
                if (j < n) {
                    // candidates: rows q .. q + km of the panel
                    const int km = kl < n - 1 - j ? kl : n - 1 - j;
                    unsigned key[H], k = 0;
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        key[h] = pivot_key(v[h][q], pos[h] >= q && pos[h] <= q + km);
                        k = max(k, key[h]);
                    }
                    const unsigned top = wave_max(k);
                    // the largest magnitude's lane: one of equal high word, or the
                    // first row of the largest of several; without a number
                    // among the candidates the row q stays
                    int pl = 0, ph = 0;
                    unsigned long long m[H];
                    int cnt = 0;
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        m[h] = __ballot(top ? key[h] == top : pos[h] == q);
                        cnt += __popcll(m[h]);
                        if (m[h]) { pl = __ffsll(m[h]) - 1; ph = h; }
                    }
                    if (cnt > 1) {
                        double best = -1.0;
                        int bpos = 1 << 30;
#pragma unroll
                        for (int h = 0; h < H; ++h)
                            for (unsigned long long t = m[h]; t; t &= t - 1) {
                                const int l = __ffsll(t) - 1;
                                const double x = fabs(lane_read(v[h][q], l));
                                const int xp = __builtin_amdgcn_readlane(pos[h], l);
                                if (x > best || (x == best && xp < bpos)) { best = x; bpos = xp; pl = l; ph = h; }
                            }
                        pl = __builtin_amdgcn_readfirstlane(pl);
                        ph = __builtin_amdgcn_readfirstlane(ph);
                    }
                    const bool second = H == 2 && ph == 1;
                    auto of_pivot = [&](int c) {
                        const double x = lane_read(v[0][c], pl);
                        if (H == 1) return x;
                        const double z = lane_read(v[H - 1][c], pl);
                        return second ? z : x;
                    };
                    const double piv = of_pivot(q);
                    const double rp = piv != 0.0 ? 1.0 / piv : 0.0;
                    const int p = __builtin_amdgcn_readlane(second ? pos[H - 1] : pos[0], pl);
#pragma unroll
                    for (int h = 0; h < H; ++h)
                        pos[h] = (ph == h && lane == pl) ? q : (pos[h] == q ? p : pos[h]);
                    if (lane == 0) {
                        piv_s[q] = p;
                        ipiv[j] = j0 + p + 1;
                    }
                    if (piv == 0.0 && info == 0) info = j + 1;
                    double l[H];
                    double* abj = ab + (size_t)j * ldab + (kv - q);
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        const bool below = pos[h] > q;
                        l[h] = below ? v[h][q] * rp : 0.0;
                        v[h][q] = below ? l[h] : v[h][q];
                        // the multipliers, where DGBTF2 keeps them
                        if (below && pos[h] <= q + km) abj[pos[h]] = l[h];
                    }
#pragma unroll
                    for (int c = q + 1; c < CB; ++c) {
                        const double u = of_pivot(c);
#pragma unroll
                        for (int h = 0; h < H; ++h) v[h][c] = __builtin_fma(-l[h], u, v[h][c]);
                    }
                } else if (lane == 0) {
                    piv_s[q] = q;
                }
            }
#pragma unroll
            for (int h = 0; h < H; ++h)
                if (pos[h] < LU_RW) {
                    double* o = W + (j0 + pos[h]) % LU_RW;
#pragma unroll
                    for (int c = 0; c < CB; ++c) o[((j0 + c) % LU_CS) * LU_RS] = v[h][c];
                }
        }
        __syncthreads();
        // the panel's swaps and unit-lower solve, a thread per column
        if (tid < LU_CS - CB) {
            const int c = j0 + CB + tid;
            double* col = W + (c % LU_CS) * LU_RS;
#pragma unroll
            for (int q = 0; q < CB; ++q) {
                const int p = __builtin_amdgcn_readfirstlane(piv_s[q]);
                if (p != q) {
                    const int sp = (j0 + p) % LU_RW, sq = (j0 + q) % LU_RW;
                    const double t = col[sp];
                    col[sp] = col[sq];
                    col[sq] = t;
                }
            }
            double u[CB];
            const int s0 = j0 % LU_RW;
#pragma unroll
            for (int q = 0; q < CB; ++q) u[q] = col[s0 + q];
#pragma unroll
            for (int q = 0; q < CB; ++q) {
                const double* Lq = W + ((j0 + q) % LU_CS) * LU_RS + s0;
#pragma unroll
                for (int r = q + 1; r < CB; ++r) u[r] = __builtin_fma(-Lq[r], u[q], u[r]);
            }
#pragma unroll
            for (int q = 0; q < CB; ++q) col[s0 + q] = u[q];
        }
        __syncthreads();
        // the rows below: C -= L U, a 16x16 block of the window at a time
        {
            const int g = lane >> 4, m = lane & 15, s0 = j0 % LU_RW;
            constexpr int NR = LU_RW / CB - 1, NC = LU_CS / CB - 1;
            for (int b = wv; b < NR * NC; b += LU_THREADS / 64) {
                const int rs = (j0 + CB * (1 + b % NR)) % LU_RW;
                double* Cc = W + ((j0 + CB * (1 + b / NR) + m) % LU_CS) * LU_RS;
                v4d acc = {Cc[rs + g], Cc[rs + 4 + g], Cc[rs + 8 + g], Cc[rs + 12 + g]};
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const double a = -W[((j0 + 4 * s + g) % LU_CS) * LU_RS + rs + m];
                    acc = mfma4(a, Cc[s0 + 4 * s + g], acc);
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) Cc[rs + 4 * v + g] = acc[v];
            }
        }
        // the finished rows of U
        for (int e = tid; e < CB * LU_CS; e += LU_THREADS) {
            const int r = j0 + e % CB, c = j0 + e / CB;
            if (c >= r && c - r <= kv && c < n) ab[(size_t)(kv + r - c) + (size_t)c * ldab] = W[slot(r, c)];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const int e = tid + u * LU_THREADS;
            if (e < NIN) {
                int r, c;
                entering(e, r, c);
                W[slot(r, c)] = vin[u];
            }
        }
        __syncthreads();
    }
    if (tid == 0) *info_out = info;
}

// Explicit inverse from the DGBTF2 factors: lane c of a wavefront applies
// DGBTRS('N') to the unit vector e_c (the same operations, in the same
// order, as the reference algorithm), writing column c of A^-1 into the
// row-major Ainv (lanes touch consecutive columns: coalesced).  The rows a
// substitution step touches form a window of kl+1 (forward) or kl+ku+1
// (backward) rows that slides by one row per step; it lives in LDS as a
// circular buffer, so each step is LDS traffic plus one coalesced global
// store of the row that leaves the window.
template <int INV_COLS>
__global__ __launch_bounds__(64) void k_band_inverse(const double* __restrict__ ab, int ldab, int n, int kl, int ku,
                                                     const int32_t* __restrict__ ipiv, double* __restrict__ X)
{
    extern __shared__ double win[];  // [W][INV_COLS]
    const int lane = threadIdx.x;
    const int c = blockIdx.x * INV_COLS + lane;
    const bool active = c < n;
    const size_t nn = (size_t)n;
    const int kd = ku + kl;
    // ---- forward: L^-1 P e_c, window rows [j, j+kl] -----------------------
    const int Wf = kl + 1;
    const int cmin = blockIdx.x * INV_COLS;
    const int jstart = cmin - kl > 0 ? cmin - kl : 0;  // rows before this are zero for every lane
    for (int t = 0; t < Wf; ++t) {
        const int row = jstart + t;
        win[((row % Wf) * INV_COLS) + lane] = (row == c) ? 1.0 : 0.0;
    }
    for (int i = 0; i < jstart && active; ++i) X[(size_t)i * nn + c] = 0.0;
    for (int j = jstart; j < n; ++j) {
        if (j < n - 1) {
            const int lm = kl < n - 1 - j ? kl : n - 1 - j;
            const int l = ipiv[j] - 1;
            if (l != j) {
                double& a = win[(l % Wf) * INV_COLS + lane];
                double& b = win[(j % Wf) * INV_COLS + lane];
                const double tmp = a;
                a = b;
                b = tmp;
            }
            const double bj = win[(j % Wf) * INV_COLS + lane];
            if (bj != 0.0) {
                const double temp = -1.0 * bj;
                for (int t = 1; t <= lm; ++t) {
                    double& x = win[((j + t) % Wf) * INV_COLS + lane];
                    x += ab[(size_t)(kd + t) + (size_t)j * ldab] * temp;
                }
            }
        }
        // row j is final for the forward pass; row j+kl+1 enters the window
        const double yj = win[(j % Wf) * INV_COLS + lane];
        if (active) X[(size_t)j * nn + c] = yj;
        const int enter = j + Wf;
        win[(j % Wf) * INV_COLS + lane] = (enter == c) ? 1.0 : 0.0;
    }
    __syncthreads();
    // ---- backward: U^-1 y, window rows [j-k, j] ---------------------------
    const int k = kl + ku;
    const int Wb = k + 1;
    for (int t = 0; t < Wb && t < n; ++t) {
        const int row = n - 1 - t;
        win[(row % Wb) * INV_COLS + lane] = active ? X[(size_t)row * nn + c] : 0.0;
    }
    for (int j = n - 1; j >= 0; --j) {
        double bj = win[(j % Wb) * INV_COLS + lane];
        if (bj != 0.0) {
            bj = bj / ab[(size_t)k + (size_t)j * ldab];
            const int i0 = j - k > 0 ? j - k : 0;
            for (int i = j - 1; i >= i0; --i) {
                double& x = win[(i % Wb) * INV_COLS + lane];
                x -= bj * ab[(size_t)(k + i - j) + (size_t)j * ldab];
            }
        }
        if (active) X[(size_t)j * nn + c] = bj;
        const int enter = j - Wb;
        if (enter >= 0) win[(j % Wb) * INV_COLS + lane] = active ? X[(size_t)enter * nn + c] : 0.0;
    }
}

// ---------------------------------------------------------------------------
// Explicit inverse from the DGBTF2 factors by blocks of CB rows, CB columns
// of the inverse per workgroup.
//
// Bound: the chain of 2 n / CB blocks.  With a lane per column each of the 2 n
// rows was a step of its own, with the band's whole width on one wavefront
// (34 of them at 2145 columns, 2.0 and 3.9 us a row).  Here a row block takes
// its contributions from the other blocks as 16x16 FP64 matrix products on
// four wavefronts, and only the 16x16 triangle is solved row by row, in
// registers.
//
// k_pack_factors lays the factors out by block once: for block I
//   [0, KB * 256)       -U(I, I + kb), kb = 1..KB, in the products' lane order
//   + 256, + 256        U(I, I) (identity past n), unit-lower L(I, I) by rows
//   + RB * 256          -L of the RB row blocks below, in lane order
//   + CB                reciprocals of U's diagonal
//   + PK_PERM           the rows' order after the block's swaps (ints)
// with L's rows in that order, so that a block's CB interchange-and-eliminate
// steps are one gather, a triangle and RB products.
//
// Forward: y = L^-1 P e_c over a window of (RB + 1) * CB rows in LDS; rows
// above the workgroup's first column - kl stay zero.  Backward: wavefront 0
// adds the nearest block's product and solves the triangle of block I while
// the other three form what block I - 1 needs of the blocks beyond; one
// barrier a block.  Measured, columns and bandwidth: 2145, 66 10.7 -> 0.51 ms;
// 897, 46 4.50 -> 0.21; 280, 28 0.73 -> 0.08; 81, 18 0.22 -> 0.03.  The rms of
// A X - I in extended precision is 10% smaller on average than the row-wise
// kernels' (15 biharmonic operators of these sizes, -27 to +2%).
// ---------------------------------------------------------------------------
constexpr int PK_PERM = LU_RW / 2;
__host__ __device__ constexpr int pk_kb(int kd) { return (kd + CB - 1) / CB; }
__host__ __device__ constexpr int pk_rb(int kl) { return (kl + CB - 1) / CB; }
__host__ __device__ constexpr size_t pk_size(int kl, int kd)
{
    return (size_t)(pk_kb(kd) + 2 + pk_rb(kl)) * 256 + CB + PK_PERM;
}

__global__ __launch_bounds__(256) void k_pack_factors(const double* __restrict__ ab, int ldab, int n, int kl, int ku,
                                                      const int32_t* __restrict__ ipiv, double* __restrict__ pk)
{
    __shared__ double Lp[CB][LU_RW];
    __shared__ int perm[LU_RW];
    const int tid = threadIdx.x, kd = kl + ku, KB = pk_kb(kd), RB = pk_rb(kl);
    const int j0 = blockIdx.x * CB;
    double* o = pk + blockIdx.x * pk_size(kl, kd);
    auto U = [&](int r, int c) -> double {
        return (r < n && c < n && c >= r && c - r <= kd) ? ab[(size_t)(kd + r - c) + (size_t)c * ldab] : 0.0;
    };
    for (int e = tid; e < KB * 256; e += 256) {
        const int l = e & 63, st = (e >> 6) & 3, kb = (e >> 8) + 1;
        o[e] = -U(j0 + (l & 15), j0 + CB * kb + 4 * st + (l >> 4));
    }
    {
        const int r = tid >> 4, c = tid & 15;
        o[KB * 256 + tid] = (j0 + r < n) ? U(j0 + r, j0 + c) : (r == c ? 1.0 : 0.0);
    }
    for (int r = tid; r < LU_RW; r += 256) perm[r] = r;
    for (int e = tid; e < CB * LU_RW; e += 256) {
        const int q = e / LU_RW, r = e % LU_RW, j = j0 + q;
        Lp[q][r] = (j < n && j0 + r < n && r > q && r - q <= kl) ? ab[(size_t)(kd + r - q) + (size_t)j * ldab] : 0.0;
    }
    __syncthreads();
    // the later swaps of the block, on the order and on the columns before
    for (int q = 0; q < CB && j0 + q < n - 1; ++q) {
        const int p = ipiv[j0 + q] - 1 - j0;
        if (p != q && p > q && p < LU_RW) {
            if (tid == CB) {
                const int t = perm[q];
                perm[q] = perm[p];
                perm[p] = t;
            } else if (tid < q) {
                const double t = Lp[tid][q];
                Lp[tid][q] = Lp[tid][p];
                Lp[tid][p] = t;
            }
        }
        __syncthreads();
    }
    double* oL = o + (KB + 1) * 256;
    oL[tid] = (tid >> 4) > (tid & 15) ? Lp[tid & 15][tid >> 4] : 0.0;
    for (int e = tid; e < RB * 256; e += 256) {
        const int l = e & 63, st = (e >> 6) & 3, rb = e >> 8;
        oL[256 + e] = -Lp[4 * st + (l >> 4)][CB * (rb + 1) + (l & 15)];
    }
    double* oR = oL + 256 + RB * 256;
    if (tid < CB) oR[tid] = (j0 + tid < n) ? 1.0 / U(j0 + tid, j0 + tid) : 1.0;
    int* oP = reinterpret_cast<int*>(oR + CB);
    for (int r = tid; r < LU_RW; r += 256) oP[r] = perm[r];
}

__global__ __launch_bounds__(256) void k_inv_blocks(const double* __restrict__ pk, int n, int kl, int ku,
                                                    double* __restrict__ X)
{
    // forward: two windows of LU_RW rows; backward: 16 blocks of x
    __shared__ double buf[16 * 256];
    __shared__ double part[2][3][256];
    __shared__ double tri[2][256 + CB];
    __shared__ double ys[256];
    __shared__ int perm[2][LU_RW];
    static_assert(2 * LU_RW * CB <= 16 * 256, "both windows fit");
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, m = lane & 15;
    const int kd = kl + ku, KB = pk_kb(kd), RB = pk_rb(kl), nblk = (n + CB - 1) / CB;
    const size_t psz = pk_size(kl, kd);
    const int c0 = blockIdx.x * CB, c = c0 + m;
    const bool col = c < n;
    auto row_at = [&](int r) -> double* { return X + (size_t)r * n + c; };

    // ---- forward --------------------------------------------------------------
    const int J0 = (c0 > kl ? c0 - kl : 0) / CB;
    for (int r = tid >> 4; r < J0 * CB; r += CB)
        if (col) *row_at(r) = 0.0;
    double* Yc = buf;
    double* Yn = buf + LU_RW * CB;
    for (int e = tid; e < LU_RW * CB; e += 256) Yc[e] = (J0 * CB + e / CB == c0 + e % CB) ? 1.0 : 0.0;
    const double* pL = pk + (size_t)J0 * psz + (KB + 1) * 256;
    tri[0][tid] = pL[tid];
    if (tid < LU_RW) perm[0][tid] = reinterpret_cast<const int*>(pL + 256 + RB * 256 + CB)[tid];
    double a[2][4];
    auto load_l = [&](const double* p, double (&d)[2][4]) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                const int rb = wv + 4 * u;
                d[u][st] = rb < RB ? p[256 + rb * 256 + st * 64 + lane] : 0.0;
            }
    };
    load_l(pL, a);
    __syncthreads();
    for (int J = J0; J < nblk; ++J) {
        const int par = (J - J0) & 1;
        // the next block's factors, on their way while this one is solved
        const double* pn = pL + (J + 1 < nblk ? psz : 0);
        double an[2][4];
        load_l(pn, an);
        const double tn = pn[tid];
        const int permn = tid < LU_RW ? reinterpret_cast<const int*>(pn + 256 + RB * 256 + CB)[tid] : 0;
        if (wv == 0) {
            double w[CB];
#pragma unroll
            for (int q = 0; q < CB; ++q) w[q] = Yc[perm[par][q] * CB + m];
#pragma unroll
            for (int q = 0; q < CB; ++q)
#pragma unroll
                for (int r = q + 1; r < CB; ++r) w[r] = __builtin_fma(-tri[par][r * CB + q], w[q], w[r]);
            if (g == 0) {
#pragma unroll
                for (int q = 0; q < CB; ++q) ys[q * CB + m] = w[q];
            }
        }
        tri[par ^ 1][tid] = tn;
        if (tid < LU_RW) perm[par ^ 1][tid] = permn;
        __syncthreads();
        {
            const int r = 4 * wv + g;
            if (col && J * CB + r < n) *row_at(J * CB + r) = ys[r * CB + m];
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int rb = wv + 4 * u;
            if (rb < RB) {
                v4d acc;
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] = Yc[perm[par][CB * (rb + 1) + 4 * v + g] * CB + m];
#pragma unroll
                for (int st = 0; st < 4; ++st) acc = mfma4(a[u][st], ys[(4 * st + g) * CB + m], acc);
#pragma unroll
                for (int v = 0; v < 4; ++v) Yn[(CB * rb + 4 * v + g) * CB + m] = acc[v];
            }
        }
        // the entering rows
        {
            const int r = CB * RB + 4 * wv + g;
            Yn[r * CB + m] = ((J + 1) * CB + r == c) ? 1.0 : 0.0;
        }
        __syncthreads();
        double* t = Yc;
        Yc = Yn;
        Yn = t;
        pL = pn;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int st = 0; st < 4; ++st) a[u][st] = an[u][st];
    }

    // ---- backward -------------------------------------------------------------
    for (int e = tid; e < 16 * 256; e += 256) buf[e] = 0.0;
    for (int e = tid; e < 2 * 3 * 256; e += 256) (&part[0][0][0])[e] = 0.0;
    // block b's triangle and reciprocals; block b's rows of y; the products'
    // factors: wavefront 0 takes kb = 1, the others kb = 2.. in turn
    constexpr int FAR = 3;
    auto load_tri = [&](int b, int i) {
        return i < 256 ? pk[(size_t)b * psz + KB * 256 + i]
                       : pk[(size_t)b * psz + (size_t)(KB + 2 + RB) * 256 + (i - 256)];
    };
    double ua[FAR][4];
    auto load_u = [&](int b, double (&d)[FAR][4]) {
#pragma unroll
        for (int u = 0; u < FAR; ++u)
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                const int kb = wv == 0 ? (u == 0 ? 1 : KB + 1) : 1 + wv + 3 * u;
                d[u][st] = (b >= 0 && kb <= KB) ? pk[(size_t)b * psz + (size_t)(kb - 1) * 256 + st * 64 + lane] : 0.0;
            }
    };
    auto load_y = [&](int b, v4d& y) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = b * CB + 4 * v + g;
            y[v] = (b >= 0 && r < n && col) ? *row_at(r) : 0.0;
        }
    };
    // (the far products of step I are block I - 1's)
    const int I0 = nblk - 1;
    load_u(wv == 0 ? I0 : I0 - 1, ua);
    v4d y = {0.0, 0.0, 0.0, 0.0};
    if (wv == 0) load_y(I0, y);
    tri[I0 & 1][tid] = load_tri(I0, tid);
    if (tid < CB) tri[I0 & 1][256 + tid] = load_tri(I0, 256 + tid);
    __syncthreads();
    for (int I = I0; I >= 0; --I) {
        const int par = I & 1;
        double un[FAR][4];
        load_u((wv == 0 ? I : I - 1) - 1, un);
        if (wv == 0) {
            v4d yn;
            load_y(I - 1, yn);
            v4d acc = y;
#pragma unroll
            for (int v = 0; v < 4; ++v)
                acc[v] += (part[par][0][(4 * v + g) * CB + m] + part[par][1][(4 * v + g) * CB + m]) +
                          part[par][2][(4 * v + g) * CB + m];
            const double* xb = buf + ((I + 1) & 15) * 256;
#pragma unroll
            for (int st = 0; st < 4; ++st) acc = mfma4(ua[0][st], xb[(4 * st + g) * CB + m], acc);
#pragma unroll
            for (int v = 0; v < 4; ++v) ys[(4 * v + g) * CB + m] = acc[v];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            double w[CB];
#pragma unroll
            for (int q = 0; q < CB; ++q) w[q] = ys[q * CB + m];
            const double* T = tri[par];
#pragma unroll
            for (int r = CB - 1; r >= 0; --r) {
                w[r] = div_by(w[r], T[r * CB + r], T[256 + r]);
#pragma unroll
                for (int q = 0; q < r; ++q) w[q] = __builtin_fma(-T[q * CB + r], w[r], w[q]);
            }
            if (g == 0) {
                double* xo = buf + (I & 15) * 256;
#pragma unroll
                for (int q = 0; q < CB; ++q) xo[q * CB + m] = w[q];
            }
            y = yn;
        } else {
            const int t = tid - 64;  // 0..191
            if (I > 0) {
                const double t0 = load_tri(I - 1, t), t1 = t < 64 + CB ? load_tri(I - 1, 192 + t) : 0.0;
                v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int u = 0; u < FAR; ++u) {
                    const int kb = 1 + wv + 3 * u;
                    if (kb <= KB) {
                        const double* xb = buf + ((I - 1 + kb) & 15) * 256;
#pragma unroll
                        for (int st = 0; st < 4; ++st) acc = mfma4(ua[u][st], xb[(4 * st + g) * CB + m], acc);
                    }
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) part[par ^ 1][wv - 1][(4 * v + g) * CB + m] = acc[v];
                tri[par ^ 1][t] = t0;
                if (t < 64 + CB) tri[par ^ 1][192 + t] = t1;
            }
            // the block before this one is final
            for (int e = t; e < 256 && I < I0; e += 192) {
                const int r = (I + 1) * CB + (e >> 4), cc = c0 + (e & 15);
                if (r < n && cc < n) X[(size_t)r * n + cc] = buf[((I + 1) & 15) * 256 + e];
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < FAR; ++u)
#pragma unroll
            for (int st = 0; st < 4; ++st) ua[u][st] = un[u][st];
    }
    {
        const int r = tid >> 4;
        if (r < n && col) X[(size_t)r * n + c] = buf[tid];
    }
}

// Coarse solve: B(p) = RHS(grids,i,k)*R(p) on interior rows (0 on walls),
// x = A^-1 B, error(grids) <- x on the interior with the ghost mirrors of
// enforceBCs_stream (walls stay 0).  One workgroup per interior row.
__global__ __launch_bounds__(256) void k_coarse_apply(const double* __restrict__ Ainv, const double* __restrict__ RowB,
                                                      const double* __restrict__ rhs, double* __restrict__ E, Grid g,
                                                      int n, double zsg)
{
    const int nxc = g.nx, nzc = g.nz, N = nzc + 1;
    const int ip = blockIdx.x + 1, kp = blockIdx.y + 1;  // interior unknown
    const int prow = N * ip + kp;                         // 0-based row of A^-1
    const double* row = Ainv + (size_t)prow * (size_t)n;
    double acc = 0.0;
    for (int q = threadIdx.x; q < n; q += blockDim.x) {
        const int kq = q % N, iq = q / N;
        if (iq > 0 && iq < nxc && kq > 0 && kq < nzc) acc += row[q] * (rhs[g.at(iq, kq)] * RowB[q]);
    }
    acc = block_sum(acc);
    if (threadIdx.x == 0) {
        E[g.at(ip, kp)] = acc;
        stream_ghosts(E, g, ip, kp, acc, zsg);
    }
}

// Coarse solve by banded substitution with the DGBTF2 factors (DGBTRS 'N',
// iterative_solver.f90:139-142): one workgroup, the solution vector in LDS,
// one barrier per substitution step.
__global__ __launch_bounds__(256) void k_coarse_lusolve(const double* __restrict__ ab, int ldab, int n, int kl, int ku,
                                                        const int32_t* __restrict__ ipiv,
                                                        const double* __restrict__ RowB, const double* __restrict__ rhs,
                                                        double* __restrict__ E, Grid g, double zsg)
{
    extern __shared__ double b[];
    const int tid = threadIdx.x, nt = blockDim.x;
    const int nxc = g.nx, nzc = g.nz, N = nzc + 1;
    for (int q = tid; q < n; q += nt) {
        const int kq = q % N, iq = q / N;
        b[q] = (iq > 0 && iq < nxc && kq > 0 && kq < nzc) ? rhs[g.at(iq, kq)] * RowB[q] : 0.0;
    }
    __syncthreads();
    const int kd = ku + kl;
    for (int j = 0; j < n - 1; ++j) {
        const int lm = kl < n - 1 - j ? kl : n - 1 - j;
        const int l = ipiv[j] - 1;
        double bj;
        if (l != j) {
            const double bl = b[l], bjj = b[j];
            __syncthreads();
            if (tid == 0) { b[l] = bjj; b[j] = bl; }
            bj = bl;
        } else {
            bj = b[j];
        }
        __syncthreads();
        if (bj != 0.0) {
            const double temp = -1.0 * bj;
            for (int t = 1 + tid; t <= lm; t += nt) b[j + t] += ABx(kd + t, j) * temp;
        }
        __syncthreads();
    }
    const int k = kl + ku;
    for (int j = n - 1; j >= 0; --j) {
        double bj = b[j];
        if (bj != 0.0) {
            bj = bj / ABx(k, j);
            const int i0 = j - k > 0 ? j - k : 0;
            for (int i = j - 1 - tid; i >= i0; i -= nt) b[i] -= bj * ABx(k + i - j, j);
        }
        __syncthreads();
        if (tid == 0) b[j] = bj;
        __syncthreads();
    }
    for (int q = tid; q < n; q += nt) {
        const int kq = q % N, iq = q / N;
        if (iq > 0 && iq < nxc && kq > 0 && kq < nzc) {
            E[g.at(iq, kq)] = b[q];
            stream_ghosts(E, g, iq, kq, b[q], zsg);
        }
    }
}

#undef ABx

void launch_coarse_lusolve(hipStream_t st, const double* ab, int ldab, int n, int kl, int ku, const int32_t* ipiv,
                           const double* RowB, const Level& L, double* E, double zsg)
{
    hipLaunchKernelGGL(k_coarse_lusolve, dim3(1), dim3(256), sizeof(double) * (size_t)n, st, ab, ldab, n, kl, ku, ipiv,
                       RowB, L.rhs, E, L.g, zsg);
}

void launch_coarse_assemble(hipStream_t st, double* Mc, double* RowB, const Level& L, const FD& F, const Spacing& h,
                            int ivis, int Vbc, int kl, int ku, int ngc)
{
    hipLaunchKernelGGL(k_coarse_assemble, dim3((ngc + 255) / 256), dim3(256), 0, st, Mc, RowB, L.vis, L.visx, L.visz,
                       L.visxx, L.viszz, L.visxz, L.g, F, h, ivis, Vbc, kl, ku, ngc);
}

void launch_dgbtf2(hipStream_t st, double* ab, int ldab, int n, int kl, int ku, int32_t* ipiv, int32_t* info)
{
    if (coarse_blocked(kl, ku)) {
        const size_t lds = sizeof(double) * LU_CS * LU_RS;
        auto go = [&](auto* k) {
            hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            hipLaunchKernelGGL(k, dim3(1), dim3(LU_THREADS), lds, st, ab, ldab, n, kl, ku, ipiv, info);
        };
        if (CB + kl <= 64) go(k_lu_panels<1>);
        else go(k_lu_panels<2>);
    } else {
        hipLaunchKernelGGL(k_dgbtf2, dim3(1), dim3(256), 0, st, ab, ldab, n, kl, ku, ipiv, info);
    }
}

size_t band_inverse_scratch(int n, int kl, int ku)
{
    return coarse_blocked(kl, ku) ? (size_t)((n + CB - 1) / CB) * pk_size(kl, kl + ku) : 1;
}

void launch_band_inverse(hipStream_t st, const double* ab, int ldab, int n, int kl, int ku, const int32_t* ipiv,
                         double* Ainv, double* scratch)
{
    if (coarse_blocked(kl, ku)) {
        const dim3 blocks((n + CB - 1) / CB);
        hipLaunchKernelGGL(k_pack_factors, blocks, dim3(256), 0, st, ab, ldab, n, kl, ku, ipiv, scratch);
        hipLaunchKernelGGL(k_inv_blocks, blocks, dim3(256), 0, st, scratch, n, kl, ku, Ainv);
        return;
    }
    // wide bands: one lane per column with an LDS window of kl+ku+1 rows
    const size_t row_bytes = sizeof(double) * (size_t)(kl + ku + 1);
    if (64 * row_bytes <= 65536)
        hipLaunchKernelGGL((k_band_inverse<64>), dim3((n + 63) / 64), dim3(64), 64 * row_bytes, st, ab, ldab, n, kl, ku,
                           ipiv, Ainv);
    else if (32 * row_bytes <= 65536)
        hipLaunchKernelGGL((k_band_inverse<32>), dim3((n + 31) / 32), dim3(32), 32 * row_bytes, st, ab, ldab, n, kl, ku,
                           ipiv, Ainv);
    else if (16 * row_bytes <= 65536)
        hipLaunchKernelGGL((k_band_inverse<16>), dim3((n + 15) / 16), dim3(16), 16 * row_bytes, st, ab, ldab, n, kl, ku,
                           ipiv, Ainv);
    else
        hipLaunchKernelGGL((k_band_inverse<8>), dim3((n + 7) / 8), dim3(8), 8 * row_bytes, st, ab, ldab, n, kl, ku, ipiv,
                           Ainv);
}

void launch_coarse_apply(hipStream_t st, const double* Ainv, const double* RowB, const Level& L, double* E, int ngc,
                         double zsg)
{
    hipLaunchKernelGGL(k_coarse_apply, dim3(L.g.nx - 1, L.g.nz - 1), dim3(256), 0, st, Ainv, RowB, L.rhs, E, L.g, ngc,
                       zsg);
}

}  // namespace tc
