// libmusic_hip: Ewald real-space node sums of an orthorhombic cell.
//
// Two routes, both in FP64:
//   * direct: every atom for every node (FP64 maps).  The reference's terms,
//     not its rounding: Gaussians as products of three per-axis factors, FMAs,
//     1/r and the A&S t from hardware estimates refined to the last bit.
//     Against long double sums the median error of a node is 4e-16 to 6e-16,
//     as with IEEE square roots and divisions (5e-16 to 6e-16);
//   * near + far (FP32 maps): the grid is cut into tiles of SB^3 nodes.  For
//     each tile the atoms within R0 = 2 a of the tile's box (a = its half
//     edge; 3.5 A at least), and those whose minimum image changes inside the
//     box, are summed node by node; the field of the others up to the
//     real-space cutoff is smooth in the box, so it is summed at FP^3
//     Chebyshev points only and interpolated to the nodes axis by axis
//     (polynomial interpolation at Chebyshev points: Trefethen, Approximation
//     Theory and Approximation Practice, ch. 4 and 8).
//     Tiles of twice the edge do the same for the atoms that are far from
//     them, and pass their polynomial on to the points of their eight tiles,
//     where it is exact.  Along an axis the field of an atom beside the box is
//     singular at +-2i a: the interpolation converges as (2 + sqrt 5)^-FP =
//     4.2^-16 = 1e-10 of that atom's V (atoms ahead of the box: 5.8^-16).
// R0 is what the derivative columns need: against the reference's sums their
// largest errors were 1.6e-6 of a column's rms (mixed second derivatives) with
// 1.4 a, where FP32 pair terms leave 5e-8 to 9e-7.  With 2 a, and 3.5 A for the
// smallest tiles, they are below those of the FP32 pair terms in every column.
// The reference differentiates erfc exactly but evaluates it with the A&S
// 7.1.26 fit (ewald.F90:874-916), so its derivative sums are not the
// derivatives of its V.  The far field is therefore carried twice: with the
// A&S erfc (for V) and as the potential whose first derivative is the
// reference's term exactly (far_h); its second and third derivatives differ
// from the reference's by the fit's own slope, 1e-6 / r^3 and / r^4.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "mh_device.h"
#include "mh_internal.h"

namespace mh {

constexpr int FP = 16;            // Chebyshev points per axis
constexpr int FPV = FP * FP * FP;
constexpr int FDEG = 10;          // degree of the far-field fit
constexpr int FCH = 32;           // far atoms staged per pass
constexpr double kFarR0 = 2.0;    // R0 / a
constexpr double kFarR0Min = 3.5; // least R0 (A)
constexpr double kEwTokcal = 332.064;   // ewald.F90:60
constexpr double kEwVeryLrg = 1.0e10;   // mapmaker.F90:57
constexpr double kEwLowCut2 = 1.0e-6;   // ewald.F90:361-362

struct EwP {
    int n[3];            // grid nodes
    int natoms;
    double step[3], L[3];
    double kappa, kappa2, pk, twoksp, charge1;
    // tiles
    int SB, nt[3], nsplit;
    double rc2, r02;
    double half[3], ihalf[3];  // half edges of a tile's box and their inverses
    double xk[FP];       // Chebyshev points on [-1, 1]
    // bricks with a node near the compaction's cutoff
    float cut, win;
    int bdim[3], *blist, *bflag;
    double tc, ith;      // variable of the far-field fit, (t - tc) * ith
    double fit[FDEG + 1];
};

// 1/sqrt(x) and 1/x: the hardware's 24-bit approximations and one step,
// without the scaling of the IEEE division that the pair sums do not need.
// Newton's step leaves about 5e-15 (FP32 maps), the third-order one the last
// bit (FP64 maps).
template <bool THIRD>
__device__ __forceinline__ double rsq_nr(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y), y, 1.0);
    return THIRD ? fma(y * e, fma(0.375, e, 0.5), y) : fma(0.5 * y, e, y);
}
template <bool THIRD>
__device__ __forceinline__ double rcp_nr(double x) {
    const double y = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, y, 1.0);
    return fma(y, THIRD ? fma(e, e, e) : e, y);
}

// t (a1 + t (a2 + ...)) of A&S 7.1.26 with the reference's single-precision
// coefficients (utils.F90:2090-2101)
__device__ __forceinline__ double as_poly(double t) {
    const double a1 = (double)0.254829592f, a2 = (double)-0.284496736f, a3 = (double)1.421413741f,
                 a4 = (double)-1.453152027f, a5 = (double)1.061405429f;
    return t * fma(t, fma(t, fma(t, fma(t, a5, a4), a3), a2), a1);
}

__device__ __forceinline__ double ew_fold(double d, double L) {
    const double h = 0.5 * L;
    if (d > h) d = d - L;
    else if (d < -h) d = d + L;
    return d;
}

__global__ void k_ew_zero(int n, int *__restrict__ v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] = 0;
}

// near (front, count[2 t]) and far (back, count[2 t + 1]) atoms of each tile,
// in atom order from their end of list[t][natoms]; one workgroup per tile.
// With a parent level (tiles of twice the edge, pt tiles per axis) only the
// atoms near the parent are looked at: the others are in its far field.
__global__ void __launch_bounds__(256) k_ew_lists(EwP p, int ptx, int pty, const int *__restrict__ plist,
                                                  const int *__restrict__ pcount, const double *__restrict__ xyz,
                                                  int *__restrict__ list, int *__restrict__ count) {
    __shared__ int s_w[2][4];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tix[3] = {t % p.nt[0], (t / p.nt[0]) % p.nt[1], t / (p.nt[0] * p.nt[1])};
    double cen[3];
    for (int d = 0; d < 3; d++) cen[d] = (double)(tix[d] * p.SB) * p.step[d] + p.half[d];
    int nn = 0, nf = 0, total = p.natoms;
    const int *src = nullptr;
    if (plist) {
        const long long pt = (tix[0] >> 1) + (long long)ptx * ((tix[1] >> 1) + (long long)pty * (tix[2] >> 1));
        total = pcount[2 * pt];
        src = plist + pt * p.natoms;
    }
    int *l = list + (long long)t * p.natoms;
    for (int a0 = 0; a0 < total; a0 += 256) {
        int a = a0 + tid;
        int cls = 0;  // 1 near, 2 far
        if (a < total) {
            if (src) a = src[a];
            double lb2 = 0.0;
            bool cross = false;
            for (int d = 0; d < 3; d++) {
                const double s = fabs(ew_fold(cen[d] - xyz[3 * a + d], p.L[d]));
                // the image nearest to the box: beyond the fold on its far side
                const double in = fmax(s - p.half[d], 0.0);
                const bool c = s + p.half[d] >= 0.5 * p.L[d] * (1.0 - 1e-12);
                const double wrap = fmax(p.L[d] - s - p.half[d], 0.0);
                const double m = c ? fmin(in, wrap) : in;
                cross |= c;
                lb2 += m * m;
            }
            if (lb2 <= p.rc2) cls = (cross || lb2 <= p.r02) ? 1 : 2;
        }
        const unsigned long long mn = __ballot(cls == 1), mf = __ballot(cls == 2);
        if (lane == 0) {
            s_w[0][wave] = __popcll(mn);
            s_w[1][wave] = __popcll(mf);
        }
        __syncthreads();
        int on = nn, of = nf;
        for (int w = 0; w < 4; w++) {
            if (w < wave) {
                on += s_w[0][w];
                of += s_w[1][w];
            }
            nn += s_w[0][w];
            nf += s_w[1][w];
        }
        const unsigned long long below = (1ull << lane) - 1ull;
        if (cls == 1) l[on + __popcll(mn & below)] = a;
        if (cls == 2) l[p.natoms - 1 - (of + __popcll(mf & below))] = a;
        __syncthreads();
    }
    if (tid == 0) {
        count[2 * t] = nn;
        count[2 * t + 1] = nf;
    }
}

// F of each tile += its parent's polynomial at the tile's points (C[o]: the
// 16 x 16 interpolation matrix of the lower / upper half of an axis): three
// in-place line transforms in LDS, one workgroup per tile.
__global__ void __launch_bounds__(256) k_ew_shift(EwP p, int ptx, int pty, int psplit, long long ptiles,
                                                  const double *__restrict__ PF, const double *__restrict__ C,
                                                  double *__restrict__ F) {
    __shared__ double s_f[FP][FP][FP + 1];
    const int t = blockIdx.x, tid = threadIdx.x, i = tid & (FP - 1), j = tid >> 4;
    const int tix[3] = {t % p.nt[0], (t / p.nt[0]) % p.nt[1], t / (p.nt[0] * p.nt[1])};
    const long long pt = (tix[0] >> 1) + (long long)ptx * ((tix[1] >> 1) + (long long)pty * (tix[2] >> 1));
    for (int f = 0; f < 2; f++) {
        for (int k = 0; k < FP; k++) {
            double v = 0.0;
            for (int s = 0; s < psplit; s++) v += PF[((s * ptiles + pt) * 2 + f) * FPV + k * FP * FP + tid];
            s_f[k][j][i] = v;
        }
        for (int d = 0; d < 3; d++) {
            __syncthreads();
            const double *c = C + (tix[d] & 1) * FP * FP;
            double v[FP];
#pragma unroll
            for (int k = 0; k < FP; k++) v[k] = d == 0 ? s_f[j][i][k] : (d == 1 ? s_f[j][k][i] : s_f[k][j][i]);
#pragma unroll 1
            for (int r = 0; r < FP; r++) {
                double o = 0.0;
#pragma unroll
                for (int k = 0; k < FP; k++) o = fma(c[r * FP + k], v[k], o);
                if (d == 0) s_f[j][i][r] = o;
                else if (d == 1) s_f[j][r][i] = o;
                else F[((long long)t * 2 + f) * FPV + r * FP * FP + tid] += o;
            }
        }
        __syncthreads();
    }
}

// Far field at the Chebyshev points: F[split][tile][field][z][y][x], field 0
// with the A&S erfc, 1 the potential of the derivatives (far_h).  A lane owns the 16 points of one (x, y)
// line.  The Gaussian factor e^{-kappa^2 r^2} is a product of three per-axis
// factors formed once per atom (48 exponentials for 4096 points), so a point
// costs r^-1, the A&S t and two polynomials: about 43 FP64 instructions, the
// bound of this kernel (FP64 issue rate, no HBM traffic to speak of).  334^3
// nodes of the charged 50 A lattice: 2.9 ms for the parents, 2.6 for the tiles.
__global__ void __launch_bounds__(256, 4) k_ew_far(EwP p, const double *__restrict__ xyz, const double *__restrict__ q,
                                                   const int *__restrict__ list, const int *__restrict__ count,
                                                   double *__restrict__ F) {
    __shared__ double2 s_ax[FCH][3][FP];  // (squared separation, Gaussian factor; axis 2 with the charge)
    const int t = blockIdx.x, sp = blockIdx.y, tid = threadIdx.x;
    const int ix = tid & (FP - 1), iy = tid >> 4;
    const int tix[3] = {t % p.nt[0], (t / p.nt[0]) % p.nt[1], t / (p.nt[0] * p.nt[1])};
    double cen[3];
    for (int d = 0; d < 3; d++) cen[d] = (double)(tix[d] * p.SB) * p.step[d] + p.half[d];
    const int nf = count[2 * t + 1];
    const int per = (nf + p.nsplit - 1) / p.nsplit;
    const int f0 = sp * per, f1 = min(nf, f0 + per);
    const int *l = list + (long long)(t + 1) * p.natoms - 1;
    double va[FP], vt[FP];
#pragma unroll
    for (int k = 0; k < FP; k++) va[k] = vt[k] = 0.0;
    for (int c0 = f0; c0 < f1; c0 += FCH) {
        const int m = min(FCH, f1 - c0);
        __syncthreads();
        for (int i = tid; i < m * 3 * FP; i += 256) {
            const int j = i / (3 * FP), r = i - j * 3 * FP, d = r / FP, k = r - d * FP;
            const int a = l[-(c0 + j)];
            const double s = ew_fold(cen[d] - xyz[3 * a + d], p.L[d]) + p.half[d] * p.xk[k];
            const double s2 = s * s;
            double g = exp(-p.kappa2 * s2);
            if (d == 2) g *= p.charge1 * q[a];
            s_ax[j][d][k] = make_double2(s2, g);
        }
        __syncthreads();
        for (int j = 0; j < m; j++) {
            const double2 ax = s_ax[j][0][ix], ay = s_ax[j][1][iy];
            const double rxy = ax.x + ay.x, gxy = ax.y * ay.y;
#pragma unroll
            for (int k = 0; k < FP; k++) {
                const double2 az = s_ax[j][2][k];
                const double r2 = rxy + az.x;
                const double ri = rsq_nr<false>(r2);
                const double tt = rcp_nr<false>(fma(p.pk, r2 * ri, 1.0));
                const double g = (gxy * az.y) * ri;
                const double u = (tt - p.tc) * p.ith;
                double h = p.fit[FDEG];
#pragma unroll
                for (int i = FDEG - 1; i >= 0; i--) h = fma(h, u, p.fit[i]);
                va[k] = fma(as_poly(tt), g, va[k]);
                vt[k] = fma(h, g, vt[k]);
            }
        }
    }
    double *o = F + ((long long)sp * gridDim.x + t) * 2 * FPV + tid;
#pragma unroll
    for (int k = 0; k < FP; k++) {
        o[k * FP * FP] = va[k];
        o[FPV + k * FP * FP] = vt[k];
    }
}

// Node values of 8 x 8 columns: a lane owns a column (x, y) and NZ nodes of
// it at a time (the x, y parts of a pair are shared), the waves take turns
// over the column's groups of NZ nodes.
// FAR: the block covers a column set of one tile; the interpolated far field
// is expanded along x and y into LDS (5 fields: V, dx, dy, value, dxdy), along
// z in registers; the near atoms are the tile's list.  Otherwise the column
// set has 4 groups of NZ nodes (one per wave) and every atom is summed.
// The separations (folded) and the per-axis Gaussian factors of a staged atom
// are formed once per axis position of the block, not per pair.
// Bound by the FP64 issue rate of the near pairs (about 50 instructions each):
// 3.8 ms for 334^3 nodes of the charged 50 A lattice (29 near atoms a node);
// direct, 101^3 nodes of 324 atoms: 0.79 ms.
template <int NZ, bool FAR>
__global__ void __launch_bounds__(256, 3) k_ew_nodes(EwP p, const double *__restrict__ xyz,
                                                     const double *__restrict__ q, const int *__restrict__ list,
                                                     const int *__restrict__ count, const double *__restrict__ F,
                                                     const double *__restrict__ M /* [2][SB][FP] */,
                                                     const double *__restrict__ recip, float *__restrict__ out32,
                                                     double *__restrict__ out64) {
    // atoms staged per pass: per atom 8 x, 8 y and 4 NZ z entries
    // (separation, Gaussian factor; along z with the charge)
    constexpr int NZB = 4 * NZ, NE = 16 + NZB, NCH = 768 / NE;
    __shared__ double s_y[FAR ? 5 * FP * 64 : 1];
    union Scratch {
        double x[FAR ? 3 * 4 * FP * 8 : 1];
        double2 at[NCH][NE];
    };
    __shared__ Scratch s_u;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int x0, y0, z0, zn, na, t = 0;
    if (FAR) {
        const int nb = p.SB / 8, per = nb * nb;
        t = blockIdx.x / per;
        const int b = blockIdx.x - t * per;
        x0 = (t % p.nt[0]) * p.SB + (b % nb) * 8;
        y0 = ((t / p.nt[0]) % p.nt[1]) * p.SB + (b / nb) * 8;
        z0 = (t / (p.nt[0] * p.nt[1])) * p.SB;
        zn = min(p.SB, p.n[2] - z0);
        if (x0 >= p.n[0] || y0 >= p.n[1]) return;
        na = count[2 * t];
    } else {
        const int nbx = (p.n[0] + 7) / 8, nby = (p.n[1] + 7) / 8;
        x0 = (blockIdx.x % nbx) * 8;
        y0 = ((blockIdx.x / nbx) % nby) * 8;
        z0 = (blockIdx.x / (nbx * nby)) * 4 * NZ;
        zn = min(4 * NZ, p.n[2] - z0);
        na = p.natoms;
    }
    const int x = x0 + (lane & 7), y = y0 + (lane >> 3);
    const bool valid = x < p.n[0] && y < p.n[1];
    if (FAR) {
        // x and y stages, four z points at a time
        const long long tiles = (long long)p.nt[0] * p.nt[1] * p.nt[2];
        const int xo = x0 % p.SB, yo = y0 % p.SB;
        const double *M0 = M, *M1 = M + p.SB * FP;
#pragma unroll 1
        for (int zc0 = 0; zc0 < FP; zc0 += 4) {
            {
                // line (field, zc, yc), half of the eight x
                const int ln = tid >> 1, hx = (tid & 1) * 4;
                const int f = ln >> 6, zc = (ln >> 4) & 3, yc = ln & 15;
                double v[FP];
#pragma unroll
                for (int k = 0; k < FP; k++) v[k] = 0.0;
                for (int s = 0; s < p.nsplit; s++) {
                    const double2 *src = reinterpret_cast<const double2 *>(
                        F + (((long long)s * tiles + t) * 2 + f) * FPV + ((zc0 + zc) * FP + yc) * FP);
#pragma unroll
                    for (int k = 0; k < FP / 2; k++) {
                        const double2 w = src[k];
                        v[2 * k] += w.x;
                        v[2 * k + 1] += w.y;
                    }
                }
#pragma unroll 1
                for (int i = 0; i < 4; i++) {
                    const double *m0 = M0 + (xo + hx + i) * FP, *m1 = M1 + (xo + hx + i) * FP;
                    double a = 0.0, b = 0.0;
#pragma unroll
                    for (int k = 0; k < FP; k++) {
                        a = fma(m0[k], v[k], a);
                        b = fma(m1[k], v[k], b);
                    }
                    const int o = (zc * FP + yc) * 8 + hx + i;
                    s_u.x[(f == 0 ? 0 : 4 * FP * 8) + o] = a;
                    if (f == 1) s_u.x[2 * 4 * FP * 8 + o] = b;
                }
            }
            __syncthreads();
            {
                const int zc = wave;  // a wave per z point, a lane per column
                const double *m0 = M0 + (yo + (lane >> 3)) * FP, *m1 = M1 + (yo + (lane >> 3)) * FP;
                double o[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 2
                for (int k = 0; k < FP; k++) {
                    const int c = (zc * FP + k) * 8 + (lane & 7);
                    const double a0 = s_u.x[c], t0 = s_u.x[4 * FP * 8 + c], t1 = s_u.x[2 * 4 * FP * 8 + c];
                    const double u0 = m0[k], u1 = m1[k];
                    o[0] = fma(a0, u0, o[0]);
                    o[1] = fma(t1, u0, o[1]);
                    o[2] = fma(t0, u1, o[2]);
                    o[3] = fma(t0, u0, o[3]);
                    o[4] = fma(t1, u1, o[4]);
                }
                for (int f = 0; f < 5; f++) s_y[(f * FP + zc0 + zc) * 64 + lane] = o[f];
            }
            __syncthreads();
        }
    }
    const int groups = (zn + NZ - 1) / NZ;
#pragma unroll 1
    for (int g0 = 0; g0 < groups; g0 += 4) {
        const int zl = (g0 + wave) * NZ;  // first node of the group in the column (zl >= zn: idle)
        const bool act = zl < zn;
        double S[NZ][8];
#pragma unroll
        for (int i = 0; i < NZ; i++)
            for (int k = 0; k < 8; k++) S[i][k] = 0.0;
        if (FAR && act) {
            const double *M0 = M, *M1 = M + p.SB * FP;
#pragma unroll 1
            for (int k = 0; k < FP; k++) {
                double yv[5];
#pragma unroll
                for (int f = 0; f < 5; f++) yv[f] = s_y[(f * FP + k) * 64 + lane];
#pragma unroll
                for (int i = 0; i < NZ; i++) {
                    const double m0 = M0[(zl + i) * FP + k], m1 = M1[(zl + i) * FP + k];
                    S[i][0] = fma(yv[0], m0, S[i][0]);
                    S[i][1] = fma(yv[1], m0, S[i][1]);
                    S[i][2] = fma(yv[2], m0, S[i][2]);
                    S[i][3] = fma(yv[3], m1, S[i][3]);
                    S[i][4] = fma(yv[4], m0, S[i][4]);
                    S[i][5] = fma(yv[1], m1, S[i][5]);
                    S[i][6] = fma(yv[2], m1, S[i][6]);
                    S[i][7] = fma(yv[4], m1, S[i][7]);
                }
            }
            const double hx = p.ihalf[0], hy = p.ihalf[1], hz = p.ihalf[2];
            const double sc[8] = {1.0, hx, hy, hz, hx * hy, hx * hz, hy * hz, hx * hy * hz};
#pragma unroll
            for (int i = 0; i < NZ; i++)
#pragma unroll
                for (int k = 1; k < 8; k++) S[i][k] *= sc[k];
        }
        double rmin[NZ];
#pragma unroll
        for (int i = 0; i < NZ; i++) rmin[i] = 1.0;
#pragma unroll 1
        for (int c0 = 0; c0 < na; c0 += NCH) {
            const int m = min(NCH, na - c0);
            __syncthreads();
            for (int w = tid; w < m * NE; w += 256) {
                const int j = w / NE, e = w - j * NE;
                const int a = FAR ? list[(long long)t * p.natoms + c0 + j] : c0 + j;
                const int d = e < 8 ? 0 : (e < 16 ? 1 : 2);
                const int node = d == 0 ? x0 + e : (d == 1 ? y0 + e - 8 : z0 + g0 * NZ + e - 16);
                const double s = ew_fold((double)node * p.step[d] - xyz[3 * a + d], p.L[d]);
                double g = exp(-p.kappa2 * (s * s));
                if (d == 2) g *= p.charge1 * q[a];
                s_u.at[j][e] = make_double2(s, g);
            }
            __syncthreads();
            if (!act) continue;
#pragma unroll 1
            for (int j = 0; j < m; j++) {
                const double2 ax = s_u.at[j][lane & 7], ay = s_u.at[j][8 + (lane >> 3)];
                const double rxy = fma(ax.x, ax.x, ay.x * ay.x), sxy = ax.x * ay.x, gxy = ax.y * ay.y;
#pragma unroll
                for (int i = 0; i < NZ; i++) {
                    const double2 az = s_u.at[j][16 + wave * NZ + i];
                    const double sz = az.x, r2 = fma(sz, sz, rxy);
                    rmin[i] = fmin(rmin[i], r2);
                    // with u = q erfc / r, g = (2 kappa / sqrt pi) q e^{-k^2 r^2}, w = 1 / r^2:
                    // V = u; -(u + g) w s; (3 (u + g) + 2 k^2 r^2 g) w^2;
                    // -(15 (u + g) + (10 + 4 k^2 r^2) k^2 r^2 g) w^3
                    const double ri = rsq_nr<!FAR>(r2);
                    const double tt = rcp_nr<!FAR>(fma(p.pk, r2 * ri, 1.0));
                    const double k2 = p.kappa2 * r2;
                    const double qe = gxy * az.y;
                    const double u = as_poly(tt) * (qe * ri);
                    const double gg = p.twoksp * qe;
                    const double s1 = u + gg, w = ri * ri, gk = gg * k2;
                    S[i][0] += u;
                    const double t1 = s1 * w;
                    S[i][1] = fma(-t1, ax.x, S[i][1]);
                    S[i][2] = fma(-t1, ay.x, S[i][2]);
                    S[i][3] = fma(-t1, sz, S[i][3]);
                    const double w2 = w * w, t2 = fma(2.0, gk, 3.0 * s1) * w2;
                    const double tz = t2 * sz;
                    S[i][4] = fma(t2, sxy, S[i][4]);
                    S[i][5] = fma(tz, ax.x, S[i][5]);
                    S[i][6] = fma(tz, ay.x, S[i][6]);
                    const double t3 = fma(fma(4.0, k2, 10.0), gk, 15.0 * s1) * (w2 * w);
                    S[i][7] = fma(-t3 * sz, sxy, S[i][7]);
                }
            }
        }
        if (!act || !valid) continue;
#pragma unroll
        for (int i = 0; i < NZ; i++) {
            const int z = z0 + zl + i;
            if (zl + i >= zn) continue;
            const long long m = (long long)x + (long long)p.n[0] * ((long long)y + (long long)p.n[1] * z);
            const long long s = ((long long)x * p.n[1] + y) * p.n[2] + z;
            double o[8];
            if (rmin[i] < kEwLowCut2) {
                o[0] = kEwVeryLrg;
                for (int k = 1; k < 8; k++) o[k] = 0.0;
            } else {
                const double2 *rp = reinterpret_cast<const double2 *>(recip + 8 * m);
                for (int k = 0; k < 4; k++) {
                    const double2 r = rp[k];
                    o[2 * k] = (S[i][2 * k] + r.x) * kEwTokcal;
                    o[2 * k + 1] = (S[i][2 * k + 1] + r.y) * kEwTokcal;
                }
            }
            if (FAR && fabsf((float)o[0] - p.cut) <= p.win) {
                const int nbx = (p.n[0] + p.bdim[0] - 1) / p.bdim[0], nby = (p.n[1] + p.bdim[1] - 1) / p.bdim[1];
                const int b = x / p.bdim[0] + nbx * (y / p.bdim[1] + nby * (z / p.bdim[2]));
                if (atomicExch(p.bflag + b, 1) == 0) p.blist[1 + atomicAdd(p.blist, 1)] = b;
            }
            float4 *d32 = reinterpret_cast<float4 *>(out32 + 8 * s);
            d32[0] = make_float4((float)o[0], (float)o[1], (float)o[2], (float)o[3]);
            d32[1] = make_float4((float)o[4], (float)o[5], (float)o[6], (float)o[7]);
            if (out64) {
                double2 *d64 = reinterpret_cast<double2 *>(out64 + 8 * s);
                for (int k = 0; k < 4; k++) d64[k] = make_double2(o[2 * k], o[2 * k + 1]);
            }
        }
    }
}

// ------------------------------------------------------------ host side
// coefficients of the degree-(n - 1) interpolant through values f at the n
// Chebyshev points, as a Chebyshev series
static void cheb_series(const double *f, int n, double *c) {
    for (int j = 0; j < n; j++) {
        double s = 0.0;
        for (int k = 0; k < n; k++) s += f[k] * std::cos(M_PI * j * (k + 0.5) / n);
        c[j] = s * (j == 0 ? 1.0 : 2.0) / n;
    }
}

// The potential of the derivative columns: with x = kappa r its pair term is
// q T(x) / r with T(x) = x * integral over y > x of e(y) / y^2 + c e^{-y^2} / y,
// e the A&S erfc and c the reference's 2 / sqrt(pi): d/dr of it is the
// reference's -(u + g) / r.  far_h = e^{x^2} T(x) at the n points x (ascending):
// eight-point Gauss-Legendre sums from point to point and, beyond the last, on
// 16 panels in ln y up to e^{-42}.
static void far_h(const double *x, int n, double *h) {
    static const double gx[4] = {0.1834346424956498, 0.5255324099163290, 0.7966664774136267, 0.9602898564975363};
    static const double gw[4] = {0.3626837833783620, 0.3137066458778873, 0.2223810344533745, 0.1012285362903763};
    const double a[5] = {(double)0.254829592f, (double)-0.284496736f, (double)1.421413741f, (double)-1.453152027f,
                         (double)1.061405429f};
    // integral over ln y in [l0, l1] of e^{x0^2} (e(y) / y + c e^{-y^2})
    auto panel = [&](double l0, double l1, double x0) {
        double s = 0.0;
        for (int k = 0; k < 8; k++) {
            const double y = std::exp(0.5 * (l0 + l1) + 0.5 * (l1 - l0) * (k < 4 ? -gx[k] : gx[k - 4]));
            const double t = 1.0 / (1.0 + (double)0.3275911f * y);
            const double e = t * (a[0] + t * (a[1] + t * (a[2] + t * (a[3] + t * a[4]))));
            s += gw[k & 3] * std::exp(x0 * x0 - y * y) * (e / y + 2.0 * 0.5641896);
        }
        return 0.5 * (l1 - l0) * s;
    };
    double tail = 0.0;
    const double xn = x[n - 1], ln0 = std::log(xn), dl = (0.5 * std::log(xn * xn + 42.0) - ln0) / 16;
    for (int i = 0; i < 16; i++) tail += panel(ln0 + i * dl, ln0 + (i + 1) * dl, xn);
    for (int i = n - 1; i >= 0; i--) {
        if (i < n - 1)
            tail = tail * std::exp(x[i] * x[i] - x[i + 1] * x[i + 1]) + panel(std::log(x[i]), std::log(x[i + 1]), x[i]);
        h[i] = x[i] * tail;
    }
}

// fit of far_h over [x0, x1] in the variable of the A&S t; false where it
// misses 1e-9 (a range too wide for the degree)
static bool fit_far(double x0, double x1, EwP &p) {
    const double pp = (double)0.3275911f;
    const double ta = 1.0 / (1.0 + pp * x1), tb = 1.0 / (1.0 + pp * x0);
    p.tc = 0.5 * (ta + tb);
    p.ith = 2.0 / (tb - ta);
    // the interpolation points and 64 others, x ascending (u descending)
    constexpr int NI = FDEG + 1, NC = 64;
    struct Pt {
        double u;
        int k;  // interpolation point k, or -1
    } pt[NI + NC];
    for (int k = 0; k < NI; k++) pt[k] = {std::cos(M_PI * (k + 0.5) / NI), k};
    for (int k = 0; k < NC; k++) pt[NI + k] = {1.0 - 2.0 * (k + 0.25) / NC, -1};
    std::sort(pt, pt + NI + NC, [](const Pt &l, const Pt &r) { return l.u > r.u; });
    double x[NI + NC], h[NI + NC], f[NI], c[NI];
    for (int k = 0; k < NI + NC; k++) x[k] = (1.0 / (p.tc + pt[k].u / p.ith) - 1.0) / pp;
    far_h(x, NI + NC, h);
    for (int k = 0; k < NI + NC; k++)
        if (pt[k].k >= 0) f[pt[k].k] = h[k];
    cheb_series(f, NI, c);
    // Chebyshev series to monomials
    double T[2][NI], nx[NI];
    std::memset(T, 0, sizeof T);
    for (int i = 0; i <= FDEG; i++) p.fit[i] = 0.0;
    T[0][0] = 1.0;
    T[1][1] = 1.0;
    p.fit[0] += c[0];
    p.fit[1] += c[1];
    for (int j = 2; j <= FDEG; j++) {
        for (int i = 0; i <= FDEG; i++) nx[i] = (i ? 2.0 * T[1][i - 1] : 0.0) - T[0][i];
        std::memcpy(T[0], T[1], sizeof nx);
        std::memcpy(T[1], nx, sizeof nx);
        for (int i = 0; i <= FDEG; i++) p.fit[i] += c[j] * nx[i];
    }
    for (int k = 0; k < NI + NC; k++) {
        double v = p.fit[FDEG];
        for (int i = FDEG - 1; i >= 0; i--) v = v * pt[k].u + p.fit[i];
        if (!(std::fabs(v - h[k]) <= 1e-9 * h[k])) return false;
    }
    return true;
}

// interpolation from the Chebyshev points to n positions xi on [-1, 1]:
// M[i][k] values, D[i][k] derivatives (D may be NULL)
static void cheb_matrix(int n, const double *xi, double *M, double *Dm) {
    double W[FP][FP];  // series coefficient j of the point k's cardinal function
    for (int j = 0; j < FP; j++)
        for (int k = 0; k < FP; k++) W[j][k] = std::cos(M_PI * j * (k + 0.5) / FP) * (j == 0 ? 1.0 : 2.0) / FP;
    for (int i = 0; i < n; i++) {
        const double x = xi[i];
        double T[FP], D[FP];  // T_j and T_j' (recurrences)
        T[0] = 1.0, T[1] = x, D[0] = 0.0, D[1] = 1.0;
        for (int j = 2; j < FP; j++) {
            T[j] = 2.0 * x * T[j - 1] - T[j - 2];
            D[j] = 2.0 * T[j - 1] + 2.0 * x * D[j - 1] - D[j - 2];
        }
        for (int k = 0; k < FP; k++) {
            double v = 0.0, d = 0.0;
            for (int j = 0; j < FP; j++) {
                v += W[j][k] * T[j];
                d += W[j][k] * D[j];
            }
            M[i * FP + k] = v;
            if (Dm) Dm[i * FP + k] = d;
        }
    }
}

// volume of a box of edges e grown by r
static double grown(const double e[3], double r) {
    return e[0] * e[1] * e[2] + 2.0 * (e[0] * e[1] + e[1] * e[2] + e[0] * e[2]) * r +
           M_PI * r * r * (e[0] + e[1] + e[2]) + 4.0 / 3.0 * M_PI * r * r * r;
}

// Expected near and far atoms of a tile of SB^3 nodes with a lattice's uniform
// density dens: the grown box in closed form, the atoms whose image changes
// inside the box (and the far ones) by counting the points of a 16^3 grid over
// the octant of separations of a periodic cell.
static void tile_counts(const EwP &p, double rc, double dens, int SB, double &near, double &far) {
    constexpr int G = 16;
    double m2[3][G], e[3], hs = 0.0;
    bool cross[3][G];
    for (int d = 0; d < 3; d++) {
        e[d] = (SB - 1) * p.step[d];
        const double h = 0.5 * e[d];
        hs = std::max(hs, h);
        for (int i = 0; i < G; i++) {
            const double s = (i + 0.5) / G * 0.5 * p.L[d], in = std::max(s - h, 0.0);
            cross[d][i] = s + h >= 0.5 * p.L[d];
            const double m = cross[d][i] ? std::min(in, std::max(p.L[d] - s - h, 0.0)) : in;
            m2[d][i] = m * m;
        }
    }
    const double r0 = std::max(kFarR0 * hs, kFarR0Min), rc2 = rc * rc, r02 = r0 * r0;
    int nc = 0, nf = 0;
    for (int i = 0; i < G; i++)
        for (int j = 0; j < G; j++)
            for (int k = 0; k < G; k++) {
                const double lb2 = m2[0][i] + m2[1][j] + m2[2][k];
                if (lb2 > rc2 || lb2 <= r02) continue;
                if (cross[0][i] || cross[1][j] || cross[2][k]) nc++;
                else nf++;
            }
    const double all = dens * p.L[0] * p.L[1] * p.L[2];
    near = std::min(all, dens * grown(e, r0)) + all * nc / (G * G * G);
    far = all * nf / (G * G * G);
}

// Estimated time (us) of the near + far route with tiles of SB^3 nodes (and
// parents of (2 SB)^3 with two levels), at least `best` where it is not the
// faster one.  Fitted to 40 maps of 3 to 7 unit cells a side, spacing 0.14 to
// 0.5 A, alpha 0.2 to 0.45, each with every tile size and level (the largest
// deviations are a quarter): the choice loses 2 % on average to the fastest
// one and none of the 40 to the pair kernel.  Tiles of 16 nodes on one level,
// of 32 and of 40 were never the fastest.
static double far_time(const EwP &p, double rc, double dens, int SB, bool two, double best) {
    double near, far, pnear = 0.0, pfar = 0.0, nodes = 1.0, tiles = 1.0, ptiles = 1.0, e[3], hs = 0.0;
    for (int d = 0; d < 3; d++) {
        nodes *= p.n[d];
        tiles *= (p.n[d] + SB - 1) / SB;
        ptiles *= (p.n[d] + 2 * SB - 1) / (2 * SB);
        e[d] = (SB - 1) * p.step[d];
        hs = std::max(hs, 0.5 * e[d]);
    }
    const double all = dens * p.L[0] * p.L[1] * p.L[2];
    // the near atoms of the grown box alone
    near = std::min(all, dens * grown(e, std::max(kFarR0 * hs, kFarR0Min)));
    if (256.0 + 2.6e-6 * nodes * (11.0 + near) >= best) return best;
    tile_counts(p, rc, dens, SB, near, far);
    if (two) {
        tile_counts(p, rc, dens, 2 * SB, pnear, pfar);
        far = std::max(0.0, std::min(near + far, pnear) - near);
    }
    return (two ? 390.0 : 256.0) + 2.6e-6 * nodes * (11.0 + near) + 1.14e-6 * FPV * (tiles * far + ptiles * pfar);
}

// the same of the FP32 pair kernel: the atoms its bricks of bd nodes keep
static double pair_time(const EwP &p, double rc, double dens, const int bd[3]) {
    double e[3], nodes = 1.0;
    for (int d = 0; d < 3; d++) {
        e[d] = (bd[d] - 1) * p.step[d];
        nodes *= p.n[d];
    }
    const double kept = std::min(dens * p.L[0] * p.L[1] * p.L[2], dens * grown(e, rc));
    return 117.0 + 1.33e-6 * nodes * (56.0 + kept);
}

// tiles of SB^3 nodes of the grid in p
static void set_tiles(EwP &p, int SB) {
    double hmax = 0.0;
    p.SB = SB;
    long long tiles = 1;
    for (int d = 0; d < 3; d++) {
        p.nt[d] = (p.n[d] + SB - 1) / SB;
        tiles *= p.nt[d];
        p.half[d] = 0.5 * (SB - 1) * p.step[d];
        p.ihalf[d] = 1.0 / p.half[d];
        hmax = std::max(hmax, p.half[d]);
    }
    const double r0 = std::max(kFarR0 * hmax, kFarR0Min);
    p.r02 = r0 * r0;
    // at least 2048 workgroups: eight waves of four on each CU
    p.nsplit = (int)std::max<long long>(1, std::min<long long>(16, (2047 + tiles) / tiles));
}

// Real-space sums of every node of an orthorhombic cell plus the reciprocal
// table: FP64 maps directly, FP32 maps (rc_real > 0) by near pairs and the
// far field.  *done = false (and nothing launched) where the FP32 pair
// kernel is the better route.  Which nodes a map holds must not depend on
// the route: bricks with a node near the cutoff are listed in cb and take
// the FP32 pair kernel's values (some 70 of 150000 bricks at 334^3 nodes).
int ewald_nodes(mh_ctx *ctx, double charge1, double rc_real, const int np[3], const double step[3],
                const double *recip, float *full32, double *o64, CutBricks &cb, bool *done) {
    EwP p;
    std::memset(&p, 0, sizeof p);
    *done = false;
    for (int d = 0; d < 3; d++) {
        p.n[d] = np[d];
        p.step[d] = step[d];
        p.L[d] = ctx->full_ell[d];
    }
    p.natoms = ctx->natoms;
    p.kappa = ctx->ew.kappa;
    p.kappa2 = p.kappa * p.kappa;
    p.pk = (double)0.3275911f * p.kappa;
    p.twoksp = 2.0 * 0.5641896 * p.kappa;
    p.charge1 = charge1;
    const double *xyz = ctx->xyz.as<double>(), *q = ctx->q.as<double>();
    hipStream_t st = ctx->stream;
    const long long nodes = (long long)np[0] * np[1] * np[2];
    if (rc_real <= 0.0) {
        // four nodes per lane share the x, y parts of a pair; small grids
        // take one, for four times the waves
        const bool four = nodes >= 64LL * 4 * 2048;
        const int nz = four ? 16 : 4;
        const long long nblk = (long long)((np[0] + 7) / 8) * ((np[1] + 7) / 8) * ((np[2] + nz - 1) / nz);
        if (four)
            hipLaunchKernelGGL((k_ew_nodes<4, false>), dim3((unsigned)nblk), dim3(256), 0, st, p, xyz, q,
                               (const int *)nullptr, (const int *)nullptr, (const double *)nullptr,
                               (const double *)nullptr, recip, full32, o64);
        else
            hipLaunchKernelGGL((k_ew_nodes<1, false>), dim3((unsigned)nblk), dim3(256), 0, st, p, xyz, q,
                               (const int *)nullptr, (const int *)nullptr, (const double *)nullptr,
                               (const double *)nullptr, recip, full32, o64);
        MH_HIP(hipGetLastError());
        *done = true;
        return MH_OK;
    }
    // tile size and levels: the cheapest estimate
    const double dens = p.natoms / (p.L[0] * p.L[1] * p.L[2]);
    double best = pair_time(p, rc_real, dens, cb.b);
    int SB = 0;
    bool two = false;
    auto fits = [&](int sb) {  // a box stays well under the single fold of the reference
        bool ok = true;
        for (int d = 0; d < 3; d++) ok = ok && (sb - 1) * step[d] < 0.45 * p.L[d];
        return ok;
    };
    const struct {
        int sb;
        bool two;
    } choice[3] = {{24, false}, {24, true}, {16, true}};
    for (auto &o : choice) {
        if (!fits(o.sb << (o.two ? 1 : 0))) continue;
        const double c = far_time(p, rc_real, dens, o.sb, o.two, best);
        if (c < best) best = c, SB = o.sb, two = o.two;
    }
    if (SB == 0) return MH_OK;
    p.rc2 = rc_real * rc_real;
    set_tiles(p, SB);
    EwP pp = p;
    set_tiles(pp, 2 * SB);
    double diag2 = 0.0;
    for (int d = 0; d < 3; d++) diag2 += 4.0 * (two ? pp : p).half[d] * (two ? pp : p).half[d];
    const long long tiles = (long long)p.nt[0] * p.nt[1] * p.nt[2];
    const long long ptiles = two ? (long long)pp.nt[0] * pp.nt[1] * pp.nt[2] : 0;
    const long long maxlist = 1LL << 27;  // 512 MB of list entries
    if ((tiles + ptiles) * p.natoms > maxlist || tiles > (1LL << 20)) return MH_OK;
    // beyond kappa r = 5.5 the fit runs on under a Gaussian below 1e-13
    if (!fit_far(p.kappa * std::sqrt(p.r02), std::min(5.5, p.kappa * (rc_real + std::sqrt(diag2))), p)) return MH_OK;
    for (int k = 0; k < FP; k++) p.xk[k] = std::cos(M_PI * (k + 0.5) / FP);
    std::memcpy(pp.xk, p.xk, sizeof p.xk);
    std::memcpy(pp.fit, p.fit, sizeof p.fit);
    pp.tc = p.tc;
    pp.ith = p.ith;
    // matrices: tile nodes (values, derivatives), then the two halves of a
    // parent axis
    std::vector<double> xi(SB), M((size_t)2 * SB * FP + 2 * FP * FP);
    for (int i = 0; i < SB; i++) xi[i] = 2.0 * i / (SB - 1) - 1.0;
    cheb_matrix(SB, xi.data(), M.data(), M.data() + (size_t)SB * FP);
    double *C = M.data() + (size_t)2 * SB * FP;
    for (int o = 0; o < 2; o++) {
        double xs[FP];
        // the tile's points on the parent's [-1, 1], in units of the grid step
        const double h0 = 0.5 * (SB - 1), h1 = 0.5 * (2 * SB - 1);
        for (int k = 0; k < FP; k++) xs[k] = (o * SB + h0 * (1.0 + p.xk[k]) - h1) / h1;
        cheb_matrix(FP, xs, C + o * FP * FP, nullptr);
    }
    // one scratch block: matrices, far field, lists, counts, bricks (number,
    // flags, list); where it is not to be had, the pair kernel needs none of it
    const size_t nF = (size_t)2 * FPV * (tiles * p.nsplit + ptiles * pp.nsplit), nl = (size_t)(tiles + ptiles);
    int rc;
    double *dM = (double *)ws_get(ctx, "ewald_far", sizeof(double) * (M.size() + nF) +
                                  sizeof(int) * (nl * p.natoms + 2 * nl + 2 * (size_t)cb.nbricks + 2), &rc);
    if (rc == MH_ENOMEM) return MH_OK;
    if (rc) return rc;
    double *F = dM + M.size();
    int *list = (int *)(F + nF), *count = list + nl * p.natoms, *bl = count + 2 * nl;
    p.blist = bl + cb.nbricks;
    p.bflag = bl;
    p.cut = cb.cut;
    p.win = cb.win;
    for (int d = 0; d < 3; d++) p.bdim[d] = cb.b[d];
    cb.list = p.blist;
    MH_HIP(hipMemcpyAsync(dM, M.data(), sizeof(double) * M.size(), hipMemcpyHostToDevice, st));
    KTimer tfar(ctx, !two ? "ewald_far24" : SB == 24 ? "ewald_far24_two" : "ewald_far16_two");
    int *plist = two ? list + tiles * p.natoms : nullptr, *pcount = two ? count + 2 * tiles : nullptr;
    double *PF = F + (size_t)2 * FPV * tiles * p.nsplit;
    if (two) {
        hipLaunchKernelGGL(k_ew_lists, dim3((unsigned)ptiles), dim3(256), 0, st, pp, 0, 0, (const int *)nullptr,
                           (const int *)nullptr, xyz, plist, pcount);
        hipLaunchKernelGGL(k_ew_far, dim3((unsigned)ptiles, (unsigned)pp.nsplit), dim3(256), 0, st, pp, xyz, q, plist,
                           pcount, PF);
        MH_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_ew_lists, dim3((unsigned)tiles), dim3(256), 0, st, p, pp.nt[0], pp.nt[1],
                       (const int *)plist, (const int *)pcount, xyz, list, count);
    hipLaunchKernelGGL(k_ew_far, dim3((unsigned)tiles, (unsigned)p.nsplit), dim3(256), 0, st, p, xyz, q, list, count,
                       F);
    if (two)
        hipLaunchKernelGGL(k_ew_shift, dim3((unsigned)tiles), dim3(256), 0, st, p, pp.nt[0], pp.nt[1], pp.nsplit,
                           ptiles, PF, dM + (size_t)2 * SB * FP, F);
    MH_HIP(hipGetLastError());
    const int nb = SB / 8;
    hipLaunchKernelGGL(k_ew_zero, dim3((unsigned)((cb.nbricks + 256) / 256)), dim3(256), 0, st, cb.nbricks + 1, bl);
    hipLaunchKernelGGL((k_ew_nodes<4, true>), dim3((unsigned)(tiles * nb * nb)), dim3(256), 0, st, p, xyz, q, list,
                       count, F, dM, recip, full32, o64);
    MH_HIP(hipGetLastError());
    *done = true;
    return MH_OK;
}

}  // namespace mh
