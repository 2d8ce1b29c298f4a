// libmusic_hip: Ewald real-space node sums of an orthorhombic cell.
//
// Two routes, both in FP64:
//   * direct: every atom for every node (FP64 maps, the reference's sum);
//   * near + far (FP32 maps): the grid is cut into tiles of SB^3 nodes.  For
//     each tile the atoms within R0 = 1.4 a of the tile's box (a = its half
//     edge), and those whose minimum image changes inside the box, are summed
//     node by node; the field of the others up to the real-space cutoff is
//     smooth in the box, so it is summed at FP^3 Chebyshev points only and
//     interpolated to the nodes axis by axis.  The nearest singularity of a
//     far atom's field lies at 2.4 a from the box centre: the interpolation
//     converges as 4.6^-FP, 1e-9 of V and 1e-7 of the derivatives for FP = 16,
//     below the rounding of the FP32 values stored in the map.
// The reference differentiates erfc exactly but evaluates it with the A&S
// 7.1.26 fit (ewald.F90:874-916): the far field is therefore carried twice,
// with the A&S erfc (for V) and with erfc to 1e-12 (whose interpolant is
// differentiated); the derivative terms differ from the reference's by the
// fit's 1.5e-7 / r^2 alone.
#include <cmath>
#include <cstring>
#include <vector>

#include "mh_device.h"
#include "mh_internal.h"

namespace mh {

constexpr int FP = 16;            // Chebyshev points per axis
constexpr int FPV = FP * FP * FP;
constexpr int FDEG = 12;          // degree of the erfcx fit
constexpr int FCH = 32;           // far atoms staged per pass
constexpr double kFarZ0 = 2.4;    // (a + R0) / a
constexpr double kEwTokcal = 332.064;   // ewald.F90:60
constexpr double kEwVeryLrg = 1.0e10;   // mapmaker.F90:57
constexpr double kEwLowCut2 = 1.0e-6;   // ewald.F90:361-362

struct EwP {
    int n[3];            // grid nodes
    int natoms;
    double step[3], L[3];
    double kappa, kappa2, pk, twoksp, charge1;
    int refold;          // separations folded per node
    // tiles
    int SB, nt[3], nsplit;
    double rc2, r02;
    double half[3], ihalf[3];  // half edges of a tile's box and their inverses
    double xk[FP];       // Chebyshev points on [-1, 1]
    double tc, ith;      // erfcx fit variable (t - tc) * ith
    double fit[FDEG + 1];
};

// 1/sqrt(x) and 1/x: the hardware's 24-bit approximations and one Newton
// step (about 5e-15), without the scaling and rounding steps of the IEEE
// division that the pair sums do not need
__device__ __forceinline__ double rsq_nr(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y), y, 1.0);
    return fma(0.5 * y, e, y);
}
__device__ __forceinline__ double rcp_nr(double x) {
    const double y = __builtin_amdgcn_rcp(x);
    return fma(y, fma(-x, y, 1.0), y);
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

// near (front, count[2 t]) and far (back, count[2 t + 1]) atoms of each tile,
// in atom order from their end of list[t][natoms]; one workgroup per tile
__global__ void __launch_bounds__(256) k_ew_lists(EwP p, const double *__restrict__ xyz, int *__restrict__ list,
                                                  int *__restrict__ count) {
    __shared__ int s_w[2][4];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tix[3] = {t % p.nt[0], (t / p.nt[0]) % p.nt[1], t / (p.nt[0] * p.nt[1])};
    double cen[3];
    for (int d = 0; d < 3; d++) cen[d] = (double)(tix[d] * p.SB) * p.step[d] + p.half[d];
    int nn = 0, nf = 0;
    int *l = list + (long long)t * p.natoms;
    for (int a0 = 0; a0 < p.natoms; a0 += 256) {
        const int a = a0 + tid;
        int cls = 0;  // 1 near, 2 far
        if (a < p.natoms) {
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

// Far field at the Chebyshev points: F[split][tile][field][z][y][x], field 0
// with the A&S erfc, 1 with erfc.  A lane owns the 16 points of one (x, y)
// line.  The Gaussian factor e^{-kappa^2 r^2} is a product of three per-axis
// factors formed once per atom (48 exponentials for 4096 points), so a point
// costs r^-1, the A&S t and two polynomials: about 43 FP64 instructions, the
// bound of this kernel (FP64 issue rate, no HBM traffic to speak of).
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
                const double ri = rsq_nr(r2);
                const double tt = rcp_nr(fma(p.pk, r2 * ri, 1.0));
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
// Bound by the FP64 issue rate of the near pairs (about 70 instructions each).
template <int NZ, bool FAR>
__global__ void __launch_bounds__(256, NZ == 4 ? 3 : 4) k_ew_nodes(EwP p, const double *__restrict__ xyz,
                                                     const double *__restrict__ q, const int *__restrict__ list,
                                                     const int *__restrict__ count, const double *__restrict__ F,
                                                     const double *__restrict__ M /* [2][SB][FP] */,
                                                     const double *__restrict__ recip, float *__restrict__ out32,
                                                     double *__restrict__ out64) {
    __shared__ double s_y[FAR ? 5 * FP * 64 : 1];
    __shared__ double s_x[FAR ? 3 * 4 * FP * 8 : 1];
    constexpr int NCH = FAR ? 32 : 128;  // atoms staged per pass (FAR: three workgroups' LDS on a CU)
    __shared__ double4 s_at[NCH];
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
    const double px = (double)x * p.step[0], py = (double)y * p.step[1];
    double cen[3];  // near separations as (node - c) + fold(c - atom) when no fold can change in the box
    if (FAR) {
        const int tx = t % p.nt[0], ty = (t / p.nt[0]) % p.nt[1], tz = t / (p.nt[0] * p.nt[1]);
        cen[0] = (double)(tx * p.SB) * p.step[0] + p.half[0];
        cen[1] = (double)(ty * p.SB) * p.step[1] + p.half[1];
        cen[2] = (double)(tz * p.SB) * p.step[2] + p.half[2];
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
                    s_x[(f == 0 ? 0 : 4 * FP * 8) + o] = a;
                    if (f == 1) s_x[2 * 4 * FP * 8 + o] = b;
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
                    const double a0 = s_x[c], t0 = s_x[4 * FP * 8 + c], t1 = s_x[2 * 4 * FP * 8 + c];
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
        unsigned failed = 0;
        double pz[NZ];
#pragma unroll
        for (int i = 0; i < NZ; i++) pz[i] = (double)(z0 + zl + i) * p.step[2];
#pragma unroll 1
        for (int c0 = 0; c0 < na; c0 += NCH) {
            const int m = min(NCH, na - c0);
            __syncthreads();
            if (tid < m) {
                const int a = FAR ? list[(long long)t * p.natoms + c0 + tid] : c0 + tid;
                double r[3] = {xyz[3 * a], xyz[3 * a + 1], xyz[3 * a + 2]};
                if (FAR)
                    for (int d = 0; d < 3; d++) r[d] = cen[d] - ew_fold(cen[d] - r[d], p.L[d]);
                s_at[tid] = make_double4(r[0], r[1], r[2], p.charge1 * q[a]);
            }
            __syncthreads();
            if (!act) continue;
#pragma unroll 1
            for (int j = 0; j < m; j++) {
                const double4 at = s_at[j];
                double sx = px - at.x, sy = py - at.y;
                if (!FAR || p.refold) {
                    sx = ew_fold(sx, p.L[0]);
                    sy = ew_fold(sy, p.L[1]);
                }
                const double rxy = fma(sx, sx, sy * sy), sxy = sx * sy;
#pragma unroll
                for (int i = 0; i < NZ; i++) {
                    double sz = pz[i] - at.z;
                    if (!FAR || p.refold) sz = ew_fold(sz, p.L[2]);
                    double r2 = fma(sz, sz, rxy);
                    if (r2 < kEwLowCut2) {  // the node fails; keep the arithmetic finite
                        failed |= 1u << i;
                        r2 = 1.0;
                    }
                    // with u = q erfc / r, g = (2 kappa / sqrt pi) q e^{-k^2 r^2}, w = 1 / r^2:
                    // V = u; -(u + g) w s; (3 (u + g) + 2 k^2 r^2 g) w^2;
                    // -(15 (u + g) + (10 + 4 k^2 r^2) k^2 r^2 g) w^3
                    const double ri = rsq_nr(r2);
                    const double tt = rcp_nr(fma(p.pk, r2 * ri, 1.0));
                    const double k2 = p.kappa2 * r2;
                    const double qe = at.w * exp(-k2);
                    const double u = as_poly(tt) * (qe * ri);
                    const double gg = p.twoksp * qe;
                    const double s1 = u + gg, w = ri * ri, gk = gg * k2;
                    S[i][0] += u;
                    const double t1 = s1 * w;
                    S[i][1] = fma(-t1, sx, S[i][1]);
                    S[i][2] = fma(-t1, sy, S[i][2]);
                    S[i][3] = fma(-t1, sz, S[i][3]);
                    const double w2 = w * w, t2 = fma(2.0, gk, 3.0 * s1) * w2;
                    const double tz = t2 * sz;
                    S[i][4] = fma(t2, sxy, S[i][4]);
                    S[i][5] = fma(tz, sx, S[i][5]);
                    S[i][6] = fma(tz, sy, S[i][6]);
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
            if ((failed >> i) & 1u) {
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

// exp(x^2) erfc(x)
static double erfcx_host(double x) {
    if (x < 5.0) return std::exp(x * x) * std::erfc(x);
    // continued fraction x + (1/2)/(x + 1/(x + (3/2)/(x + ...))), from its tail
    double d = x;
    for (int k = 60; k >= 1; k--) d = x + 0.5 * k / d;
    return 1.0 / (d * std::sqrt(M_PI));
}

// fit of erfcx over [x0, x1] in the variable of the A&S t; false where it
// misses 1e-11 (a range too wide for the degree)
static bool fit_erfcx(double x0, double x1, EwP &p) {
    const double pp = (double)0.3275911f;
    const double ta = 1.0 / (1.0 + pp * x1), tb = 1.0 / (1.0 + pp * x0);
    p.tc = 0.5 * (ta + tb);
    p.ith = 2.0 / (tb - ta);
    auto at = [&](double u) { return (1.0 / (p.tc + u / p.ith) - 1.0) / pp; };
    double f[FDEG + 1], c[FDEG + 1];
    for (int k = 0; k <= FDEG; k++) f[k] = erfcx_host(at(std::cos(M_PI * (k + 0.5) / (FDEG + 1))));
    cheb_series(f, FDEG + 1, c);
    // Chebyshev series to monomials
    double T[2][FDEG + 1], nx[FDEG + 1];
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
    for (int k = 0; k <= 64; k++) {
        const double u = -1.0 + k / 32.0, ex = erfcx_host(at(u));
        double h = p.fit[FDEG];
        for (int i = FDEG - 1; i >= 0; i--) h = h * u + p.fit[i];
        if (!(std::fabs(h - ex) <= 1e-11 * ex)) return false;
    }
    return true;
}

// interpolation from the Chebyshev points to nodes i = 0..SB-1 of a tile:
// M[i][k] values, M[SB + i][k] derivatives on [-1, 1]
static void cheb_matrices(int SB, double *M) {
    for (int i = 0; i < SB; i++) {
        const double xi = SB > 1 ? 2.0 * i / (SB - 1) - 1.0 : 0.0;
        double T[FP], D[FP];  // T_j and T_j' (recurrences)
        T[0] = 1.0, T[1] = xi, D[0] = 0.0, D[1] = 1.0;
        for (int j = 2; j < FP; j++) {
            T[j] = 2.0 * xi * T[j - 1] - T[j - 2];
            D[j] = 2.0 * T[j - 1] + 2.0 * xi * D[j - 1] - D[j - 2];
        }
        for (int k = 0; k < FP; k++) {
            double v = 0.0, d = 0.0;
            for (int j = 0; j < FP; j++) {
                const double w = std::cos(M_PI * j * (k + 0.5) / FP) * (j == 0 ? 1.0 : 2.0) / FP;
                v += w * T[j];
                d += w * D[j];
            }
            M[i * FP + k] = v;
            M[(SB + i) * FP + k] = d;
        }
    }
}

// Estimated FP64 instructions per node of the near + far route for tiles of
// SB^3 nodes: 70 per near pair, 43 per far pair and point, 250 for the
// expansion; the FP32 kernel's direct sum costs 60 per pair and 2500 for its
// FP64 near pairs.
static double far_cost(const EwP &p, const double rc, const double dens, int SB, double *direct) {
    double hs = 0.0, vol = 1.0, nodes = 1.0, tiles = 1.0, e[3];
    for (int d = 0; d < 3; d++) {
        e[d] = (SB - 1) * p.step[d];
        hs = std::max(hs, 0.5 * e[d]);
        tiles *= (p.n[d] + SB - 1) / SB;
        nodes *= p.n[d];
        vol *= e[d];
    }
    const double area = 2.0 * (e[0] * e[1] + e[1] * e[2] + e[0] * e[2]);
    const double edges = e[0] + e[1] + e[2];
    auto grown = [&](double r) { return vol + area * r + M_PI * r * r * edges + 4.0 / 3.0 * M_PI * r * r * r; };
    const double cell = p.L[0] * p.L[1] * p.L[2];
    const double nall = std::min(dens * cell, dens * grown(rc));
    // atoms whose image changes inside the box: slabs of the box's width
    double keep = 1.0;
    for (int d = 0; d < 3; d++)
        if (rc + e[d] >= 0.5 * p.L[d]) keep *= std::max(0.0, 1.0 - e[d] / p.L[d]);
    const double near0 = std::min(nall, dens * grown((kFarZ0 - 1.0) * hs));
    const double near = near0 + (nall - near0) * (1.0 - keep);
    *direct = 2500.0 + 60.0 * std::min(dens * cell, dens * 4.0 / 3.0 * M_PI * rc * rc * rc * 1.25);
    return 250.0 + 70.0 * near + 43.0 * (nall - near) * tiles * FPV / nodes;
}

// Real-space sums of every node of an orthorhombic cell plus the reciprocal
// table: FP64 maps directly, FP32 maps (rc_real > 0) by near pairs and the
// far field.  *done = false (and nothing launched) where the FP32 pair
// kernel is the better route.
int ewald_nodes(mh_ctx *ctx, double charge1, double rc_real, const int np[3], const double step[3],
                const double *recip, float *full32, double *o64, bool *done) {
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
        const bool four = nodes >= 64LL * 4 * 4096;
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
    // tile size: the cheapest estimate
    const double dens = p.natoms / (p.L[0] * p.L[1] * p.L[2]);
    double best = 0.0, direct = 0.0;
    for (int SB : {16, 24, 32, 40}) {
        bool fits = true;  // a box stays well under the single fold of the reference
        for (int d = 0; d < 3; d++) fits = fits && (SB - 1) * step[d] < 0.45 * p.L[d];
        if (!fits) continue;
        const double c = far_cost(p, rc_real, dens, SB, &direct);
        if (p.SB == 0 || c < best) best = c, p.SB = SB;
    }
    if (p.SB == 0 || best > 0.9 * direct) return MH_OK;
    long long tiles = 1;
    double hmax = 0.0, diag2 = 0.0, reach = rc_real;
    for (int d = 0; d < 3; d++) {
        p.nt[d] = (np[d] + p.SB - 1) / p.SB;
        tiles *= p.nt[d];
        p.half[d] = 0.5 * (p.SB - 1) * step[d];
        hmax = std::max(hmax, p.half[d]);
        diag2 += 4.0 * p.half[d] * p.half[d];
        p.ihalf[d] = 1.0 / p.half[d];
    }
    const long long maxlist = 1LL << 27;  // 512 MB of list entries
    if (tiles * p.natoms > maxlist || tiles > (1LL << 22)) return MH_OK;
    const double R0 = (kFarZ0 - 1.0) * hmax;
    p.rc2 = rc_real * rc_real;
    p.r02 = R0 * R0;
    reach += std::sqrt(diag2);
    p.refold = reach >= 0.5 * std::min(p.L[0], std::min(p.L[1], p.L[2])) ? 1 : 0;
    if (!fit_erfcx(p.kappa * R0, p.kappa * (rc_real + std::sqrt(diag2)), p)) return MH_OK;
    for (int k = 0; k < FP; k++) p.xk[k] = std::cos(M_PI * (k + 0.5) / FP);
    // at least 2048 workgroups: eight waves of four on each CU
    p.nsplit = (int)std::max<long long>(1, std::min<long long>(16, (2047 + tiles) / tiles));
    std::vector<double> M(2 * (size_t)p.SB * FP);
    cheb_matrices(p.SB, M.data());
    int rc;
    int *list = (int *)ws_get(ctx, "ewlist", sizeof(int) * tiles * p.natoms, &rc);
    if (rc) return rc;
    int *count = (int *)ws_get(ctx, "ewcount", sizeof(int) * 2 * tiles, &rc);
    if (rc) return rc;
    double *F = (double *)ws_get(ctx, "ewfar", sizeof(double) * 2 * FPV * tiles * p.nsplit, &rc);
    if (rc) return rc;
    double *dM = (double *)ws_get(ctx, "ewcheb", sizeof(double) * M.size(), &rc);
    if (rc) return rc;
    MH_HIP(hipMemcpyAsync(dM, M.data(), sizeof(double) * M.size(), hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_ew_lists, dim3((unsigned)tiles), dim3(256), 0, st, p, xyz, list, count);
    MH_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_ew_far, dim3((unsigned)tiles, (unsigned)p.nsplit), dim3(256), 0, st, p, xyz, q, list, count,
                       F);
    MH_HIP(hipGetLastError());
    const int nb = p.SB / 8;
    hipLaunchKernelGGL((k_ew_nodes<4, true>), dim3((unsigned)(tiles * nb * nb)), dim3(256), 0, st, p, xyz, q, list,
                       count, F, dM, recip, full32, o64);
    MH_HIP(hipGetLastError());
    *done = true;
    return MH_OK;
}

}  // namespace mh
