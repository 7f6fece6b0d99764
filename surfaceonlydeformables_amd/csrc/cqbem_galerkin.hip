// Galerkin assembly on gfx950.
//
// Regular (non-touching) face pairs (integrate_galerkin_nonsingular,
// integrator_galerkin.hpp:214-260): the collocation kernels run with every test
// quadrature point as a row that excludes the faces touching its test face, and
// k_gal_project weights the rows by the test basis.  Test faces are taken by
// vertex-disjoint colour classes, so that the row blocks a projection adds into
// are its own within a launch: plain read-modify-write, no atomics, a fixed
// summation order.  The star kernels (k_gal_gh: one lane per test face, source
// vertex and frequency; k_gal_b: one block per test face and frequency) form
// point rows and projection in one; CQBEM_GALERKIN_KERNEL=star selects them.
//
// Touching pairs (Sauter-Schwab, integrator_galerkin.hpp:42-212): one lane per
// direction of the 4D rule (k_gal_touch, k_gal_touch_b), or one lane per point of
// it (k_gal_sing, CQBEM_GALERKIN_SINGULAR=lane), reduced to the pair's corner
// blocks in a per-pair scratch.  A gather kernel then owns each output block and
// adds its pairs' contributions in a fixed order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <stdexcept>
#include <string>
#include <vector>

#include "cqbem_galerkin.hpp"
#include "cqbem_pool.hpp"

namespace cqbem {

namespace {

__device__ inline bool same_v(const Geom &g, int a, int b) { return a == b || (g.vmap != nullptr && g.vmap[a] == g.vmap[b]); }

__device__ inline bool faces_touch(const Geom &g, const int *f1v, int f2) {
    const int b0 = g.F[3 * f2], b1 = g.F[3 * f2 + 1], b2 = g.F[3 * f2 + 2];
    for (int k = 0; k < 3; k++)
        if (same_v(g, f1v[k], b0) || same_v(g, f1v[k], b1) || same_v(g, f1v[k], b2)) return true;
    return false;
}

// ---------------------------------------------------------------------------
// Regular G/H: grid (ceil(nv/64), nl, faces in colour)
// ---------------------------------------------------------------------------
template <bool DG, bool DH>
__global__ void __launch_bounds__(64) k_gal_gh(Geom g, const double4 *__restrict__ quad, int npts,
                                                const Freq *__restrict__ freqs, Mat m, const int *__restrict__ faces,
                                                cd *__restrict__ UG, cd *__restrict__ UH, long long ld, long long lstride) {
    const int j = blockIdx.x * 64 + threadIdx.x;
    const int l = blockIdx.y;
    const int f1 = faces[blockIdx.z];
    if (j >= g.nv) return;
    const Freq f = freqs[l];
    const int tv[3] = {g.F[3 * f1], g.F[3 * f1 + 1], g.F[3 * f1 + 2]};
    const double *X0 = g.V + 3 * tv[0], *X1 = g.V + 3 * tv[1], *X2 = g.V + 3 * tv[2];
    const double tarea = g.area[f1];
    cd ga[3][6], gb[3], hh[3][9];
    for (int k = 0; k < 3; k++) {
        gb[k] = cd{0, 0};
        for (int e = 0; e < 6; e++) ga[k][e] = cd{0, 0};
        for (int e = 0; e < 9; e++) hh[k][e] = cd{0, 0};
    }
    const int t0 = g.vs_ptr[j], t1 = g.vs_ptr[j + 1];
    for (int a = 0; a < npts; ++a) {
        const double4 Qa = quad[a];
        const double x0 = Qa.x * X0[0] + Qa.y * X1[0] + Qa.z * X2[0];
        const double x1 = Qa.x * X0[1] + Qa.y * X1[1] + Qa.z * X2[1];
        const double x2 = Qa.x * X0[2] + Qa.y * X1[2] + Qa.z * X2[2];
        const double wa = Qa.w * tarea;
        cd pa[6], pb = {0, 0}, ph[9];
        for (int e = 0; e < 6; e++) pa[e] = cd{0, 0};
        for (int e = 0; e < 9; e++) ph[e] = cd{0, 0};
        for (int t = t0; t < t1; ++t) {
            const int pk = g.vs_face[t];
            const int fc = pk >> 2, c = pk & 3;
            if (faces_touch(g, tv, fc)) continue;
            const int a0 = g.F[3 * fc], a1 = g.F[3 * fc + 1], a2 = g.F[3 * fc + 2];
            const double *p0 = g.V + 3 * a0, *p1 = g.V + 3 * a1, *p2 = g.V + 3 * a2;
            const double n0 = g.N[3 * fc], n1 = g.N[3 * fc + 1], n2 = g.N[3 * fc + 2];
            const double ar = g.area[fc];
            cd v1[3], v2[3], s2 = {0, 0}, m4[6];
            if (DH) {
                for (int k = 0; k < 3; k++) v1[k] = v2[k] = cd{0, 0};
                for (int k = 0; k < 6; k++) m4[k] = cd{0, 0};
            }
            for (int q = 0; q < npts; ++q) {
                const double4 Q = quad[q];
                const double r0 = Q.x * p0[0] + Q.y * p1[0] + Q.z * p2[0] - x0;
                const double r1 = Q.x * p0[1] + Q.y * p1[1] + Q.z * p2[1] - x1;
                const double r2 = Q.x * p0[2] + Q.y * p1[2] + Q.z * p2[2] - x2;
                const double d2 = r0 * r0 + r1 * r1 + r2 * r2;
                const double ir = rsqrt_nr(d2), r = d2 * ir, ir2 = ir * ir;
                const double h0 = r0 * ir, h1 = r1 * ir, h2 = r2 * ir;
                const double bc = c == 0 ? Q.x : (c == 1 ? Q.y : Q.z);
                const double wL = Q.w * ar * bc;
                const Expo E = expo(r, f);
                if (DG) {
                    cd al, be;
                    g_coef(E, ir, ir2, m, al, be);
                    const double wr = wL * ir;
                    al = al * wr;
                    fma_cr(pb, be, wr);
                    fma_cr(pa[0], al, h0 * h0);
                    fma_cr(pa[1], al, h1 * h1);
                    fma_cr(pa[2], al, h2 * h2);
                    fma_cr(pa[3], al, h0 * h1);
                    fma_cr(pa[4], al, h0 * h2);
                    fma_cr(pa[5], al, h1 * h2);
                }
                if (DH) {
                    cd c1, c2, c4;
                    h_coef(E, ir, ir2, f, m, c1, c2, c4);
                    const double rn = h0 * n0 + h1 * n1 + h2 * n2;
                    c1 = c1 * wL;
                    c2 = c2 * wL;
                    c4 = c4 * (wL * rn);
                    fma_cr(v1[0], c1, h0), fma_cr(v1[1], c1, h1), fma_cr(v1[2], c1, h2);
                    fma_cr(v2[0], c2, h0), fma_cr(v2[1], c2, h1), fma_cr(v2[2], c2, h2);
                    fma_cr(s2, c2, rn);
                    fma_cr(m4[0], c4, h0 * h0);
                    fma_cr(m4[1], c4, h1 * h1);
                    fma_cr(m4[2], c4, h2 * h2);
                    fma_cr(m4[3], c4, h0 * h1);
                    fma_cr(m4[4], c4, h0 * h2);
                    fma_cr(m4[5], c4, h1 * h2);
                }
            }
            if (DH) {
                const double n[3] = {n0, n1, n2};
                for (int p = 0; p < 3; p++)
                    for (int b = 0; b < 3; b++) {
                        cd v = m4[sidx(p, b)];
                        fma_cr(v, v1[p], n[b]);
                        fma_cr(v, v2[b], n[p]);
                        if (p == b) v += s2;
                        ph[p * 3 + b] += v;
                    }
            }
        }
        const double wk[3] = {wa * Qa.x, wa * Qa.y, wa * Qa.z};
        for (int k = 0; k < 3; k++) {
            if (DG) {
                fma_cr(gb[k], pb, wk[k]);
                for (int e = 0; e < 6; e++) fma_cr(ga[k][e], pa[e], wk[k]);
            }
            if (DH)
                for (int e = 0; e < 9; e++) fma_cr(hh[k][e], ph[e], wk[k]);
        }
    }
    for (int k = 0; k < 3; k++) {
        const long long base = (long long)l * lstride + (long long)(3 * tv[k]) * ld + 3 * (long long)j;
        for (int p = 0; p < 3; p++)
            for (int b = 0; b < 3; b++) {
                if (DG) {
                    cd v = ga[k][sidx(p, b)];
                    if (p == b) v += gb[k];
                    UG[base + p * ld + b] += v;
                }
                if (DH) UH[base + p * ld + b] += hh[k][p * 3 + b] * kInv4Pi;
            }
    }
}

__device__ inline double block_sum256(double v, double *red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    const double s = red[0] + red[1] + red[2] + red[3];
    __syncthreads();
    return s;
}

// ---------------------------------------------------------------------------
// Regular B_trans / B_angular: grid (nl, faces in colour), 256 lanes.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_gal_b(Geom g, const double4 *__restrict__ quad, int npts,
                                                const Freq *__restrict__ freqs, Mat m, const int *__restrict__ faces,
                                                cd *__restrict__ Bt, cd *__restrict__ Ba, long long nv3) {
    __shared__ double red[4];
    __shared__ double corner[3][24][2];
    const int l = blockIdx.x;
    const int f1 = faces[blockIdx.y];
    const Freq f = freqs[l];
    const int tv[3] = {g.F[3 * f1], g.F[3 * f1 + 1], g.F[3 * f1 + 2]};
    const double *X0 = g.V + 3 * tv[0], *X1 = g.V + 3 * tv[1], *X2 = g.V + 3 * tv[2];
    const double tarea = g.area[f1];
    if (threadIdx.x < 3 * 24 * 2) (&corner[0][0][0])[threadIdx.x] = 0.0;
    __syncthreads();
    for (int a = 0; a < npts; ++a) {
        const double4 Qa = quad[a];
        const double x0 = Qa.x * X0[0] + Qa.y * X1[0] + Qa.z * X2[0];
        const double x1 = Qa.x * X0[1] + Qa.y * X1[1] + Qa.z * X2[1];
        const double x2 = Qa.x * X0[2] + Qa.y * X1[2] + Qa.z * X2[2];
        cd bt[6], ba[18];
        for (int k = 0; k < 6; k++) bt[k] = cd{0, 0};
        for (int k = 0; k < 18; k++) ba[k] = cd{0, 0};
        for (int fc = threadIdx.x; fc < g.nf; fc += 256) {
            if (faces_touch(g, tv, fc)) continue;
            const int a0 = g.F[3 * fc], a1 = g.F[3 * fc + 1], a2 = g.F[3 * fc + 2];
            const double *p0 = g.V + 3 * a0, *p1 = g.V + 3 * a1, *p2 = g.V + 3 * a2;
            const double n[3] = {g.N[3 * fc], g.N[3 * fc + 1], g.N[3 * fc + 2]};
            const double ar = g.area[fc];
            cd mt[3] = {{0, 0}, {0, 0}, {0, 0}}, m2 = {0, 0}, M[6], S = {0, 0}, S3 = {0, 0};
            for (int k = 0; k < 6; k++) M[k] = cd{0, 0};
            for (int q = 0; q < npts; ++q) {
                const double4 Q = quad[q];
                const double r0 = Q.x * p0[0] + Q.y * p1[0] + Q.z * p2[0] - x0;
                const double r1 = Q.x * p0[1] + Q.y * p1[1] + Q.z * p2[1] - x1;
                const double r2 = Q.x * p0[2] + Q.y * p1[2] + Q.z * p2[2] - x2;
                const double d2 = r0 * r0 + r1 * r1 + r2 * r2;
                const double ir = rsqrt_nr(d2), r = d2 * ir, ir2 = ir * ir;
                const double h[3] = {r0 * ir, r1 * ir, r2 * ir};
                const double w = Q.w * ar;
                const Expo E = expo(r, f);
                cd t1, t2, u1, u12, u3;
                b_coef(E, ir, ir2, f, m, t1, t2, u1, u12, u3);
                const double rn = h[0] * n[0] + h[1] * n[1] + h[2] * n[2];
                t1 = t1 * w;
                u1 = u1 * w;
                for (int p = 0; p < 3; p++) fma_cr(mt[p], t1, h[p]);
                fma_cr(m2, t2, w * rn);
                for (int p = 0; p < 3; p++)
                    for (int b = p; b < 3; b++) fma_cr(M[sidx(p, b)], u1, h[p] * h[b]);
                fma_cr(S, u12, w);
                fma_cr(S3, u3, w);
            }
            for (int p = 0; p < 3; p++)
                for (int b = p; b < 3; b++) {
                    cd v = {0, 0};
                    fma_cr(v, mt[p], n[b]);
                    fma_cr(v, mt[b], n[p]);
                    if (p == b) v += m2;
                    bt[sidx(p, b)] += v;
                    for (int k = 0; k < 3; k++) {
                        cd u = {0, 0};
                        fma_cr(u, M[sidx(p, k)], n[b]);
                        fma_cr(u, M[sidx(b, k)], n[p]);
                        fma_cr(u, S, (b == k ? n[p] : 0.0) + (p == k ? n[b] : 0.0));
                        if (p == b) fma_cr(u, S3, n[k]);
                        ba[sidx(p, b) * 3 + k] += u;
                    }
                }
        }
        const double wa = Qa.w * tarea;
        const double wk[3] = {wa * Qa.x, wa * Qa.y, wa * Qa.z};
#pragma unroll
        for (int e = 0; e < 24; e++) {
            const cd v = e < 6 ? bt[e] : ba[e - 6];
            const double sx = block_sum256(v.x, red), sy = block_sum256(v.y, red);
            if (threadIdx.x == 0)
                for (int k = 0; k < 3; k++) corner[k][e][0] += wk[k] * sx, corner[k][e][1] += wk[k] * sy;
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const int k = threadIdx.x;
        cd *bt_out = Bt + (long long)l * nv3 * 3 + (long long)(3 * tv[k]) * 3;
        cd *ba_out = Ba + (long long)l * nv3 * 9 + (long long)(3 * tv[k]) * 9;
        for (int p = 0; p < 3; p++)
            for (int b = 0; b < 3; b++) {
                const int e = sidx(p, b);
                bt_out[p * 3 + b] += cd{corner[k][e][0], corner[k][e][1]};
                for (int q = 0; q < 3; q++) ba_out[p * 9 + b * 3 + q] += cd{corner[k][6 + e * 3 + q][0], corner[k][6 + e * 3 + q][1]};
            }
    }
}

// ---------------------------------------------------------------------------
// Touching pairs, Sauter-Schwab.  Pair record: kind (1 coincident, 2 edge, 3 vertex),
// f2 (source normal), j1[3], j2[3] (re-ordered corner vertices, integrator_galerkin.hpp:262-334).
// ---------------------------------------------------------------------------
struct Pair {
    int kind, f2;
    int j1[3], j2[3];
    int f1;
};

// Output per pair and frequency (complex): G 81 (row 3i+p, col 3j+q), H 81, Bt 27 (row 3i+p, col q), Ba 81 (row 3i+p, col q*3+k)
constexpr int kPairG = 0, kPairH = 81, kPairBt = 162, kPairBa = 189, kPairStride = 270;

// Point-pair kernel accumulation for MODE 0 (G), 1 (H), 2 (B).
template <int MODE> struct SingAcc {
    cd v[MODE == 0 ? 63 : (MODE == 1 ? 81 : 36)];
};

template <int MODE>
__device__ __forceinline__ void sing_eval(const double x[3], const double y[3], const double Lx[3], const double Ly[3], double wt,
                                 const double n[3], const Freq &f, const Mat &m, const MathTables *M, cd *acc) {
    const double r0 = y[0] - x[0], r1 = y[1] - x[1], r2 = y[2] - x[2];
    const double d2 = r0 * r0 + r1 * r1 + r2 * r2;
    const double ir = rsqrt_nr(d2), r = d2 * ir, ir2 = ir * ir;
    const double h[3] = {r0 * ir, r1 * ir, r2 * ir};
    const Expo E = expo(r, f, M);
    if (MODE == 0) {
        cd al, be;
        g_coef(E, ir, ir2, m, al, be);
        al = al * ir;
        be = be * ir;
        const double hh[6] = {h[0] * h[0], h[1] * h[1], h[2] * h[2], h[0] * h[1], h[0] * h[2], h[1] * h[2]};
        #pragma unroll
        for (int i = 0; i < 3; i++)
            #pragma unroll
            for (int j = 0; j < 3; j++) {
                const double w = wt * Lx[i] * Ly[j];
                const cd aw = al * w;
                cd *a = acc + (i * 3 + j) * 7;
                #pragma unroll
                for (int e = 0; e < 6; e++) fma_cr(a[e], aw, hh[e]);
                fma_cr(a[6], be, w);
            }
    } else if (MODE == 1) {
        cd c1, c2, c4;
        h_coef(E, ir, ir2, f, m, c1, c2, c4);
        const double rn = h[0] * n[0] + h[1] * n[1] + h[2] * n[2];
        cd pv[9];
        #pragma unroll
        for (int p = 0; p < 3; p++)
            #pragma unroll
            for (int b = 0; b < 3; b++) {
                cd v = c1 * (h[p] * n[b]);
                fma_cr(v, c2, n[p] * h[b] + (p == b ? rn : 0.0));
                fma_cr(v, c4, rn * h[p] * h[b]);
                pv[p * 3 + b] = v;
            }
        #pragma unroll
        for (int i = 0; i < 3; i++)
            #pragma unroll
            for (int j = 0; j < 3; j++) {
                const double w = wt * Lx[i] * Ly[j];
                cd *a = acc + (i * 3 + j) * 9;
                #pragma unroll
                for (int e = 0; e < 9; e++) fma_cr(a[e], pv[e], w);
            }
    } else {
        cd t1, t2, u1, u12, u3;
        b_coef(E, ir, ir2, f, m, t1, t2, u1, u12, u3);
        const double rn = h[0] * n[0] + h[1] * n[1] + h[2] * n[2];
        #pragma unroll
        for (int i = 0; i < 3; i++) {
            const double wi = wt * Lx[i];
            cd *a = acc + i * 12;
            const cd tw = t1 * wi, uw = u1 * wi;
            #pragma unroll
            for (int p = 0; p < 3; p++) fma_cr(a[p], tw, h[p]);
            fma_cr(a[3], t2, wi * rn);
            #pragma unroll
            for (int p = 0; p < 3; p++)
                #pragma unroll
                for (int b = p; b < 3; b++) fma_cr(a[4 + sidx(p, b)], uw, h[p] * h[b]);
            fma_cr(a[10], u12, wi);
            fma_cr(a[11], u3, wi);
        }
    }
}

// Point r of the Sauter-Schwab region maps (integrator_galerkin.hpp:42-212) at the 4D rule point
// (e1, e2, e3, xi) with rule weight w: test barycentric coordinates (a0, a1), source (b0, b1), weight wt.
template <int KIND>
__device__ __forceinline__ void region_point(int r, double e1, double e2, double e3, double xi, double w, double &a0,
                                             double &a1, double &b0, double &b1, double &wt) {
    if (KIND == 1) {
        wt = w * xi * xi * xi * e1 * e1 * e2;
        switch (r) {
        case 0: a0 = xi, a1 = xi * (1.0 - e1 + e1 * e2), b0 = xi * (1.0 - e1 * e2 * e3), b1 = xi * (1.0 - e1); break;
        case 1: a0 = xi * (1.0 - e1 * e2 * e3), a1 = xi * (1.0 - e1), b0 = xi, b1 = xi * (1.0 - e1 + e1 * e2); break;
        case 2: a0 = xi, a1 = xi * e1 * (1.0 - e2 + e2 * e3), b0 = xi * (1.0 - e1 * e2), b1 = xi * e1 * (1.0 - e2); break;
        case 3: a0 = xi * (1.0 - e1 * e2), a1 = xi * e1 * (1.0 - e2), b0 = xi, b1 = xi * e1 * (1.0 - e2 + e2 * e3); break;
        case 4: a0 = xi * (1.0 - e1 * e2 * e3), a1 = xi * e1 * (1.0 - e2 * e3), b0 = xi, b1 = xi * e1 * (1.0 - e2); break;
        default: a0 = xi, a1 = xi * e1 * (1.0 - e2), b0 = xi * (1.0 - e1 * e2 * e3), b1 = xi * e1 * (1.0 - e2 * e3); break;
        }
    } else if (KIND == 2) {
        const double W = w * xi * xi * xi * e1 * e1;
        wt = r == 0 ? W : W * e2;
        switch (r) {
        case 0: a0 = xi, a1 = xi * e1 * e3, b0 = xi * (1.0 - e1 * e2), b1 = xi * e1 * (1.0 - e2); break;
        case 1: a0 = xi, a1 = xi * e1, b0 = xi * (1.0 - e1 * e2 * e3), b1 = xi * e1 * e2 * (1.0 - e3); break;
        case 2: a0 = xi * (1.0 - e1 * e2), a1 = xi * e1 * (1.0 - e2), b0 = xi, b1 = xi * e1 * e2 * e3; break;
        case 3: a0 = xi * (1.0 - e1 * e2 * e3), a1 = xi * e1 * e2 * (1.0 - e3), b0 = xi, b1 = xi * e1; break;
        default: a0 = xi * (1.0 - e1 * e2 * e3), a1 = xi * e1 * (1.0 - e2 * e3), b0 = xi, b1 = xi * e1 * e2; break;
        }
    } else {
        wt = w * xi * xi * xi * e2;
        if (r == 0) a0 = xi, a1 = xi * e1, b0 = xi * e2, b1 = xi * e2 * e3;
        else a0 = xi * e2, a1 = xi * e2 * e3, b0 = xi, b1 = xi * e1;
    }
}

// The lane variant (CQBEM_GALERKIN_SINGULAR=lane): every region of every ordered pair, one lane per 4D rule point.
// B (MODE 2) is held to 2 waves per SIMD: its 36 accumulators and working set take 316 registers at 1 wave; at 2 it
// spills 46-59 of them to scratch and still runs 15% faster.  G and H (the lane variant) keep 1 wave.
template <int MODE, int KIND>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(MODE == 2 ? 2 : 1, 2))) k_gal_sing(Geom g, const Pair *__restrict__ pairs, int pair0,
                                                  const double2 *__restrict__ line, int nline,
                                                  const Freq *__restrict__ freqs, Mat m, cd *__restrict__ out) {
    constexpr int NA = MODE == 0 ? 63 : (MODE == 1 ? 81 : 36);
    const int pi = pair0 + blockIdx.x, l = blockIdx.y;
    const Pair P = pairs[pi];
    const Freq f = freqs[l];
    __shared__ MathTables mtab;  // tables of the exponentials
    load_math_tables(&mtab);
    __syncthreads();
    const double n[3] = {g.N[3 * P.f2], g.N[3 * P.f2 + 1], g.N[3 * P.f2 + 2]};
    // x(xh) = px + dx0 xh0 + dx1 xh1 and y likewise; barycentrics (1-h0, h0-h1, h1)
    double px[3], dx0[3], dx1[3], dy0[3], dy1[3], jac;
    {
        const double *A = g.V + 3 * P.j1[0], *B = g.V + 3 * P.j1[1], *Cc = g.V + 3 * P.j1[2];
        #pragma unroll
        for (int k = 0; k < 3; k++) px[k] = A[k];
        if (KIND == 1) {
            #pragma unroll
            for (int k = 0; k < 3; k++) dx0[k] = dy0[k] = B[k] - A[k], dx1[k] = dy1[k] = Cc[k] - B[k];
        } else if (KIND == 2) {
            const double *Y2 = g.V + 3 * P.j2[2];
            #pragma unroll
            for (int k = 0; k < 3; k++) dx0[k] = dy0[k] = B[k] - A[k], dx1[k] = Cc[k] - B[k], dy1[k] = Y2[k] - B[k];
        } else {
            const double *Y1 = g.V + 3 * P.j2[1], *Y2 = g.V + 3 * P.j2[2];
            #pragma unroll
            for (int k = 0; k < 3; k++) dx0[k] = B[k] - A[k], dx1[k] = Cc[k] - B[k], dy0[k] = Y1[k] - A[k], dy1[k] = Y2[k] - Y1[k];
        }
        const double cx[3] = {dx0[1] * dx1[2] - dx0[2] * dx1[1], dx0[2] * dx1[0] - dx0[0] * dx1[2], dx0[0] * dx1[1] - dx0[1] * dx1[0]};
        const double cy[3] = {dy0[1] * dy1[2] - dy0[2] * dy1[1], dy0[2] * dy1[0] - dy0[0] * dy1[2], dy0[0] * dy1[1] - dy0[1] * dy1[0]};
        jac = sqrt(cx[0] * cx[0] + cx[1] * cx[1] + cx[2] * cx[2]) * sqrt(cy[0] * cy[0] + cy[1] * cy[1] + cy[2] * cy[2]);
    }
    cd acc[NA];
    #pragma unroll
    for (int k = 0; k < NA; k++) acc[k] = cd{0, 0};
    const int n4 = nline * nline * nline * nline;
    for (int p = threadIdx.x; p < n4; p += 64) {
        const int ia = p / (nline * nline * nline), ib = (p / (nline * nline)) % nline, ic = (p / nline) % nline, id = p % nline;
        const double e1 = line[ia].x, e2 = line[ib].x, e3 = line[ic].x, xi = line[id].x;
        const double w = line[ia].y * line[ib].y * line[ic].y * line[id].y;
        constexpr int NR = KIND == 1 ? 6 : (KIND == 2 ? 5 : 2);
#pragma unroll 1
        for (int r = 0; r < NR; r++) {
            double a0, a1, b0, b1, wt;
            region_point<KIND>(r, e1, e2, e3, xi, w, a0, a1, b0, b1, wt);
            double x[3], y[3];
            #pragma unroll
            for (int k = 0; k < 3; k++) x[k] = px[k] + dx0[k] * a0 + dx1[k] * a1, y[k] = px[k] + dy0[k] * b0 + dy1[k] * b1;
            const double Lx[3] = {1.0 - a0, a0 - a1, a1}, Ly[3] = {1.0 - b0, b0 - b1, b1};
            sing_eval<MODE>(x, y, Lx, Ly, wt, n, f, m, &mtab, acc);
        }
    }
    // wave reduction; lane 0 expands and writes
    #pragma unroll
    for (int k = 0; k < NA; k++) {
        double vx = acc[k].x, vy = acc[k].y;
        #pragma unroll
        for (int o = 32; o > 0; o >>= 1) vx += __shfl_xor(vx, o, 64), vy += __shfl_xor(vy, o, 64);
        acc[k] = cd{vx * jac, vy * jac};
    }
    if (threadIdx.x != 0) return;
    cd *o = out + ((long long)pi * gridDim.y + l) * kPairStride;
    if (MODE == 0) {
        #pragma unroll
        for (int i = 0; i < 3; i++)
            #pragma unroll
            for (int j = 0; j < 3; j++)
                #pragma unroll
                for (int p = 0; p < 3; p++)
                    #pragma unroll
                    for (int b = 0; b < 3; b++) {
                        cd v = acc[(i * 3 + j) * 7 + sidx(p, b)];
                        if (p == b) v += acc[(i * 3 + j) * 7 + 6];
                        o[kPairG + (3 * i + p) * 9 + 3 * j + b] = v;
                    }
    } else if (MODE == 1) {
        #pragma unroll
        for (int i = 0; i < 3; i++)
            #pragma unroll
            for (int j = 0; j < 3; j++)
                #pragma unroll
                for (int p = 0; p < 3; p++)
                    #pragma unroll
                    for (int b = 0; b < 3; b++) o[kPairH + (3 * i + p) * 9 + 3 * j + b] = acc[(i * 3 + j) * 9 + p * 3 + b] * kInv4Pi;
    } else {
        #pragma unroll
        for (int i = 0; i < 3; i++) {
            const cd *a = acc + i * 12;
            #pragma unroll
            for (int p = 0; p < 3; p++)
                #pragma unroll
                for (int b = 0; b < 3; b++) {
                    cd v = {0, 0};
                    fma_cr(v, a[p], n[b]);
                    fma_cr(v, a[b], n[p]);
                    if (p == b) v += a[3];
                    o[kPairBt + (3 * i + p) * 3 + b] = v;
                    #pragma unroll
                    for (int k = 0; k < 3; k++) {
                        cd u = {0, 0};
                        fma_cr(u, a[4 + sidx(p, k)], n[b]);
                        fma_cr(u, a[4 + sidx(b, k)], n[p]);
                        fma_cr(u, a[10], (b == k ? n[p] : 0.0) + (p == k ? n[b] : 0.0));
                        if (p == b) fma_cr(u, a[11], n[k]);
                        o[kPairBa + (3 * i + p) * 9 + b * 3 + k] = u;
                    }
                }
        }
    }
}

// ---------------------------------------------------------------------------
// Touching pairs, direction form.  Every Sauter-Schwab map scales with its last coordinate xi: both faces' points are
// xi times a point that depends on the other three, so along xi the direction of y - x is constant, r = xi |d|, and
// the basis products Lx_i Ly_j are polynomials of degree 2 in xi.  A lane takes one direction (e1, e2, e3, region),
// sums the functions e^-z1, e^-z2 and s^2 (A1 - A2) times the needed powers of xi over the xi rule (24 or 18 FMAs per
// point), and only then, once per direction, forms the kernel entries and multiplies them by the basis.  With the
// reduced basis {1, Lx1, Lx2} x {1, Ly1, Ly2} (Lx0 = 1 - Lx1 - Lx2 is restored at the end) every product has a single
// power of xi: T_0 for 1, T_1 for the four linear ones, T_2 for the four quadratic ones.  The two sets of four are the
// rows of 4x4x4 FP64 matrix products: lane (j, b, k) = j + 4 b + 16 k holds item j's entry at direction (b, k) as the
// B operand and row j's basis value at that direction as the A operand, which is the same for every item, since the
// basis depends on the rule alone.  An item is a (pair, frequency); a wave works on four items and 16 directions.
// The entries are those of the source face's frame (see FaceFrame).
// Bound by FP64 VALU issue: 117 instructions per point for vertex-adjacent pairs and B, 190 where r is formed from
// coordinates (touch_distance), and 450 to 700 per direction of n points; the per-point kernels took about 430 (G),
// 520 (H) and 280 (B) per point and formed all 9 basis products at each.  Icosphere level 3, L = 32, rule 5 x 2 (n = 10):
// all touching pairs 352 -> 101 ms.
// ---------------------------------------------------------------------------
constexpr int kTouchXi = 8;      // words of the xi table per point: xi, w / xi, w, w xi, .., w xi^4, -
constexpr int kTouchMaxLine = 80;

// The xi table of a composite rule of n points, and after it the sums of w xi and w xi^2.
__global__ void k_gal_xi(const double2 *__restrict__ line, int n, double *__restrict__ tab) {
    const int q = threadIdx.x;
    if (q < n) {
        const double xi = line[q].x, w = line[q].y;
        double *t = tab + kTouchXi * q;
        t[0] = xi, t[1] = w / xi, t[2] = w, t[3] = w * xi, t[4] = w * xi * xi, t[5] = w * xi * xi * xi, t[6] = w * xi * xi * xi * xi;
        t[7] = 0.0;
    }
    if (q == 0) {
        double k0 = 0, k1 = 0;
        for (int k = 0; k < n; k++) k0 += line[k].y * line[k].x, k1 += line[k].y * line[k].x * line[k].x;
        tab[kTouchXi * n] = k0, tab[kTouchXi * n + 1] = k1;
    }
}

// One item's constants, in the LDS: the edges in the source face's frame (y's lie in its plane), the frequency and the
// rotation back.
struct TouchItem {
    double dx0[3], dx1[3], dy0[2], dy1[2];
    cd sc1, sc2, is2, is, s;
    double Q[3][3], jac;
    double px[3], gx0[3], gx1[3], gy0[3], gy1[3];  // the shared vertex and the edges in the global axes
};

// Fills item `it` (clamped to the last) of the pairs from pair0 on; called by one lane per item.
template <int KIND>
__device__ inline void load_item(const Geom &g, const Pair *__restrict__ pairs, const Freq *__restrict__ freqs, long long it,
                                 int pair0, int nl, TouchItem &I) {
    const Pair P = pairs[pair0 + (int)(it / nl)];
    const Freq f = freqs[(int)(it % nl)];
    const double *A = g.V + 3 * P.j1[0], *B = g.V + 3 * P.j1[1], *C = g.V + 3 * P.j1[2];
    const double *Y1 = KIND == 3 ? g.V + 3 * P.j2[1] : B, *Y2 = KIND == 1 ? C : g.V + 3 * P.j2[2];
    double dx0[3], dx1[3], dy0[3], dy1[3];
    for (int k = 0; k < 3; k++) dx0[k] = B[k] - A[k], dx1[k] = C[k] - B[k], dy0[k] = Y1[k] - A[k], dy1[k] = Y2[k] - Y1[k];
    auto area2 = [](const double *u, const double *v) {
        const double c[3] = {u[1] * v[2] - u[2] * v[1], u[2] * v[0] - u[0] * v[2], u[0] * v[1] - u[1] * v[0]};
        return sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
    };
    I.jac = area2(dx0, dx1) * area2(dy0, dy1);
    const double il = 1.0 / sqrt(dy0[0] * dy0[0] + dy0[1] * dy0[1] + dy0[2] * dy0[2]);
    double n[3], t1[3], t2[3];
    for (int k = 0; k < 3; k++) n[k] = g.N[3 * P.f2 + k], t1[k] = dy0[k] * il;
    for (int k = 0; k < 3; k++) t2[k] = n[(k + 1) % 3] * t1[(k + 2) % 3] - n[(k + 2) % 3] * t1[(k + 1) % 3];
    auto dot = [](const double *u, const double *v) { return u[0] * v[0] + u[1] * v[1] + u[2] * v[2]; };
    I.dx0[0] = dot(dx0, t1), I.dx0[1] = dot(dx0, t2), I.dx0[2] = KIND == 3 ? dot(dx0, n) : 0.0;
    I.dx1[0] = dot(dx1, t1), I.dx1[1] = dot(dx1, t2), I.dx1[2] = KIND == 1 ? 0.0 : dot(dx1, n);
    I.dy0[0] = dot(dy0, t1), I.dy0[1] = dot(dy0, t2), I.dy1[0] = dot(dy1, t1), I.dy1[1] = dot(dy1, t2);
    I.sc1 = f.sc1, I.sc2 = f.sc2, I.is2 = f.is2, I.is = f.is, I.s = f.s;
    for (int k = 0; k < 3; k++) I.px[k] = A[k], I.gx0[k] = dx0[k], I.gx1[k] = dx1[k], I.gy0[k] = dy0[k], I.gy1[k] = dy1[k];
    for (int k = 0; k < 3; k++) I.Q[0][k] = t1[k], I.Q[1][k] = t2[k], I.Q[2][k] = n[k];
}

// What the directions of one lane keep in the LDS while the xi rule runs: 1/|d|, the direction (a, b, c), the direction's
// weight, the A operands of the linear and the quadratic basis, |d| and (e1, e2, e3).
struct TouchDir {
    double2 id_a, bc, wA1, A2_len, e12, e3_;
};

// Direction dd (0 .. n^3 - 1) of region r for a lane of item I: z_k at xi = 1, and the rest into D.  A direction past
// the end has weight 0.
template <int KIND>
__device__ __forceinline__ void touch_direction(int r, int dd, int nline, const double2 *line, const TouchItem &I, int row,
                                                cd &zd1, cd &zd2, TouchDir &D) {
    const int n2 = nline * nline, nd = n2 * nline, p = min(dd, nd - 1);
    const int ia = p / n2, ib = (p - ia * n2) / nline, ic = p - ia * n2 - ib * nline;
    const double2 la = line[ia], lb = line[ib], lc = line[ic];
    double a0, a1, b0, b1, wt;
    region_point<KIND>(r, la.x, lb.x, lc.x, 1.0, dd < nd ? la.y * lb.y * lc.y : 0.0, a0, a1, b0, b1, wt);
    double d[3];
#pragma unroll
    for (int k = 0; k < 2; k++) d[k] = fma(I.dy0[k], b0, I.dy1[k] * b1) - fma(I.dx0[k], a0, I.dx1[k] * a1);
    d[2] = -fma(I.dx0[2], a0, I.dx1[2] * a1);
    const double d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
    const double id = rsqrt_nr(d2), len = d2 * id;
    zd1 = I.sc1 * len, zd2 = I.sc2 * len;
    const double x1 = a0 - a1, x2 = a1, y1 = b0 - b1, y2 = b1;
    const double A1 = row < 2 ? (row == 0 ? x1 : x2) : (row == 2 ? y1 : y2);
    const double A2 = (row < 2 ? x1 : x2) * (row & 1 ? y2 : y1);
    D.id_a = make_double2(id, d[0] * id), D.bc = make_double2(d[1] * id, d[2] * id), D.wA1 = make_double2(wt, wt * A1);
    D.A2_len = make_double2(wt * A2, len), D.e12 = make_double2(la.x, lb.x), D.e3_ = make_double2(lc.x, 0.0);
}

// |y - x| at one point of the rule, from the points' coordinates in the global axes.  Coincident and edge-adjacent
// pairs have rule points so close that the rounding of z = s r / c decides, through the exponentials, the last digits
// of what is left of A1 - A2, different at every frequency; the late weights amplify those digits by R^-n.  Their r is
// therefore formed with the roundings of the per-point kernels.
template <int KIND>
__device__ __forceinline__ double touch_distance(int region, const TouchDir &D, double xi, const TouchItem &I) {
    double a0, a1, b0, b1, wt, x[3], y[3];
    region_point<KIND>(region, D.e12.x, D.e12.y, D.e3_.x, xi, 1.0, a0, a1, b0, b1, wt);
#pragma unroll
    for (int k = 0; k < 3; k++)
        x[k] = I.px[k] + I.gx0[k] * a0 + I.gx1[k] * a1, y[k] = I.px[k] + I.gy0[k] * b0 + I.gy1[k] * b1;
    const double r0 = y[0] - x[0], r1 = y[1] - x[1], r2 = y[2] - x[2];
    const double d2 = r0 * r0 + r1 * r1 + r2 * r2;
    return d2 * rsqrt_nr(d2);
}

__device__ inline void mfma_acc(cd &acc, double A, const cd &T) {
    acc.x = __builtin_amdgcn_mfma_f64_4x4x4f64(A, T.x, acc.x, 0, 0, 0);
    acc.y = __builtin_amdgcn_mfma_f64_4x4x4f64(A, T.y, acc.y, 0, 0, 0);
}

// Adds the wave's sums of NC entries into the block's Phi[item][basis product][entry] (wave 0 stores), all over the four
// blocks of their rows: c1 and (QUAD) c2 as rows of basis products, c0 with QUAD as rows of entries (entry 4 g + i in row
// i of c0[g]), without it as one sum per lane.  Basis products: 1, Lx1, Lx2, Ly1, Ly2, then Lx_i Ly_j.
template <int NC, bool QUAD>
__device__ inline void touch_reduce(const cd *c0, const cd *c1, const cd *c2, int wave, int nwaves, cd *Phi) {
    constexpr int NB = QUAD ? 9 : 5;
    const int lane = threadIdx.x & 63, j = lane & 3, row = lane >> 4;
    auto sum = [&](cd v, int last) {
        for (int o = 4; o < last; o <<= 1) v.x += __shfl_xor(v.x, o, 64), v.y += __shfl_xor(v.y, o, 64);
        return v;
    };
    for (int w = 0; w < nwaves; w++) {
        if (w == wave) {
            auto put = [&](int basis, int e, const cd &v) {
                cd *p = Phi + (j * NB + basis) * NC + e;
                *p = w == 0 ? v : cd{p->x + v.x, p->y + v.y};
            };
#pragma unroll
            for (int e = 0; e < NC; e++) {
                const cd s1 = sum(c1[e], 16), s2 = QUAD ? sum(c2[e], 16) : cd{0, 0};
                if ((lane & 12) == 0) {
                    put(1 + row, e, s1);
                    if (QUAD) put(5 + row, e, s2);
                }
                if (!QUAD) {
                    const cd s0 = sum(c0[e], 64);
                    if (lane < 4) put(0, e, s0);
                } else if (e % 4 == 0) {
                    const cd s0 = sum(c0[e / 4], 16);
                    if ((lane & 12) == 0 && e + row < NC) put(0, e + row, s0);
                }
            }
        }
        __syncthreads();
    }
}

// HALF (coincident pairs only): regions 1, 3, 5 of the six, whose exchanged images are the other three; the exchanged
// half is added afterwards by k_gal_coincident_sym.  NW waves share a block's four items, each taking every NW-th group
// of 16 directions.
template <bool DG, bool DH, int KIND, bool HALF, int NW>
__global__ void __launch_bounds__(64 * NW, 2) k_gal_touch(Geom g, const Pair *__restrict__ pairs, int pair0, long long nitems,
                                                          const double2 *__restrict__ line, int nline,
                                                          const double *__restrict__ xtab, const Freq *__restrict__ freqs,
                                                          int nl, Mat m, cd *__restrict__ out) {
    constexpr int NG = DG ? 6 : 0, NC = NG + (DH ? 8 : 0);
    constexpr int NR = KIND == 1 ? (HALF ? 3 : 6) : (KIND == 2 ? 5 : 2);
    __shared__ MathTables mtab;
    __shared__ TouchItem item[4];
    __shared__ double2 lin[kTouchMaxLine];
    __shared__ TouchDir dir[64 * NW];
    __shared__ cd Phi[4 * 9 * NC];
    constexpr bool CLOSE = KIND != 3;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long long it0 = 4LL * blockIdx.x;
    load_math_tables(&mtab);
    for (int k = tid; k < nline; k += 64 * NW) lin[k] = line[k];
    if (tid < 4) load_item<KIND>(g, pairs, freqs, it0 + tid < nitems ? it0 + tid : nitems - 1, pair0, nl, item[tid]);
    __syncthreads();
    const int j = lane & 3, slot = lane >> 2;
    const int nd = nline * nline * nline;
    const const_double *xt = (const const_double *)xtab;
    cd c0[(NC + 3) / 4], c1[NC], c2[NC];
#pragma unroll
    for (int e = 0; e < NC; e++) c0[e / 4] = c1[e] = c2[e] = cd{0, 0};
#pragma unroll 1
    for (int r = 0; r < NR; r++) {
        const int region = HALF ? 2 * r : r;
#pragma unroll 1
        for (int d0 = 16 * wave; d0 < nd; d0 += 16 * NW) {
            cd zd1, zd2;
            touch_direction<KIND>(region, d0 + slot, nline, lin, item[j], j, zd1, zd2, dir[tid]);
            // moments with w xi^3: powers p of xi from kE on for e1, e2 and from -4 on for the others
            constexpr int kE = CLOSE ? -3 : -2, nE = 2 - kE;
            cd e1[nE], e2[nE], ds[4], da[3];
#pragma unroll
            for (int k = 0; k < nE; k++) e1[k] = e2[k] = cd{0, 0};
#pragma unroll
            for (int k = 0; k < 4; k++) ds[k] = cd{0, 0};
#pragma unroll
            for (int k = 0; k < 3; k++) da[k] = cd{0, 0};
#pragma unroll 1
            for (int q = 0; q < nline; q++) {
                const const_double *X = xt + kTouchXi * q;
                cd z1, z2;
                if (CLOSE) {
                    int jj = j;
                    asm volatile("" : "+v"(jj));  // the item stays in the LDS
                    const TouchItem &I = item[jj];
                    const double len = touch_distance<KIND>(region, dir[tid], X[0], I);
                    z1 = I.sc1 * len, z2 = I.sc2 * len;
                } else {
                    z1 = zd1 * X[0], z2 = zd2 * X[0];
                }
                const cd E1 = cexp_neg_tab(z1, &mtab), E2 = cexp_neg_tab(z2, &mtab);
                const cd dS = CLOSE ? E1 - E2 : (z1 * E1 + E1) - (z2 * E2 + E2);
#pragma unroll
                for (int k = 0; k < nE; k++) fma_cr(e1[k], E1, X[5 + kE + k]), fma_cr(e2[k], E2, X[5 + kE + k]);
#pragma unroll
                for (int k = 0; k < 4; k++) fma_cr(ds[k], dS, X[1 + k]);
                if (DG && KIND == 1) {  // A1 - A2
                    const cd is2 = item[j].is2;
                    const cd A1 = (z1 + cd{1.0, 0.0}) * E1 * is2, A2 = (z2 + cd{1.0, 0.0}) * E2 * is2, dA = A1 - A2;
#pragma unroll
                    for (int k = 0; k < 3; k++) fma_cr(da[k], dA, X[2 + k]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            int ln = tid;  // read back, not kept in registers across the rule
            asm volatile("" : "+v"(ln));
            const TouchDir D = dir[ln];
            const double a = D.id_a.y, b = D.bc.x, c = D.bc.y;
            PointExpo<cd> E;
            E.ir = D.id_a.x, E.ir2 = E.ir * E.ir;
            const TouchItem &I = item[j];
            const cd q1 = I.is * E.ir, q2 = CLOSE ? q1 * q1 : I.is2 * E.ir2;
            if (CLOSE) zd1 = I.sc1 * D.A2_len.y, zd2 = I.sc2 * D.A2_len.y;
            // (A1 - A2) / r^2 times xi^p: the moment ds[p + 4] of (z1 + 1) e1 - (z2 + 1) e2 over (s |d|)^2, or, for close
            // pairs, q (e1 / c1 - e2 / c2) + q^2 (e1 - e2) with q = 1 / (s r)
            auto dd = [&](int p) {
                if (!CLOSE) return ds[p + 2] * q2;
                return (e1[p - 1 - kE] * m.ic1 - e2[p - 1 - kE] * m.ic2) * q1 + ds[p + 2] * q2;
            };
            const double row0[4] = {j == 0 ? D.wA1.x : 0.0, j == 1 ? D.wA1.x : 0.0, j == 2 ? D.wA1.x : 0.0, j == 3 ? D.wA1.x : 0.0};
#pragma unroll
            for (int mm = 0; mm < 3; mm++) {
                cd T[NC > 0 ? NC : 1];
                if (DG) {
                    E.e1 = e1[mm - 1 - kE], E.e2 = e2[mm - 1 - kE];
                    E.dd = KIND == 1 ? da[mm] * E.ir2 : dd(mm - 1);
                    point_g(E, a, b, c, m, T);
                }
                if (DH) {
                    E.e1 = e1[mm - 2 - kE], E.e2 = e2[mm - 2 - kE], E.dd = dd(mm - 2);
                    E.w1 = zd1 * e1[mm - 1 - kE], E.w2 = zd2 * e2[mm - 1 - kE];
                    point_h(E, a, b, c, m, T + NG);
                }
#pragma unroll
                for (int e = 0; e < NC; e++) {
                    if (mm == 0) mfma_acc(c0[e / 4], row0[e % 4], T[e]);
                    else if (mm == 1) mfma_acc(c1[e], D.wA1.y, T[e]);
                    else mfma_acc(c2[e], D.A2_len.x, T[e]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    touch_reduce<NC, true>(c0, c1, c2, wave, NW, Phi);
    // one lane per (item, test corner, source corner): the corner basis from the products, then the global axes
    if (tid >= 36 || it0 + tid / 9 >= nitems) return;
    const int jt = tid / 9, ti = (tid % 9) / 3, tj = tid % 3;
    const cd *ph = Phi + jt * 9 * NC;
    const TouchItem &I = item[jt];
    double A[3][3];
    for (int k = 0; k < 3; k++)
        for (int d = 0; d < 3; d++) A[k][d] = I.Q[k][d] * I.jac;
    auto corner = [&](int e) {
        auto p = [&](int k) { return ph[k * NC + e]; };
        if (ti && tj) return p(2 + 2 * ti + tj);
        if (ti) return p(ti) - p(3 + 2 * ti) - p(4 + 2 * ti);
        if (tj) return p(2 + tj) - p(4 + tj) - p(6 + tj);
        return (p(0) - p(1) - p(2)) - (p(3) + p(4)) + ((p(5) + p(6)) + (p(7) + p(8)));
    };
    const long long it = it0 + jt;
    cd *o = out + ((long long)(pair0 + (int)(it / nl)) * nl + (int)(it % nl)) * kPairStride;
    if (DG) {
        double Sx[6], Sy[6], Rx[6], Ry[6];
        for (int e = 0; e < 6; e++) {
            const cd v = corner(e);
            Sx[e] = v.x, Sy[e] = v.y;
        }
        rotate_sym(Sx, I.Q, A, Rx), rotate_sym(Sy, I.Q, A, Ry);
        for (int p = 0; p < 3; p++)
            for (int b = 0; b < 3; b++)
                o[kPairG + (3 * ti + p) * 9 + 3 * tj + b] = cd{Rx[sidx(p, b)], Ry[sidx(p, b)]} * m.g_scale;
    }
    if (DH) {
        double Sx[8], Sy[8], Rx[9], Ry[9];
        for (int e = 0; e < 8; e++) {
            const cd v = corner(NG + e);
            Sx[e] = v.x, Sy[e] = v.y;
        }
        rotate_gen(Sx, I.Q, A, Rx), rotate_gen(Sy, I.Q, A, Ry);
        for (int p = 0; p < 3; p++)
            for (int b = 0; b < 3; b++) o[kPairH + (3 * ti + p) * 9 + 3 * tj + b] = cd{Rx[p * 3 + b], Ry[p * 3 + b]} * kInv4Pi;
    }
}

// The same for B_trans and B_angular, which have the test basis only: T_0 for 1 and T_1 for Lx1, Lx2 (and Ly1, Ly2).
// Entries, in units of 1/(8 pi s^2): the odd ones t1 h (3) and t2 c, the even ones u1 h h + u12 I (6) and u3.  HALF
// (coincident pairs): regions 1, 3, 5, each point standing for its exchanged image too, whose test basis is Ly: the odd
// entries take Lx - Ly and the even ones Lx + Ly.
template <int KIND, bool HALF, int NW>
__global__ void __launch_bounds__(64 * NW, 2) k_gal_touch_b(Geom g, const Pair *__restrict__ pairs, int pair0, long long nitems,
                                                            const double2 *__restrict__ line, int nline,
                                                            const double *__restrict__ xtab, const Freq *__restrict__ freqs,
                                                            int nl, Mat m, cd *__restrict__ out) {
    constexpr int NC = 11, NO = 4;  // entries, of which the first NO are odd in y - x
    constexpr int NR = KIND == 1 ? (HALF ? 3 : 6) : (KIND == 2 ? 5 : 2);
    __shared__ MathTables mtab;
    __shared__ TouchItem item[4];
    __shared__ double2 lin[kTouchMaxLine];
    __shared__ TouchDir dir[64 * NW];
    __shared__ cd Phi[4 * 5 * NC];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long long it0 = 4LL * blockIdx.x;
    load_math_tables(&mtab);
    for (int k = tid; k < nline; k += 64 * NW) lin[k] = line[k];
    if (tid < 4) load_item<KIND>(g, pairs, freqs, it0 + tid < nitems ? it0 + tid : nitems - 1, pair0, nl, item[tid]);
    __syncthreads();
    const int j = lane & 3, slot = lane >> 2;
    const int nd = nline * nline * nline;
    const const_double *xt = (const const_double *)xtab;
    cd c0[NC], c1[NC];
#pragma unroll
    for (int e = 0; e < NC; e++) c0[e] = c1[e] = cd{0, 0};
#pragma unroll 1
    for (int r = 0; r < NR; r++) {
#pragma unroll 1
        for (int d0 = 16 * wave; d0 < nd; d0 += 16 * NW) {
            cd zd1, zd2;
            touch_direction<KIND>(HALF ? 2 * r : r, d0 + slot, nline, lin, item[j], j, zd1, zd2, dir[tid]);
            cd e1[2], e2[4], ds[3];  // xi^0, xi^1; xi^-2 .. xi^1; xi^-2 .. xi^0, with w xi^3
            e1[0] = e1[1] = cd{0, 0};
#pragma unroll
            for (int k = 0; k < 4; k++) e2[k] = cd{0, 0};
#pragma unroll
            for (int k = 0; k < 3; k++) ds[k] = cd{0, 0};
#pragma unroll 1
            for (int q = 0; q < nline; q++) {
                const const_double *X = xt + kTouchXi * q;
                const cd z1 = zd1 * X[0], z2 = zd2 * X[0];
                const cd E1 = cexp_neg_tab(z1, &mtab), E2 = cexp_neg_tab(z2, &mtab);
                const cd dS = (z1 * E1 + E1) - (z2 * E2 + E2);
                fma_cr(e1[0], E1, X[5]), fma_cr(e1[1], E1, X[6]);
#pragma unroll
                for (int k = 0; k < 4; k++) fma_cr(e2[k], E2, X[3 + k]);
#pragma unroll
                for (int k = 0; k < 3; k++) fma_cr(ds[k], dS, X[3 + k]);
            }
            __builtin_amdgcn_sched_barrier(0);
            int ln = tid;
            asm volatile("" : "+v"(ln));
            const TouchDir D = dir[ln];
            const double id = D.id_a.x, id2 = id * id, h[3] = {D.id_a.y, D.bc.x, D.bc.y};
            const cd s = item[j].s;
#pragma unroll
            for (int mm = 0; mm < 2; mm++) {
                cd T[NC];
                const cd t1 = ds[mm] * id2, u1 = ds[mm + 1] * id;
                const cd v = e2[mm + 2] * m.ic2, S = s * (v - e1[mm] * m.ic1);
                cd t2 = zd2 * e2[mm + 1] + e2[mm];
                t2.x -= xt[kTouchXi * nline + mm];
#pragma unroll
                for (int k = 0; k < 3; k++) T[k] = t1 * h[k];
                T[3] = t2 * (2.0 * id2 * h[2]);
                const cd u12 = u1 + S;
#pragma unroll
                for (int p = 0; p < 3; p++)
#pragma unroll
                    for (int q = p; q < 3; q++) {
                        cd w = p == q ? u12 : cd{0, 0};
                        fma_cr(w, u1, h[p] * h[q]);
                        T[NO + sidx(p, q)] = w;
                    }
                T[10] = s * v * 2.0;
#pragma unroll
                for (int e = 0; e < NC; e++) {
                    if (mm == 0) fma_cr(c0[e], T[e], D.wA1.x);
                    else mfma_acc(c1[e], D.wA1.y, T[e]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    touch_reduce<NC, false>(c0, c1, nullptr, wave, NW, Phi);
    // one lane per (item, test corner)
    if (tid >= 12 || it0 + tid / 3 >= nitems) return;
    const int jt = tid / 3, ti = tid % 3;
    const TouchItem &I = item[jt];
    const cd *ph = Phi + jt * 5 * NC;
    cd v[NC];
    for (int e = 0; e < NC; e++) {
        auto p = [&](int k) { return ph[k * NC + e]; };
        const double sg = e < NO ? -1.0 : 1.0;  // weight of the exchanged image's basis
        if (ti) {
            v[e] = p(ti);
            if (HALF) fma_cr(v[e], p(2 + ti), sg);
        } else {
            v[e] = cd{0, 0} - (p(1) + p(2));
            if (HALF) fma_cr(v[e], p(3) + p(4), -sg);
            fma_cr(v[e], p(0), HALF ? 1.0 + sg : 1.0);
        }
        v[e] = v[e] * I.is2 * (I.jac * kInv8Pi);
    }
    cd mt[3], M[6];
    for (int d = 0; d < 3; d++) {
        mt[d] = cd{0, 0};
        for (int k = 0; k < 3; k++) fma_cr(mt[d], v[k], I.Q[k][d]);
    }
    double Sx[6], Sy[6], Rx[6], Ry[6];
    for (int e = 0; e < 6; e++) Sx[e] = v[NO + e].x, Sy[e] = v[NO + e].y;
    rotate_sym(Sx, I.Q, I.Q, Rx), rotate_sym(Sy, I.Q, I.Q, Ry);
    for (int e = 0; e < 6; e++) M[e] = cd{Rx[e], Ry[e]};
    const double *n = I.Q[2];
    const long long it = it0 + jt;
    cd *o = out + ((long long)(pair0 + (int)(it / nl)) * nl + (int)(it % nl)) * kPairStride;
    for (int p = 0; p < 3; p++)
        for (int b = 0; b < 3; b++) {
            cd t = p == b ? v[3] : cd{0, 0};
            fma_cr(t, mt[p], n[b]);
            fma_cr(t, mt[b], n[p]);
            o[kPairBt + (3 * ti + p) * 3 + b] = t;
            for (int k = 0; k < 3; k++) {
                cd u = {0, 0};
                fma_cr(u, M[sidx(p, k)], n[b]);
                fma_cr(u, M[sidx(b, k)], n[p]);
                if (p == b) fma_cr(u, v[10], n[k]);
                o[kPairBa + (3 * ti + p) * 9 + b * 3 + k] = u;
            }
        }
}

// Coincident pairs integrated over regions 1, 3, 5 only (sums S).  Regions 2, 4, 6 are those with x and y
// exchanged (integrator_galerkin.hpp:64-92), which swaps the test and source corners, keeps the G kernel
// (even in y - x) and negates the H kernel (odd in y - x; both points lie on the one face, so n is shared):
//   G(i p, j b) = S(i p, j b) + S(j p, i b),   H(i p, j b) = S(i p, j b) - S(j p, i b).
// One thread per (pair, frequency, matrix, entry pair {(i p, j b), (j p, i b)} with i <= j).
__global__ void k_gal_coincident_sym(int np, int nl, int do_g, int do_h, cd *__restrict__ out) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long long)np * nl * 2 * 54) return;
    const int u = (int)(t % 54);
    const int mat = (int)((t / 54) % 2);
    const long long kl = t / 108;
    if (mat == 0 ? !do_g : !do_h) return;
    // u = 9 c + 3 p + b over the corner pairs c: (0,0) (1,1) (2,2) (0,1) (0,2) (1,2)
    const int c = u / 9, p = (u / 3) % 3, b = u % 3;
    const int ci[6] = {0, 1, 2, 0, 0, 1}, cj[6] = {0, 1, 2, 1, 2, 2};
    const int i = ci[c], j = cj[c];
    cd *o = out + kl * kPairStride + (mat == 0 ? kPairG : kPairH);
    const int ea = (3 * i + p) * 9 + 3 * j + b, eb = (3 * j + p) * 9 + 3 * i + b;
    const cd sa = o[ea], sb = o[eb];
    if (mat == 0) {
        o[ea] = sa + sb;
        if (eb != ea) o[eb] = sb + sa;
    } else {
        o[ea] = sa - sb;
        if (eb != ea) o[eb] = sb - sa;
    }
}

// Gather touching-pair blocks into the spectra.  One lane per (output block, l);
// items[ptr[b]..ptr[b+1]) = pair*9 + i*3 + j in a fixed order.
__global__ void k_gal_gather_gh(const int2 *__restrict__ blocks, const int *__restrict__ ptr, const int *__restrict__ items,
                                int nblocks, int nl, const cd *__restrict__ scratch, cd *__restrict__ UG, cd *__restrict__ UH,
                                long long ld, long long lstride) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long long)nblocks * nl) return;
    const int b = (int)(t / nl), l = (int)(t % nl);
    const int2 uv = blocks[b];
    cd g[9], h[9];
    for (int e = 0; e < 9; e++) g[e] = h[e] = cd{0, 0};
    for (int k = ptr[b]; k < ptr[b + 1]; k++) {
        const int it = items[k];
        const int pi = it / 9, i = (it % 9) / 3, j = it % 3;
        const cd *o = scratch + ((long long)pi * nl + l) * kPairStride;
        for (int p = 0; p < 3; p++)
            for (int q = 0; q < 3; q++) {
                g[p * 3 + q] += o[kPairG + (3 * i + p) * 9 + 3 * j + q];
                h[p * 3 + q] += o[kPairH + (3 * i + p) * 9 + 3 * j + q];
            }
    }
    const long long base = (long long)l * lstride + (long long)(3 * uv.x) * ld + 3LL * uv.y;
    for (int p = 0; p < 3; p++)
        for (int q = 0; q < 3; q++) {
            if (UG) UG[base + p * ld + q] += g[p * 3 + q];
            if (UH) UH[base + p * ld + q] += h[p * 3 + q];
        }
}

// The same for B, one lane per (vertex, frequency, entry): a pair's 36 entries per corner are read by neighbouring lanes
// (icosphere level 2, L = 16: 40 us; one lane per (vertex, frequency) took 1070 us, 2754 lanes of strided 16-byte loads).
__global__ void k_gal_gather_b(const int *__restrict__ vptr, const int *__restrict__ items, int nv, int nl,
                               const cd *__restrict__ scratch, cd *__restrict__ Bt, cd *__restrict__ Ba, long long nv3) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long long)nv * nl * 36) return;
    const int e = (int)(t % 36), l = (int)(t / 36 % nl), u = (int)(t / 36 / nl);
    // entries 0..8 are B_trans's three rows, 9..35 B_angular's
    const int off = e < 9 ? kPairBt + e : kPairBa + e - 9, corner = e < 9 ? 9 : 27;
    cd s = {0, 0};
    for (int k = vptr[u]; k < vptr[u + 1]; k++) {
        const int it = items[k];
        s += scratch[((long long)(it / 3) * nl + l) * kPairStride + off + (it % 3) * corner];
    }
    if (e < 9) Bt[(long long)l * nv3 * 3 + 9LL * u + e] += s;
    else Ba[(long long)l * nv3 * 9 + 27LL * u + e - 9] += s;
}

// Test points of the faces faces[0..nfl) in that order: tpts[fi * npts + a] = (x_a, face) with x_a the a-th rule
// point of the face, and psi[3 (fi * npts + a) + k] = w_a area phi_k(x_a), the weight of x_a for test corner k.
__global__ void k_gal_points(Geom g, const double4 *__restrict__ quad, int npts, const int *__restrict__ faces, int nfl,
                             double4 *__restrict__ tpts, double *__restrict__ psi) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long long)nfl * npts) return;
    const int fi = (int)(t / npts), a = (int)(t % npts);
    const int f1 = faces[fi];
    const double *X0 = g.V + 3 * g.F[3 * f1], *X1 = g.V + 3 * g.F[3 * f1 + 1], *X2 = g.V + 3 * g.F[3 * f1 + 2];
    const double4 Qa = quad[a];
    const double x0 = Qa.x * X0[0] + Qa.y * X1[0] + Qa.z * X2[0];
    const double x1 = Qa.x * X0[1] + Qa.y * X1[1] + Qa.z * X2[1];
    const double x2 = Qa.x * X0[2] + Qa.y * X1[2] + Qa.z * X2[2];
    tpts[t] = make_double4(x0, x1, x2, (double)f1);
    const double wa = Qa.w * g.area[f1];
    psi[3 * t] = wa * Qa.x, psi[3 * t + 1] = wa * Qa.y, psi[3 * t + 2] = wa * Qa.z;
}

// Projection of per-point rows onto the test basis.  src holds, per frequency (stride src_ls), rows 3p..3p+2 of
// ew complex entries for the local test points p = fl * npts + a of the chunk faces faces[0..nfc); the faces of a
// chunk share no vertex, so dst rows 3 F[f][k] + r are owned by one thread each:
//   dst[l][3 F[f][k] + r][c] += sum_a psi[k of point row0 + p] src[l][3 p + r][c].
__global__ void k_gal_project(const cd *__restrict__ src, long long ew, long long src_ls, const double *__restrict__ psi,
                              const int *__restrict__ faces, int nfc, int npts, long long row0, const int *__restrict__ F,
                              cd *__restrict__ dst, long long dst_ls) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long long)nfc * 3 * ew) return;
    const int l = blockIdx.y;
    const int fl = (int)(t / (3 * ew));
    const long long rem = t - (long long)fl * 3 * ew;
    const int r = (int)(rem / ew);
    const long long c = rem - r * ew;
    const cd *s = src + (long long)l * src_ls + (3LL * fl * npts + r) * ew + c;
    const double *w = psi + 3 * (row0 + (long long)fl * npts);
    cd a0 = {0, 0}, a1 = {0, 0}, a2 = {0, 0};
    for (int a = 0; a < npts; a++) {
        const cd v = s[3LL * a * ew];
        fma_cr(a0, v, w[3 * a]);
        fma_cr(a1, v, w[3 * a + 1]);
        fma_cr(a2, v, w[3 * a + 2]);
    }
    const int f = faces[fl];
    cd *d = dst + (long long)l * dst_ls + r * ew + c;
    d[3LL * F[3 * f] * ew] += a0;
    d[3LL * F[3 * f + 1] * ew] += a1;
    d[3LL * F[3 * f + 2] * ew] += a2;
}

__global__ void k_fill_zero(double2 *p, long long n) {
    const long long stride = (long long)gridDim.x * 256;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) p[i] = make_double2(0.0, 0.0);
}

void check(hipError_t e, const char *what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

struct DevVec {
    void *p = nullptr;
    bool pooled = false;
    ~DevVec() { dev_free(p, pooled); }
    void alloc(size_t n, const char *what) { check(dev_alloc(&p, std::max<size_t>(n, 1), &pooled), what); }
    template <class T> T *up(const std::vector<T> &v, hipStream_t st) {
        alloc(v.size() * sizeof(T), "device allocation");
        if (!v.empty()) check(hipMemcpyAsync(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, st), "hipMemcpyAsync");
        return (T *)p;
    }
};

void zero(cd *p, long long n, int num_cus, hipStream_t st) {
    if (!p || n <= 0) return;
    long long blocks = std::min<long long>((n + 255) / 256, (long long)num_cus * 8);
    hipLaunchKernelGGL(k_fill_zero, dim3((unsigned)blocks), dim3(256), 0, st, (double2 *)p, n);
    check(hipGetLastError(), "k_fill_zero");
}

}  // namespace

int galerkin_chunk_faces(int nv, int nf, int npts, int nl, bool G, bool H, bool B, size_t budget) {
    const size_t per_face = (size_t)npts * 3 * nl * ((G ? 3ULL * nv : 0) + (H ? 3ULL * nv : 0) + (B ? 12 : 0)) * sizeof(cd);
    size_t cap = per_face ? budget / per_face : (size_t)nf;
    cap = std::max<size_t>(cap, 1);
    cap = std::min<size_t>(cap, (size_t)(65535 / std::max(npts, 1)));
    return (int)std::min<size_t>(cap, (size_t)std::max(nf, 1));
}

size_t galerkin_scratch_bytes(int nv, int nf, int npts, int nl, bool G, bool H, bool B, size_t budget) {
    const size_t cap = (size_t)galerkin_chunk_faces(nv, nf, npts, nl, G, H, B, budget);
    const size_t rows = 3 * cap * npts;
    return (size_t)nf * npts * (sizeof(double4) + 3 * sizeof(double)) +
           (size_t)nl * rows * ((G ? 3ULL * nv : 0) + (H ? 3ULL * nv : 0) + (B ? 12 : 0)) * sizeof(cd);
}

std::vector<std::vector<int>> touching_candidates(const int *F, int nf, int nv, const int *vmap) {
    // faces around each vertex, or around each original vertex when the mesh is split
    std::vector<std::vector<int>> around(nv);
    auto key = [&](int v) { return vmap ? vmap[v] : v; };
    for (int f = 0; f < nf; f++)
        for (int k = 0; k < 3; k++) around[key(F[3 * f + k])].push_back(f);
    std::vector<std::vector<int>> cand(nf);
    for (int f1 = 0; f1 < nf; f1++) {
        auto &c = cand[f1];
        for (int k = 0; k < 3; k++) {
            const auto &a = around[key(F[3 * f1 + k])];
            c.insert(c.end(), a.begin(), a.end());
        }
        std::sort(c.begin(), c.end());
        c.erase(std::unique(c.begin(), c.end()), c.end());
    }
    return cand;
}

void run_galerkin(const GalerkinJob &job, const int *F, const int *vmap, cd *U, cd *P, cd *Bt, cd *Ba, double *tm,
                  hipStream_t st) {
    const Geom &g = job.g;
    const int nv = g.nv, nf = g.nf, nl = job.nl;
    const long long n3 = 3LL * nv;
    zero(U, U ? (long long)nl * n3 * n3 : 0, job.num_cus, st);
    zero(P, P ? (long long)nl * n3 * n3 : 0, job.num_cus, st);
    zero(Bt, Bt ? (long long)nl * n3 * 3 : 0, job.num_cus, st);
    zero(Ba, Ba ? (long long)nl * n3 * 9 : 0, job.num_cus, st);

    // Greedy colouring of test faces: faces sharing a vertex get different colours.
    std::vector<int> color(nf, -1), vmark;
    std::vector<std::vector<int>> classes;
    {
        std::vector<std::vector<char>> used;  // used[c][v]
        for (int f = 0; f < nf; f++) {
            int c = 0;
            for (;; c++) {
                if (c == (int)used.size()) used.emplace_back(nv, 0), classes.emplace_back();
                if (!used[c][F[3 * f]] && !used[c][F[3 * f + 1]] && !used[c][F[3 * f + 2]]) break;
            }
            color[f] = c;
            for (int k = 0; k < 3; k++) used[c][F[3 * f + k]] = 1;
            classes[c].push_back(f);
        }
    }
    std::vector<int> flat, cls_off{0};
    for (auto &c : classes) flat.insert(flat.end(), c.begin(), c.end()), cls_off.push_back((int)flat.size());
    DevVec dfaces;
    const int *faces = dfaces.up(flat, st);
    // faces sharing an (original) vertex with each face: its touching pairs, which the regular kernels exclude
    const std::vector<std::vector<int>> cands = touching_candidates(F, nf, nv, vmap);

    const char *variant = std::getenv("CQBEM_GALERKIN_KERNEL");
    if ((U || P || Bt || Ba) && !(variant && !std::strcmp(variant, "star"))) {
        // Test-point rows: the collocation kernels evaluate, for every rule point x_a of the test faces of a
        // chunk, the row sum over the source faces not touching x_a's face; k_gal_project then weights the
        // rows by the test basis.  Chunks are runs of one colour class, so their faces share no vertex.
        PhaseTimer t(st, &tm[1]);
        const int npts = job.npts;
        const long long ntp = (long long)nf * npts;
        DevVec dtp, dpsi, dsG, dsH, dsBt, dsBa;
        dtp.alloc((size_t)ntp * sizeof(double4), "device allocation: test points");
        dpsi.alloc((size_t)ntp * 3 * sizeof(double), "device allocation: test weights");
        double4 *tpts = (double4 *)dtp.p;
        double *psi = (double *)dpsi.p;
        hipLaunchKernelGGL(k_gal_points, dim3((unsigned)((ntp + 255) / 256)), dim3(256), 0, st, g, job.quad, npts, faces, nf,
                           tpts, psi);
        check(hipGetLastError(), "k_gal_points");
        const int cap = galerkin_chunk_faces(nv, nf, npts, nl, U != nullptr, P != nullptr, Bt && Ba, job.scratch_bytes);
        const long long cap_rows = 3LL * cap * npts, ls = cap_rows * n3;
        if (U) dsG.alloc((size_t)nl * ls * sizeof(cd), "device allocation: point rows G");
        if (P) dsH.alloc((size_t)nl * ls * sizeof(cd), "device allocation: point rows H");
        if (Bt && Ba) {
            dsBt.alloc((size_t)nl * cap_rows * 3 * sizeof(cd), "device allocation: point rows Bt");
            dsBa.alloc((size_t)nl * cap_rows * 9 * sizeof(cd), "device allocation: point rows Ba");
        }
        cd *sG = (cd *)dsG.p, *sH = (cd *)dsH.p, *sBt = (cd *)dsBt.p, *sBa = (cd *)dsBa.p;
        auto project = [&](const cd *src, long long ew, long long src_ls, const int *cf, int nfc, long long row0, cd *dst,
                           long long dst_ls) {
            const long long n = (long long)nfc * 3 * ew;
            hipLaunchKernelGGL(k_gal_project, dim3((unsigned)((n + 255) / 256), nl), dim3(256), 0, st, src, ew, src_ls, psi, cf,
                               nfc, npts, row0, g.F, dst, dst_ls);
            check(hipGetLastError(), "k_gal_project");
        };
        for (size_t c = 0; c < classes.size(); c++) {
            const int cnt = cls_off[c + 1] - cls_off[c];
            for (int b = 0; b < cnt; b += cap) {
                const int nfc = std::min(cap, cnt - b), fi0 = cls_off[c] + b;
                const int row0 = fi0 * npts, nrows = nfc * npts;
                if (U || P) {
                    {
                        // the patch kernel at the test points: timed on its own, with its launches and its unique
                        // evaluations (test point, regular source face, source point, frequency)
                        PhaseTimer tp(st, &tm[2]);
                        check(launch_colloc_gh_patch(g, job.patch_pts, npts, job.freqs, 0, nl, job.real_ends, job.mat, row0, nrows,
                                                    tpts, job.patch_chunk, job.chunk_info, job.chunk_faces, job.patch_verts,
                                                    job.npatches, sG, sH, n3, ls, st),
                              "k_colloc_gh_patch (test points)");
                    }
                    tm[6] += 1;
                    for (int fi = fi0; fi < fi0 + nfc; fi++)
                        tm[7] += (double)npts * (double)(nf - (int)cands[flat[fi]].size()) * npts * nl;
                    if (U) project(sG, n3, ls, faces + fi0, nfc, row0, U, n3 * n3);
                    if (P) project(sH, n3, ls, faces + fi0, nfc, row0, P, n3 * n3);
                }
                if (Bt && Ba) {
                    if (job.freqs32)
                        check(launch_points_b32(g, job.quad, npts, job.freqs32, 0, nl, job.mat32, tpts, row0, nrows, sBt, sBa,
                                                cap_rows, st),
                              "k_colloc_b32 (test points)");
                    else
                        check(launch_points_b(g, job.quad, npts, job.freqs, 0, nl, job.real_ends, job.mat, tpts, row0, nrows, sBt, sBa,
                                              cap_rows, st),
                              "k_colloc_b (test points)");
                    project(sBt, 3, cap_rows * 3, faces + fi0, nfc, row0, Bt, n3 * 3);
                    project(sBa, 9, cap_rows * 9, faces + fi0, nfc, row0, Ba, n3 * 9);
                }
            }
        }
    } else if (U || P || Bt || Ba) {
        PhaseTimer t(st, &tm[1]);
        for (size_t c = 0; c < classes.size(); c++) {
            const int cnt = cls_off[c + 1] - cls_off[c];
            const int *fc = faces + cls_off[c];
            if (U || P) {
                dim3 grid((nv + 63) / 64, nl, cnt);
                if (U) hipLaunchKernelGGL((k_gal_gh<true, false>), grid, dim3(64), 0, st, g, job.quad, job.npts, job.freqs, job.mat, fc, U, (cd *)nullptr, n3, n3 * n3);
                if (P) hipLaunchKernelGGL((k_gal_gh<false, true>), grid, dim3(64), 0, st, g, job.quad, job.npts, job.freqs, job.mat, fc, (cd *)nullptr, P, n3, n3 * n3);
                check(hipGetLastError(), "k_gal_gh");
            }
            if (Bt && Ba) {
                hipLaunchKernelGGL(k_gal_b, dim3(nl, cnt), dim3(256), 0, st, g, job.quad, job.npts, job.freqs, job.mat, fc, Bt, Ba, n3);
                check(hipGetLastError(), "k_gal_b");
            }
        }
    }

    // Touching pairs, classified exactly as integrate_galerkin_singular (integrator_galerkin.hpp:262-334).
    std::vector<Pair> pairs;
    {
        auto same = [&](int a, int b) { return a == b || (vmap && vmap[a] == vmap[b]); };
        for (int f1 = 0; f1 < nf; f1++) {
            for (int f2 : cands[f1]) {
                Pair p{};
                p.f1 = f1, p.f2 = f2;
                const int *A = F + 3 * f1, *B = F + 3 * f2;
                if (f1 == f2) {
                    p.kind = 1;
                    for (int k = 0; k < 3; k++) p.j1[k] = p.j2[k] = A[k];
                } else {
                    for (int i = 0; i < 3; i++)
                        for (int j = 0; j < 3; j++)
                            if ((A[i] == B[j] && A[(i + 1) % 3] == B[(j + 2) % 3]) ||
                                (vmap && vmap[A[i]] == vmap[B[j]] && vmap[A[(i + 1) % 3]] == vmap[B[(j + 2) % 3]])) {
                                p.kind = 2;
                                p.j1[0] = A[i], p.j1[1] = A[(i + 1) % 3], p.j1[2] = A[(i + 2) % 3];
                                p.j2[0] = B[j], p.j2[1] = B[(j + 2) % 3], p.j2[2] = B[(j + 1) % 3];
                                break;
                            }
                    if (!p.kind)
                        for (int i = 0; i < 3; i++)
                            for (int j = 0; j < 3; j++)
                                if (same(A[i], B[j])) {
                                    p.kind = 3;
                                    p.j1[0] = A[i], p.j1[1] = A[(i + 1) % 3], p.j1[2] = A[(i + 2) % 3];
                                    p.j2[0] = B[j], p.j2[1] = B[(j + 1) % 3], p.j2[2] = B[(j + 2) % 3];
                                    break;
                                }
                }
                if (p.kind) pairs.push_back(p);
            }
        }
    }
    if (pairs.empty()) return;
    std::stable_sort(pairs.begin(), pairs.end(), [](const Pair &a, const Pair &b) { return a.kind < b.kind; });
    int kind_off[4] = {0, 0, 0, 0};
    for (const Pair &p : pairs) kind_off[p.kind]++;
    kind_off[3] += kind_off[2] += kind_off[1];  // exclusive ends per kind: [0,k1) coincident, [k1,k2) edge, [k2,k3) vertex
    const long long npairs = (long long)pairs.size();
    DevVec dpairs, dscratch, dblocks, dptr, ditems, dvptr, dvitems, dxi;
    const Pair *dp = dpairs.up(pairs, st);
    dscratch.alloc((size_t)npairs * nl * kPairStride * sizeof(cd), "device allocation: touching-pair scratch");
    cd *scratch = (cd *)dscratch.p;
    {
        PhaseTimer t(st, &tm[3]);
        const int beg[3] = {0, kind_off[1], kind_off[2]}, end[3] = {kind_off[1], kind_off[2], kind_off[3]};
#define CQBEM_SING(MODE, KIND)                                                                                        \
    if (end[KIND - 1] > beg[KIND - 1])                                                                                \
        hipLaunchKernelGGL((k_gal_sing<MODE, KIND>), dim3((unsigned)(end[KIND - 1] - beg[KIND - 1]), nl), dim3(64), 0, st, g, \
                           dp, beg[KIND - 1], job.line, job.nline, job.freqs, job.mat, scratch);
        const char *sv = std::getenv("CQBEM_GALERKIN_SINGULAR");
        const bool lane = sv && !std::strcmp(sv, "lane");  // every region of every ordered pair integrated
        if (!lane) {
            dxi.alloc(sizeof(double) * (kTouchXi * job.nline + 2), "device allocation: xi table");
            double *xtab = (double *)dxi.p;
            hipLaunchKernelGGL(k_gal_xi, dim3(1), dim3(128), 0, st, job.line, job.nline, xtab);
            // four waves per block while one wave per block would give fewer than 8 waves per SIMD
#define CQBEM_TOUCH(KERNEL, KIND, ...)                                                                                \
    if (end[KIND - 1] > beg[KIND - 1]) {                                                                              \
        const long long items = (long long)(end[KIND - 1] - beg[KIND - 1]) * nl, blocks = (items + 3) / 4;            \
        if (blocks < 8LL * 4 * job.num_cus)                                                                           \
            hipLaunchKernelGGL((KERNEL<__VA_ARGS__, 4>), dim3((unsigned)blocks), dim3(256), 0, st, g, dp, beg[KIND - 1], items, \
                               job.line, job.nline, xtab, job.freqs, nl, job.mat, scratch);                           \
        else                                                                                                          \
            hipLaunchKernelGGL((KERNEL<__VA_ARGS__, 1>), dim3((unsigned)blocks), dim3(64), 0, st, g, dp, beg[KIND - 1], items, \
                               job.line, job.nline, xtab, job.freqs, nl, job.mat, scratch);                           \
    }
#define CQBEM_TOUCH_GH(DG, DH)                                                                                        \
    {                                                                                                                 \
        CQBEM_TOUCH(k_gal_touch, 1, DG, DH, 1, true)                                                                  \
        CQBEM_TOUCH(k_gal_touch, 2, DG, DH, 2, false)                                                                 \
        CQBEM_TOUCH(k_gal_touch, 3, DG, DH, 3, false)                                                                 \
    }
            if (U && P) CQBEM_TOUCH_GH(true, true)
            else if (U) CQBEM_TOUCH_GH(true, false)
            else if (P) CQBEM_TOUCH_GH(false, true)
            if ((U || P) && end[0] > 0) {  // the coincident pairs' exchanged half
                const long long n = (long long)end[0] * nl * 108;
                hipLaunchKernelGGL(k_gal_coincident_sym, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, end[0], nl,
                                   U ? 1 : 0, P ? 1 : 0, scratch);
            }
            if (Bt && Ba) {
                CQBEM_TOUCH(k_gal_touch_b, 1, 1, true)
                CQBEM_TOUCH(k_gal_touch_b, 2, 2, false)
                CQBEM_TOUCH(k_gal_touch_b, 3, 3, false)
            }
#undef CQBEM_TOUCH_GH
#undef CQBEM_TOUCH
        } else {
            if (U) { CQBEM_SING(0, 1) CQBEM_SING(0, 2) CQBEM_SING(0, 3) }
            if (P) { CQBEM_SING(1, 1) CQBEM_SING(1, 2) CQBEM_SING(1, 3) }
            if (Bt && Ba) { CQBEM_SING(2, 1) CQBEM_SING(2, 2) CQBEM_SING(2, 3) }
        }
#undef CQBEM_SING
        check(hipGetLastError(), "k_gal_sing");
    }
    // gather lists: output block (u, v) <- (pair, i, j); vertex u <- (pair, i)
    std::map<std::pair<int, int>, std::vector<int>> bl;
    std::vector<std::vector<int>> vl(nv);
    for (long long k = 0; k < npairs; k++) {
        for (int i = 0; i < 3; i++) {
            vl[pairs[k].j1[i]].push_back((int)(k * 3 + i));
            for (int j = 0; j < 3; j++) bl[{pairs[k].j1[i], pairs[k].j2[j]}].push_back((int)(k * 9 + i * 3 + j));
        }
    }
    std::vector<int2> blocks;
    std::vector<int> ptr{0}, items, vptr{0}, vitems;
    for (auto &kv : bl) {
        blocks.push_back(make_int2(kv.first.first, kv.first.second));
        items.insert(items.end(), kv.second.begin(), kv.second.end());
        ptr.push_back((int)items.size());
    }
    for (int v = 0; v < nv; v++) vitems.insert(vitems.end(), vl[v].begin(), vl[v].end()), vptr.push_back((int)vitems.size());
    const int2 *db = dblocks.up(blocks, st);
    const int *dpt = dptr.up(ptr, st), *dit = ditems.up(items, st), *dvp = dvptr.up(vptr, st), *dvi = dvitems.up(vitems, st);
    {
        PhaseTimer t(st, &tm[3]);
        if (U || P) {
            const long long n = (long long)blocks.size() * nl;
            hipLaunchKernelGGL(k_gal_gather_gh, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, db, dpt, dit, (int)blocks.size(), nl,
                               scratch, U, P, n3, n3 * n3);
            check(hipGetLastError(), "k_gal_gather_gh");
        }
        if (Bt && Ba) {
            const long long n = (long long)nv * nl * 36;
            hipLaunchKernelGGL(k_gal_gather_b, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dvp, dvi, nv, nl, scratch, Bt, Ba, n3);
            check(hipGetLastError(), "k_gal_gather_b");
        }
    }
    check(hipStreamSynchronize(st), "galerkin sync");
}

}  // namespace cqbem
