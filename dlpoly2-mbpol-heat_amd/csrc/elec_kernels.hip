// elec_kernels.hip -- polarizable Ewald electrostatics of MB-pol water on gfx950.
//
// The reference computes, once per force evaluation (forces.f:268-404 with the
// subroutines it calls):  M sites and DMS charges (dlpoly_cmd.f:2041-2057,
// qdetermine.f90), the induced dipoles by SOR over real-space (rfield.f) and
// reciprocal-space (ewald1p.f, iflag = 0) fields (iter.f), then the polarization energy
// (coulomb_polar.f), reciprocal energy / forces / per-atom stress (ewald1p.f, iflag = 1),
// real-space pair terms (ewald2p.f), intramolecular corrections (ewald3p.f) and the
// charge-derivative forces (qdforce.f90).
//
// GPU organisation (one context, one stream, no atomics on floating-point data: every
// per-site sum is owned by one thread or one wavefront and summed in a fixed order):
//   * real space: full neighbour rows per site (both directions of each pair), so that a
//     wavefront owns a site's row; the Thole-damped dipole tensors of the polarizable
//     pairs are kept as two radial factors, built once per evaluation and read by every
//     solver iteration;
//   * reciprocal space: exp(i k.r_j) comes from per-site tables of exp(i l a*.r_j) (a* a
//     reciprocal vector).  The solver's structure factors and fields are FP64 matrix
//     products over groups of 16 (l, m) pairs and tiles of 8 n, split over chunks of sites
//     and groups of pairs (partials summed in a fixed order); the final forces and stresses
//     are site-parallel over runs of consecutive n at fixed (l, m), with a complex
//     recurrence along n and a split over chunks of runs (likewise);
//   * the solver loop runs on the device; a done flag set by the convergence check turns
//     the remaining kernels of a batch of iterations into no-ops.
#include <math.h>

#include <algorithm>

#include "mbgpu_internal.h"
#include "gen/dms_table.inc"

#define R4PIE0 138935.4835            // dl_params.inc
#define SQRPI 1.7724538509055159      // dl_params.inc
#define TWOPI (2.0 * 3.141592653589793)

namespace {

__device__ __forceinline__ double wsum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// fixed-order block reduction of NV values per thread into out[0..NV) (blockDim <= 1024)
template <int NV>
__device__ void block_sum_store(double (&v)[NV], double* out)
{
    __shared__ double red[16][NV];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nwv = (blockDim.x + 63) >> 6;
    for (int q = 0; q < NV; ++q) {
        const double s = wsum(v[q]);
        if (lane == 0) red[wv][q] = s;
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double s = 0.0;
        for (int w = 0; w < nwv; ++w) s += red[w][threadIdx.x];
        out[threadIdx.x] = s;
    }
}

// Sum over chunks of in[c * cs + off] (c = 0..nc-1) for the 64 elements of a 256-thread
// block, one element per lane: wave w adds the chunks [w nc / 4, (w + 1) nc / 4) in order
// (coalesced loads of 64 consecutive elements), and the four wave sums are added in wave
// order.  Every thread of the block must call it; the sum is returned on threads 0..63.
__device__ double chunk_sum64(const double* __restrict__ in, long cs, int nc, long off, bool valid)
{
    __shared__ double part[4][64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int c0 = (nc * wv) / 4, c1 = (nc * (wv + 1)) / 4;
    double sum = 0.0;
    if (valid) {
        const double* p = in + off;
        int c = c0;
        for (; c + 4 <= c1; c += 4) {
            const double u0 = p[c * cs], u1 = p[(c + 1) * cs], u2 = p[(c + 2) * cs], u3 = p[(c + 3) * cs];
            sum += u0;
            sum += u1;
            sum += u2;
            sum += u3;
        }
        for (; c < c1; ++c) sum += p[c * cs];
    }
    part[wv][lane] = sum;
    __syncthreads();
    const double t = wv == 0 ? ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane] : 0.0;
    __syncthreads();
    return t;
}

// Stopping test and scalars of the conjugate-gradient solver at the start of iteration `it`,
// from the block partials of its last vector update: nb blocks of (r.u, w.u,
// |polr2 r / r4pie0|^2, dipole count, max |m_i|).  Every wavefront that calls it sums the partials in
// the same order and takes lane 0's sums, so all of a launch's wavefronts reach the same
// decision without a grid-wide synchronization.  With `record`, lane 0 stores the iteration
// count, the RMS step and then the done flag or the scalars of the update: beta = g / g_prev,
// alpha = g / (d - beta g / alpha_prev) (first iteration: beta = 0, alpha = g / d), with
// g = r.u and d = w.u (the Chronopoulos-Gear recurrence), and a power of two of about
// 1 / max |m_i| for the particle mesh's spreading of m.  state = [iterations, rms step, done, g,
// alpha, beta, -, d, -, m scale].  Returns true when the dipoles have converged.
// In two parts, so that a kernel can issue its other loads between: cg_load starts the loads of the
// first 64 blocks' partials, cg_finish adds the others and decides.
struct CgSums {
    double a, b, c, d, e;
};
__device__ __forceinline__ CgSums cg_load(int nb, const double* __restrict__ blk)
{
    const int lane = threadIdx.x & 63;
    CgSums s = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (lane < nb) s = {blk[5 * lane], blk[5 * lane + 1], blk[5 * lane + 2], blk[5 * lane + 3], blk[5 * lane + 4]};
    return s;
}
__device__ __forceinline__ bool cg_finish(const ElecDev& P, const CgSums& s0, int it, int nb,
                                          const double* __restrict__ blk, double* __restrict__ state, bool record)
{
    const int lane = threadIdx.x & 63;
    double a = s0.a, b = s0.b, c = s0.c, d = s0.d, e = s0.e;
    for (int k = lane + 64; k < nb; k += 64) {
        a += blk[5 * k];
        b += blk[5 * k + 1];
        c += blk[5 * k + 2];
        d += blk[5 * k + 3];
        e = fmax(e, blk[5 * k + 4]);
    }
    a = __shfl(wsum(a), 0, 64);
    b = __shfl(wsum(b), 0, 64);
    c = __shfl(wsum(c), 0, 64);
    d = __shfl(wsum(d), 0, 64);
    for (int o = 32; o > 0; o >>= 1) e = fmax(e, __shfl_xor(e, o, 64));
    const double rms = (1.0 - P.omega) * sqrt(c / (d == 0.0 ? 1.0 : d));
    const bool done = rms <= P.toler;
    if (record && lane == 0) {
        state[0] = it;
        state[1] = rms;
        state[9] = (e > 0.0 && isfinite(e)) ? ldexp(1.0, -(ilogb(e) + 1)) : 1.0;
        if (done) {
            state[2] = 1.0;
        } else {
            const double beta = it ? a / state[3] : 0.0;
            state[4] = it ? a / (b - beta * a / state[4]) : a / b;
            state[5] = beta;
            state[3] = a;
            state[7] = b;
        }
    }
    return done;
}

__device__ __forceinline__ bool cg_step(const ElecDev& P, int it, int nb, const double* __restrict__ blk,
                                        double* __restrict__ state, bool record)
{
    return cg_finish(P, cg_load(nb, blk), it, nb, blk, state, record);
}

__device__ __forceinline__ int water_of(const ElecDev& P, int i) { return i < P.nreal ? i / 3 : i - P.nreal; }

__device__ __forceinline__ double site_polr2(const ElecDev& P, int i)
{
    return i >= P.nreal ? P.polr2[2] : ((i % 3) == 0 ? P.polr2[0] : P.polr2[1]);
}

// 0 O, 1 H, 2 M
__device__ __forceinline__ int site_type(const ElecDev& P, int i)
{
    return i >= P.nreal ? 2 : ((i % 3) == 0 ? 0 : 1);
}

// erfcc.f: Numerical Recipes erfc with single-precision literals promoted to double.
__device__ double erfcc_nr(double x)
{
    const double z = fabs(x);
    const double t = 1.0 / (1.0 + 0.5 * z);
    double r = t * exp(-z * z - (double)1.26551223f +
                       t * ((double)1.00002368f +
                            t * ((double).37409196f +
                                 t * ((double).09678418f +
                                      t * ((double)-.18628806f +
                                           t * ((double).27886807f +
                                                t * ((double)-1.13520398f +
                                                     t * ((double)1.48851587f +
                                                          t * ((double)-0.82215223f + t * (double).17087277f)))))))));
    return x < 0.0 ? 2.0 - r : r;
}

// gammq.f: gammln, gser, gcf, gammq (EPS, FPMIN single-precision values)
__device__ double gammln_nr(double xx)
{
    const double cof[6] = {76.18009172947146, -86.50532032941677, 24.01409824083091,
                           -1.231739572450155, .1208650973866179e-2, -.5395239384953e-5};
    double x = xx, y = x;
    double tmp = x + 5.5;
    tmp = (x + 0.5) * log(tmp) - tmp;
    double ser = 1.000000000190015;
    for (int j = 0; j < 6; ++j) {
        y = y + 1.0;
        ser = ser + cof[j] / y;
    }
    return tmp + log(2.5066282746310005 * ser / x);
}

__device__ double gammq_nr(double a, double x, double gln)
{
    const double EPS = (double)3.e-7f, FPMIN = (double)1.e-30f;
    if (x < a + 1.0) {
        if (x <= 0.0) return 1.0;
        double ap = a, sum = 1.0 / a, del = sum;
        for (int n = 1; n <= 800; ++n) {
            ap = ap + 1.0;
            del = del * x / ap;
            sum = sum + del;
            if (fabs(del) < fabs(sum) * EPS) break;
        }
        return 1.0 - sum * exp(-x + a * log(x) - gln);
    }
    double b = x + 1.0 - a, c = 1.0 / FPMIN, d = 1.0 / b, h = d;
    for (int i = 1; i <= 100; ++i) {
        const double an = -i * (i - a);
        b = b + 2.0;
        d = an * d + b;
        if (fabs(d) < FPMIN) d = FPMIN;
        c = b + an / c;
        if (fabs(c) < FPMIN) c = FPMIN;
        d = 1.0 / d;
        const double del = d * c;
        h = h * del;
        if (fabs(del - 1.0) < EPS) break;
    }
    return exp(-x + a * log(x) - gln) * h;
}

// 3-point interpolation of the B-function table (rfield.f:102-120, ewald2p.f:160-178); without
// an Ewald split the functions vanish (an isolated cluster)
__device__ __forceinline__ void table_interp(const ElecDev& P, const double* __restrict__ t, double rr, double* bbb)
{
    if (P.alpha < 1.0e-6) {
        bbb[0] = bbb[1] = bbb[2] = bbb[3] = 0.0;
        return;
    }
    const double q = rr / P.drewd;
    const int ll = (int)q;
    const double ppp = q - (double)ll;
    const double* r0 = t + 4 * ll;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const double vk = r0[n], vk1 = r0[4 + n], vk2 = r0[8 + n];
        const double t1 = vk + (vk1 - vk) * ppp;
        const double t2 = vk1 + (vk2 - vk1) * (ppp - 1.0);
        bbb[n] = t1 + (t2 - t1) * ppp * 0.5;
    }
}

// B functions computed directly (excluded pairs, rfield.f:365-374, ewald3p.f:100-110)
__device__ __forceinline__ void bfun_direct(double alpha, double rr, double rsqi, double* bbb)
{
    if (alpha < 1.0e-6) {   // ewald3p.f: "if ewald parameter is too small then turn it off"
        bbb[0] = bbb[1] = bbb[2] = bbb[3] = 0.0;
        return;
    }
    const double a = alpha * rr;
    bbb[0] = (erfcc_nr(a) - 1.0) / rr;
    const double exp2a = exp(-a * a);
    const double c = 2.0 * alpha * alpha;
    double cm = 1.0;
#pragma unroll
    for (int m = 1; m <= 3; ++m) {
        cm *= c;
        bbb[m] = rsqi * ((2.0 * m - 1.0) * bbb[m - 1] + cm * exp2a / alpha / SQRPI);
    }
}

// imaged separation of sites i, j in the reference's arithmetic
__device__ __forceinline__ double sep(const ElecDev& P, const double* __restrict__ x, const double* __restrict__ y,
                                      const double* __restrict__ z, int i, int j, double* d)
{
#pragma clang fp contract(off)
    double dx = x[i] - x[j], dy = y[i] - y[j], dz = z[i] - z[j];
    image_vec(P.g, dx, dy, dz);
    d[0] = dx;
    d[1] = dy;
    d[2] = dz;
    return norm2_nc(dx, dy, dz);
}

}  // namespace

// ====================================================================== set-up ======

// M sites (dlpoly_cmd.f:2041-2057) and DMS charges with their derivatives
// (qdetermine.f90:118-259; new charge assignment).  One thread per water.
__device__ __forceinline__ void water_sites(const ElecDev& P, int w, double* __restrict__ x, double* __restrict__ y,
                                            double* __restrict__ z, double* __restrict__ chge, double* __restrict__ dg,
                                            double* __restrict__ dip)
{
    // an M site carries no induced dipole (polr2 = 0): any start value cleared
    for (int q = 0; q < 3; ++q) dip[3 * (P.nreal + w) + q] = 0.0;
    const int io = 3 * w, m = P.nreal + w;
    double r1v[3], r2v[3];
    {
#pragma clang fp contract(off)
        double d1x = x[io + 1] - x[io], d1y = y[io + 1] - y[io], d1z = z[io + 1] - z[io];
        double d2x = x[io + 2] - x[io], d2y = y[io + 2] - y[io], d2z = z[io + 2] - z[io];
        image_vec(P.g, d1x, d1y, d1z);
        image_vec(P.g, d2x, d2y, d2z);
        x[m] = x[io] + (d1x + d2x) * P.gamma / 2.0;
        y[m] = y[io] + (d1y + d2y) * P.gamma / 2.0;
        z[m] = z[io] + (d1z + d2z) * P.gamma / 2.0;
        r1v[0] = d1x;
        r1v[1] = d1y;
        r1v[2] = d1z;
        r2v[0] = d2x;
        r2v[1] = d2y;
        r2v[2] = d2z;
    }
    const double r1 = sqrt(r1v[0] * r1v[0] + r1v[1] * r1v[1] + r1v[2] * r1v[2]);
    const double r2 = sqrt(r2v[0] * r2v[0] + r2v[1] * r2v[1] + r2v[2] * r2v[2]);
    const double cost = (r1v[0] * r2v[0] + r1v[1] * r2v[1] + r1v[2] * r2v[2]) / (r1 * r2);
    // reference geometry of the expansion: ps_type_pes reoh, thetae (module.f90:480-481)
    const double reoh = 0.958649, cose = cos(104.3475 * 3.141592653589793 / 180.0);
    const double x1 = (r1 - reoh) / reoh, x2 = (r2 - reoh) / reoh, x3 = cost - cose;
    double f1[8], f2[8], f3[8];
    f1[0] = f2[0] = f3[0] = 0.0;
    f1[1] = f2[1] = f3[1] = 1.0;
#pragma unroll
    for (int j = 2; j < 8; ++j) {
        f1[j] = f1[j - 1] * x1;
        f2[j] = f2[j - 1] * x2;
        f3[j] = f3[j - 1] * x3;
    }
    double p1 = 0.0, p2 = 0.0, g11 = 0.0, g12 = 0.0, g21 = 0.0, g22 = 0.0, g1c = 0.0, g2c = 0.0;
    // (the derivatives' common 1 / reoh once per sum: a division in each of the 84 terms' four
    // made this 17 us of one thread's latency, with the preconditioner's 15 after it: now 8.4 for both)
#pragma unroll
    for (int j = 1; j < DMS_NTERMS; ++j) {
        const int a = dms_idx[j][0], b = dms_idx[j][1], c = dms_idx[j][2];
        const double cf3 = dms_coef[j] * f3[c];
        const double ab = f1[a] * f2[b], ba = f1[b] * f2[a];
        p1 += cf3 * ab;
        p2 += cf3 * ba;
        if (a > 1) {
            g11 += ((a - 1) * cf3) * (f1[a - 1] * f2[b]);
            g22 += ((a - 1) * cf3) * (f1[b] * f2[a - 1]);
        }
        if (b > 1) {
            g12 += ((b - 1) * cf3) * (f1[a] * f2[b - 1]);
            g21 += ((b - 1) * cf3) * (f1[b - 1] * f2[a]);
        }
        if (c > 1) {
            const double d3 = (c - 1) * dms_coef[j] * f3[c - 1];
            g1c += d3 * ab;
            g2c += d3 * ba;
        }
    }
    g11 /= reoh;
    g12 /= reoh;
    g21 /= reoh;
    g22 /= reoh;
    // DMS parameters (module.f90:818-826)
    const double b1dms = 1.0, adms = 0.2999 * 0.529177249, bdms = -0.6932;
    const double c0 = 1.0099, c1 = -0.1801, c2 = 0.0892;
    const double pl1 = cost, pl2 = 0.5 * (3.0 * pl1 * pl1 - 1.0);
    const double damp = exp(-b1dms * ((r1 - reoh) * (r1 - reoh) + (r2 - reoh) * (r2 - reoh)));
    const double ddampdr1 = -2.0 * b1dms * (r1 - reoh) * damp;
    const double ddampdr2 = -2.0 * b1dms * (r2 - reoh) * damp;
    const double leg = c0 + pl1 * c1 + pl2 * c2;
    const double pr1 = pow(r1, bdms), pr2 = pow(r2, bdms);
    const double pc0 = adms * (pr1 + pr2) * leg;
    const double dpc0dr1 = adms * (bdms * (pr1 / r1)) * leg;
    const double dpc0dr2 = adms * (bdms * (pr2 / r2)) * leg;
    const double dpc0dcos = adms * (pr1 + pr2) * (c1 + 3.0 * c2 * pl1);
    double* G = dg + 6 * w;
    G[0] = g11 * damp + p1 * ddampdr1 + dpc0dr1;
    G[1] = g12 * damp + p1 * ddampdr2 + dpc0dr2;
    G[2] = g21 * damp + p2 * ddampdr1 + dpc0dr1;
    G[3] = g22 * damp + p2 * ddampdr2 + dpc0dr2;
    G[4] = g1c * damp + dpc0dcos;
    G[5] = g2c * damp + dpc0dcos;
    p1 = dms_coef[0] + p1 * damp + pc0;
    p2 = dms_coef[0] + p2 * damp + pc0;
    const double factor = P.gamma / 2.0 / (1.0 - P.gamma);
    const double q1 = p1 + factor * (p1 + p2), q2 = p2 + factor * (p1 + p2);
    chge[io] = P.q_o;
    chge[io + 1] = q1;
    chge[io + 2] = q2;
    chge[m] = -(q1 + q2);
}

// packed index of (i, j) in a symmetric 9 x 9 matrix stored as its lower triangle
__device__ __forceinline__ constexpr int tri9(int i, int j) { return i >= j ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i; }

// Per water: the preconditioner block M = diag(r4pie0 / polr2) - r4pie0 T_damped over the
// intramolecular pairs (the Thole-damped dipole tensor of rfield.f:419-520 without its Ewald
// split: M only has to be close to A's block, it does not move the fixed point), inverted
// by Cholesky and stored packed (45 values per water).  Rows of sites without a dipole are
// decoupled unit rows.  A block that is not positive definite falls back to the diagonal.
__device__ __forceinline__ void water_block(const ElecDev& P, int w, const double* __restrict__ x,
                                            const double* __restrict__ y, const double* __restrict__ z,
                                            double* __restrict__ minv)
{
    double a[45];
    bool on[3];
#pragma unroll
    for (int q = 0; q < 45; ++q) a[q] = 0.0;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        const double p2 = site_polr2(P, 3 * w + s);
        on[s] = p2 > P.toler;
#pragma unroll
        for (int c = 0; c < 3; ++c) a[tri9(3 * s + c, 3 * s + c)] = on[s] ? R4PIE0 / p2 : 1.0;
    }
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int t = s + 1; t < 3; ++t) {
            const int i = 3 * w + s, j = 3 * w + t;
            if (!(on[s] && on[t] && site_polr2(P, i) > 1.e-6 && site_polr2(P, j) > 1.e-6)) continue;
            double d[3];
            const double r2 = sep(P, x, y, z, i, j, d);
            const double rr = sqrt(r2);
            const double r3i = 1.0 / (rr * r2), r5i = r3i / r2;
            const double u = rr * P.bbi[site_type(P, i)][site_type(P, j)];
            const double arob4 = (s == 0 ? P.athole12 : P.athole13) * (u * u) * (u * u);
            const double dum1 = exp(-arob4);
            const double dum2 = (1.0 + (4.0 / 3.0) * arob4) * dum1;
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    a[tri9(3 * t + e, 3 * s + c)] =
                        -R4PIE0 * (3.0 * d[c] * d[e] * r5i * (1.0 - dum2) - (c == e ? r3i * (1.0 - dum1) : 0.0));
        }
    // Cholesky M = L L^T in place; the diagonal of L is kept as its inverse
    bool ok = true;
#pragma unroll
    for (int i = 0; i < 9; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j) {
            double v = a[tri9(i, j)];
#pragma unroll
            for (int k = 0; k < j; ++k) v -= a[tri9(i, k)] * a[tri9(j, k)];
            if (i == j) {
                ok = ok && v > 0.0;
                a[tri9(i, i)] = 1.0 / sqrt(fmax(v, 1.e-300));
            } else {
                a[tri9(i, j)] = v * a[tri9(j, j)];
            }
        }
    // X = L^-1 (lower), then M^-1 = X^T X
    double X[45];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        X[tri9(i, i)] = a[tri9(i, i)];
#pragma unroll
        for (int j = 0; j < i; ++j) {
            double v = 0.0;
#pragma unroll
            for (int k = j; k < i; ++k) v += a[tri9(i, k)] * X[tri9(k, j)];
            X[tri9(i, j)] = -v * a[tri9(i, i)];
        }
    }
    double* m = minv + 45L * w;
#pragma unroll
    for (int i = 0; i < 9; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j) {
            double v = 0.0;
#pragma unroll
            for (int k = i; k < 9; ++k) v += X[tri9(k, i)] * X[tri9(k, j)];
            ok = ok && isfinite(v);
            a[tri9(i, j)] = v;
        }
#pragma unroll
    for (int i = 0; i < 9; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j) {
            const int s = i / 3;
            const double jac = (i == j && on[s]) ? site_polr2(P, 3 * w + s) / R4PIE0 : 0.0;
            m[tri9(i, j)] = ok ? a[tri9(i, j)] : jac;
        }
}

// Blocks [0, nb): the M sites and charges; blocks [nb, 2 nb) (conjugate gradients): the
// preconditioner's inverse blocks, which need the real atoms alone.  One thread per water, both
// a chain of one thread's latency, side by side.
__global__ __launch_bounds__(64) void k_el_waters(ElecDev P, int nb, double* __restrict__ x, double* __restrict__ y,
                                                  double* __restrict__ z, double* __restrict__ chge,
                                                  double* __restrict__ dg, double* __restrict__ dip,
                                                  double* __restrict__ minv)
{
    const bool second = (int)blockIdx.x >= nb;
    const int w = (blockIdx.x - (second ? nb : 0)) * 64 + threadIdx.x;
    if (w >= P.nw) return;
    if (second) water_block(P, w, x, y, z, minv);
    else water_sites(P, w, x, y, z, chge, dg, dip);
}

// Reciprocal-space phase tables of each site: cos / sin (l * 2 pi * s_a), s = rcell . r,
// l = 0..kmax_a, by the reference's recurrence (ewald1p.f:196-241, 262-282), layout
// phc/phs [a][l][n] (for the final site pass) and pht[n][rs.kt] (for the matrix passes).
__device__ __forceinline__ void site_phases(const ElecDev& P, int j, const double* __restrict__ x,
                                            const double* __restrict__ y, const double* __restrict__ z,
                                            double* __restrict__ phc, double* __restrict__ phs,
                                            double2* __restrict__ pht)
{
    const double* rcell = P.rs.rc;
    if (j >= P.n) {
        // (the structure-factor pass reads up to RS_PAD sites past the last with weight 0)
        if (j < P.n + RS_PAD)
            for (int l = 0; l < P.rs.kt; ++l) pht[(long)j * P.rs.kt + l] = make_double2(0.0, 0.0);
        return;
    }
    const int ks = P.kstride;
    for (int a = 0; a < 3; ++a) {
        double2* row = pht + (long)j * P.rs.kt + (a == 0 ? 0 : a == 1 ? P.rs.ky : P.rs.kz);
        const double ss = rcell[a] * x[j] + rcell[3 + a] * y[j] + rcell[6 + a] * z[j];
        const double c1 = cos(TWOPI * ss), s1 = sin(TWOPI * ss);
        double c = 1.0, s = 0.0;
        for (int l = 0; l <= P.km[a]; ++l) {
            if (l == 1) {
                c = c1;
                s = s1;
            } else if (l > 1) {
                const double cs = c;
                c = cs * c1 - s * s1;
                s = s * c1 + cs * s1;
            }
            phc[((long)a * ks + l) * P.n + j] = c;
            phs[((long)a * ks + l) * P.n + j] = s;
            row[l] = make_double2(c, s);
            if (a == 1 && l > 0) row[-l] = make_double2(c, -s);
        }
    }
}

// Neighbour rows: every site of another water within rcut (superset by a relative 1e-9 of
// rcut^2; each kernel applies the reference's own test), found in the 27 link cells around
// the site when the box holds three cells per axis (the Verlet list over link cells of
// parlink.f), else by a scan of every site; either way in an order fixed by the positions.
// Row P holds the partners of a polarizable site that are polarizable.  One wavefront per
// site.  The first nph blocks (k-sum) form the phase tables instead, 64 sites each: both parts
// need the sites alone.
__global__ __launch_bounds__(64) void k_el_nbr(ElecDev P, int nph, const double* __restrict__ x,
                                               const double* __restrict__ y, const double* __restrict__ z,
                                               int* __restrict__ nbrA, int* __restrict__ cntA,
                                               int* __restrict__ nbrP, int* __restrict__ cntP, int* __restrict__ err,
                                               double* __restrict__ phc, double* __restrict__ phs,
                                               double2* __restrict__ pht)
{
    const int i = (int)blockIdx.x - nph;
    const int lane = threadIdx.x;
    if (i < 0) {
        site_phases(P, blockIdx.x * 64 + lane, x, y, z, phc, phs, pht);
        return;
    }
    if (i >= P.n) return;
    const int wi = water_of(P, i);
    const bool poli = site_polr2(P, i) > 1.e-6;
    const double rl2 = P.rcut * P.rcut * (1.0 + 1e-9);
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int nA = 0, nP = 0;
    // candidates j (or -1) one per lane, kept in lane order
    auto take = [&](int j) {
        bool inA = false, inP = false;
        if (j >= 0 && water_of(P, j) != wi) {
            double d[3];
            const double r2 = sep(P, x, y, z, i, j, d);
            inA = r2 < rl2;
            inP = inA && poli && site_polr2(P, j) > 1.e-6;
        }
        const unsigned long long bA = __ballot(inA), bP = __ballot(inP);
        if (inA) {
            const int p = nA + __popcll(bA & below);
            if (p < P.capA) nbrA[(long)i * P.capA + p] = j;
        }
        if (inP) {
            const int p = nP + __popcll(bP & below);
            if (p < P.capP) nbrP[(long)i * P.capP + p] = j;
        }
        nA += __popcll(bA);
        nP += __popcll(bP);
    };
    if (P.cells.on) {
        // the 27 link cells around site i: cell order fixed, ascending index within a cell
        for_neighbour_cells(P.cells, i, [&](int c0, int c1) {
            for (int base = c0; base < c1; base += 64) take(base + lane < c1 ? P.cells.idx[base + lane] : -1);
        });
    } else {
        for (int base = 0; base < P.n; base += 64) take(base + lane < P.n ? base + lane : -1);
    }
    if (lane == 0) {
        cntA[i] = min(nA, P.capA);
        cntP[i] = min(nP, P.capP);
        if (nA > P.capA || nP > P.capP) atomicOr(err, 1);
    }
}

// Per-row set-up of the real-space fields (rfield.f:62-323): the charge field of the row's
// partners (iloop = 1 part, with the lads smearing) and the Thole-damped dipole tensors of
// its polarizable partners, T = t2 d d^T - t1 1 with d the imaged separation, stored as their
// radial factors (t1, t2) [n][capP]: the solver reads them every iteration, and 16 bytes and a
// separation formed again cost less there than the six components did (emu_row).  One
// wavefront per site, one pass over its partners: row P holds the polarizable ones in row A's
// order, so a partner's place in it is the count of those before.
// Lanes 0..2 add the excluded (intramolecular) pairs of the site (rfield.f:327-525): the charge
// field with the -erf kernel, and from the lower site of each real pair the dipole tensor (Ewald +
// Applequist - Thole with athole12/athole13), stored tin[nw][pair][6] for pairs (O,H1) (O,H2)
// (O,M) (H1,H2) (H1,M) (H2,M); those of the M site, which carries no dipole, are not used.
__global__ __launch_bounds__(64) void k_el_prep(ElecDev P, const double* __restrict__ x,
                                                const double* __restrict__ y, const double* __restrict__ z,
                                                const double* __restrict__ chge, const double* __restrict__ tab,
                                                const int* __restrict__ nbrA, const int* __restrict__ cntA,
                                                double2* __restrict__ tens, double* __restrict__ tin,
                                                double* __restrict__ efk)
{
    const int i = blockIdx.x;
    const int lane = threadIdx.x;
    if (i >= P.n) return;
    const bool poli = site_polr2(P, i) > 1.e-6;
    const int ti = site_type(P, i);
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    double e[3] = {0.0, 0.0, 0.0};
    if (lane < 3) {
        const int w = water_of(P, i), a = i < P.nreal ? i - 3 * w : 3, b = lane < a ? lane : lane + 1;
        const int j = b < 3 ? 3 * w + b : P.nreal + w;
        double d[3];
        const double r2 = sep(P, x, y, z, i, j, d);
        const double rr = sqrt(r2);
        const double rri = 1.0 / rr, rsqi = rri * rri;
        const double r3i = rri * rsqi;
        double bbb[4];
        bfun_direct(P.alpha, rr, rsqi, bbb);
        const double ek = R4PIE0 * chge[j] * bbb[1];
        e[0] = ek * d[0];
        e[1] = ek * d[1];
        e[2] = ek * d[2];
        if (a < b && b < 3) {
            double t1 = 0.0, t2 = 0.0;
            if (poli && site_polr2(P, j) > 1.e-6) {
                const double u = rr * P.bbi[ti][site_type(P, j)];
                const double arob4 = (a == 0 ? P.athole12 : P.athole13) * (u * u) * (u * u);
                const double dum1 = exp(-arob4);
                const double dum2 = (1.0 + (4.0 / 3.0) * arob4) * dum1;
                t1 = bbb[1] + r3i * (1.0 - dum1);
                t2 = bbb[2] + 3.0 * r3i * rsqi * (1.0 - dum2);
            }
            double* o = tin + 36 * w + 6 * (a == 0 ? b - 1 : 3);
            o[0] = t2 * d[0] * d[0] - t1;
            o[1] = t2 * d[0] * d[1];
            o[2] = t2 * d[0] * d[2];
            o[3] = t2 * d[1] * d[1] - t1;
            o[4] = t2 * d[1] * d[2];
            o[5] = t2 * d[2] * d[2] - t1;
        }
    }
    const int na = cntA[i];
    int np = 0;
    for (int base = 0; base < na; base += 64) {
        const int s = base + lane;
        const bool in = s < na;
        const int j = in ? nbrA[(long)i * P.capA + s] : i;
        const bool inP = in && poli && site_polr2(P, j) > 1.e-6;
        const unsigned long long bP = __ballot(inP);
        const int sp = np + __popcll(bP & below);
        np += __popcll(bP);
        if (!in) continue;
        double d[3];
        const double r2 = sep(P, x, y, z, i, j, d);
        const double rr = sqrt(r2);
        double t1 = 0.0, t2 = 0.0;
        if (P.rcut > rr) {
            double bbb[4];
            table_interp(P, tab, rr, bbb);
            const double rri = 1.0 / rr, rsqi = rri * rri;
            const double r3i = rri * rsqi;
            const double u = rr * P.bbi[ti][site_type(P, j)];
            const double u4 = (u * u) * (u * u);
            const double dumq = exp(-P.ascd * u4);
            const double eki = R4PIE0 * chge[j] * (bbb[1] + r3i * (1.0 - dumq));
            e[0] += eki * d[0];
            e[1] += eki * d[1];
            e[2] += eki * d[2];
            if (inP) {
                const double arob4 = P.athole * u4;
                const double dum1 = exp(-arob4);
                const double dum2 = (1.0 + (4.0 / 3.0) * arob4) * dum1;
                t1 = R4PIE0 * (bbb[1] + r3i * (1.0 - dum1));
                t2 = R4PIE0 * (bbb[2] + 3.0 * r3i * rsqi * (1.0 - dum2));
            }
        }
        // (a partner of the row's margin past rcut has no tensor)
        if (inP && sp < P.capP) tens[(long)i * P.capP + sp] = make_double2(t1, t2);
    }
    for (int q = 0; q < 3; ++q) e[q] = wsum(e[q]);
    if (lane == 0)
        for (int q = 0; q < 3; ++q) efk[3 * i + q] = e[q];
}

// ======================================================= reciprocal-space passes ======

namespace {

// exp(i k.r_j) at the first k of a run (l, m, n0), with the reference's sign rules
// (ewald1p.f:290-306 for m, 346-352 / 392-398 for n).
__device__ __forceinline__ void run_phase(double el_c, double el_s, double em_c, double em_s, double en_c, double en_s,
                                          int m, int n0, double& ckr, double& skr)
{
    // negative m or n use the conjugate table entry; the selects keep the wavefront
    // convergent and give the same products as the reference's branches
    const double sm = m >= 0 ? em_s : -em_s;
    const double sn = n0 >= 0 ? en_s : -en_s;
    const double clm = el_c * em_c - el_s * sm;
    const double slm = el_s * em_c + sm * el_c;
    ckr = clm * en_c - slm * sn;
    skr = slm * en_c + clm * sn;
}

}  // namespace

// Real-space dipole field of one row (rfield.f:201-317 list pairs; 419-520 excluded
// pairs): emu_i = sum_j T_ij mu_j with T_ij = t2 d d^T - t1 1, by one wavefront, or by the WPR
// of a block of 64 WPR threads (which all call it).  Bound by the factors' bytes (88 MB a pass
// for a 701-water cluster, 230 MB when the six tensor components were stored: 38.5 -> 28.7 us) and,
// with one wavefront to a long row, by the chain of its gathers.
template <int WPR>
__device__ void emu_row(const ElecDev& P, int i, int t, const double* __restrict__ x, const double* __restrict__ y,
                        const double* __restrict__ z, const int* __restrict__ nbrP, const int* __restrict__ cntP,
                        const double2* __restrict__ tens, const double* __restrict__ tin,
                        const double* __restrict__ dip, double* __restrict__ emu)
{
    if (i >= P.nrow) return;
    double e[3] = {0, 0, 0};
    const int np = cntP[i];
#pragma unroll 2
    for (int s = t; s < np; s += 64 * WPR) {
        const long o = (long)i * P.capP + s;
        const int j = nbrP[o];
        const double2 tt = tens[o];
        const double mx = dip[3 * j], my = dip[3 * j + 1], mz = dip[3 * j + 2];
        double d[3];
        (void)sep(P, x, y, z, i, j, d);
        const double f = tt.y * (d[0] * mx + d[1] * my + d[2] * mz);
        e[0] += f * d[0] - tt.x * mx;
        e[1] += f * d[1] - tt.x * my;
        e[2] += f * d[2] - tt.x * mz;
    }
    // excluded partners of the same water on lanes 0 and 1: the other two real sites (the M
    // site carries no induced dipole and its entries are not part of the solve); pair order
    // of tin: (O,H1) (O,H2) (O,M) (H1,H2) (H1,M) (H2,M)
    if (t < 2) {
        const int w = i / 3, si = i - 3 * w;
        const int pt = t < si ? t : t + 1;
        const int a = min(si, pt), b = max(si, pt);
        const int pr = a == 0 ? b - 1 : 3;
        const int j = 3 * w + pt;
        if (site_polr2(P, j) > 1.e-6) {
            const double* dt = tin + 36 * w + 6 * pr;
            const double mx = dip[3 * j] * R4PIE0, my = dip[3 * j + 1] * R4PIE0, mz = dip[3 * j + 2] * R4PIE0;
            e[0] += dt[0] * mx + dt[1] * my + dt[2] * mz;
            e[1] += dt[1] * mx + dt[3] * my + dt[4] * mz;
            e[2] += dt[2] * mx + dt[4] * my + dt[5] * mz;
        }
    }
    if constexpr (WPR == 1) {
        for (int q = 0; q < 3; ++q) e[q] = wsum(e[q]);
        if (t == 0)
            for (int q = 0; q < 3; ++q) emu[3 * i + q] = e[q];
    } else {
        block_sum_store(e, emu + 3 * i);
    }
}

// ------------------------------------------- Ewald sums as FP64 matrix products ------
// S(k) = sum_j w_j(k) e^{i k.r_j} and the fields of a set of amplitudes U(k) at the sites,
// over the k list of ewald1p.f:254-345 (k = (l, m, n)).  The list is taken by its (l, m) pairs,
// 16 to a group.  With phi = l x + m y, C = cos phi, S = sin phi per (pair, site) and the
// tables (cos n z, sin n z) per (n > 0, site),
//   S(l, m, +-n) = sum_j w (C cz -+ S sz) + i sum_j w (S cz +- C sz):
// the four sums of the two k are entries of the products [w C; w S] x [cz | sz] over the
// sites, which the matrix cores form in 16 x 16 tiles (pairs x 8 n, cos and sin) four sites at
// a time.  For dipoles w = k.mu = (l alpha + m beta) +- n gamma with alpha = 2 pi a*.mu, ...:
// (l alpha + m beta) goes with the phases, n gamma with the table, in products of their own:
// 8 FLOP per (k, site) where vector sums of the three components with a phase recurrence
// took 20.  The field is the transposed product: with W = akk U the rows
//   H_C = sum_n cz (W+c + W-c) + sz (W+s - W-s),  H_S = sum_n cz (W+s + W-s) + sz (W-c - W+c)
// per (pair, site), and the same with n W for the c* component, are contracted over the pairs
// with C, S, l and m on the spot.
// FP64 matrix and vector instructions share the same units at the same peak here (a loop of
// independent 16x16x4 products reaches 68-71 TFLOP/s, of vector multiply-adds 52), so what the
// matrix form saves is instructions, phase recurrences and the idle time of few wavefronts:
// one wavefront per SIMD already runs them at rate.
// Measured against the vector form with phase recurrences (launches back to back, 2.4 us of each
// the launch itself; structure factors with their chunk sum and the real-space field, then the
// fields): 19.2 + 8.9 and 16.5 -> 10.3 and 11.6 us at 512 waters (9 966 k, 1 536 sites), 162 + 22
// and 137 -> 62 and 58 us at 2 048 waters (33 530 k, 6 144 sites).  At 512 waters what is left is
// latency (the products alone take 2.3 us a pass at rate), at 2 048 the matrix units are busy
// half the time; the rest is phases and operand set-up on the same units.
typedef double v4d __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4d mfma_f64(double a, double b, v4d c)
{
    // a: row lane % 16, column lane / 16; b: row lane / 16, column lane % 16;
    // c[v]: row lane / 16 + 4 v, column lane % 16
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// One set of weights of a structure-factor launch: dipoles mu[3 j] (dip) or scalars v[j stride],
// over the first ns sites; with pol of the polarizable sites alone (ewald1p.f takes no other
// site's dipole, and a caller's start dipoles may hold any value there).
struct RsSrc {
    const double* v;
    int stride, dip, ns, pol;
};
struct RsSrcs {
    RsSrc s[4];
};

#define RS_NT 4                       // tiles of 8 n per block
#define RS_WAVES 8                    // wavefronts per block

// (cos phi, sin phi) of a pair from the table entries of l and m
__device__ __forceinline__ void rs_phase(const double2 X, const double2 Y, double& c, double& s)
{
    c = X.x * Y.x - X.y * Y.y;
    s = X.y * Y.x + X.x * Y.y;
}

// the value of the lane 8 further on within each row of 16 lanes
__device__ __forceinline__ double row_ror8(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x128, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x128, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// A block's sums for one group of pairs, tiles [t0, t0 + NT) of n and one chunk of sites.  The
// chunk's weights are staged in LDS (2 pi a*.mu, 2 pi b*.mu, 2 pi c*.mu and the scalar weight;
// zero past the last site); wavefront w takes the steps of four sites w, w + 8, ..., with the
// next step's table entries loaded while the current one is multiplied, and the eight
// wavefronts' sums are added in order through LDS.
// `go` (the solver's stopping test) is called by every thread once the first loads are under way;
// nothing is written if it returns false.
template <int NT, class Go>
__device__ __forceinline__ void rs_sfac_block(const ElecDev& P, const RsSrc src, int spc, int g, int t0, int chunk,
                                              const double2* __restrict__ pht, double* __restrict__ out, double* lds,
                                              Go&& go)
{
    const RsPlan& R = P.rs;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int j0 = chunk * spc, nj = min(spc, src.ns - j0), nstep = (nj + 3) / 4;
    // (a chunk has at most two sites per thread)
    static_assert(RS_MAX_SPC <= 2 * 64 * RS_WAVES, "");
    double mv[2][3];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int i = tid + 64 * RS_WAVES * h;
        const double* v = src.v + (long)(j0 + i) * src.stride;
        mv[h][0] = mv[h][1] = mv[h][2] = 0.0;
        if (i < nj && (!src.pol || site_polr2(P, j0 + i) > 1.e-6)) {
            mv[h][0] = v[0];
            if (src.dip) {
                mv[h][1] = v[1];
                mv[h][2] = v[2];
            }
        }
    }
    const int4 pr = R.pair[16 * g + (lane & 15)];
    const int nt = max(0, min(NT, __builtin_amdgcn_readfirstlane(pr.w) - t0));
    const int sl = lane >> 4;
    const double dl = pr.x, dm = pr.y;
    // byte offsets from the chunk's first site (a chunk is at most RS_MAX_SPC sites)
    const char* base = reinterpret_cast<const char*>(pht + (long)j0 * R.kt);
    const unsigned step = 64u * R.kt;                     // four sites
    unsigned at = (4u * wv + sl) * 16u * R.kt;
    const unsigned ox = 16u * pr.x, oy = 16u * (R.ky + pr.y);
    unsigned oz[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        // past the largest n of the list any entry of the table will do: no k takes the sum
        const int n = 8 * (t0 + t) + 1 + (lane & 7);
        oz[t] = 16u * (R.kz + min(n, P.km[2])) + (lane & 8);
    }
    v4d ac[NT], as[NT], gc[NT], gs[NT];      // sums with l alpha + m beta (or the scalar), with gamma
#pragma unroll
    for (int t = 0; t < NT; ++t) ac[t] = as[t] = gc[t] = gs[t] = (v4d){0.0, 0.0, 0.0, 0.0};
    double c0 = 0.0, s0 = 0.0;
    double2 X, Y;
    double z[NT];
    auto load = [&](unsigned o) {
        X = *reinterpret_cast<const double2*>(base + (o + ox));
        Y = *reinterpret_cast<const double2*>(base + (o + oy));
#pragma unroll
        for (int t = 0; t < NT; ++t) z[t] = *reinterpret_cast<const double*>(base + (o + oz[t]));
    };
    if (wv < nstep) load(at);
    if (!go()) return;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int i = tid + 64 * RS_WAVES * h;
        if (i < 4 * nstep) {
            double4 w = make_double4(0.0, 0.0, 0.0, mv[h][0]);
            if (src.dip) {
                const double mx = TWOPI * mv[h][0], my = TWOPI * mv[h][1], mz = TWOPI * mv[h][2];
                w.x = R.rc[0] * mx + R.rc[3] * my + R.rc[6] * mz;
                w.y = R.rc[1] * mx + R.rc[4] * my + R.rc[7] * mz;
                w.z = R.rc[2] * mx + R.rc[5] * my + R.rc[8] * mz;
                w.w = 0.0;
            }
            reinterpret_cast<double4*>(lds)[i] = w;
        }
    }
    __syncthreads();
    for (int st = wv; st < nstep; st += RS_WAVES) {
        const double4 w = reinterpret_cast<const double4*>(lds)[4 * st + sl];
        double c, s, zc[NT];
        rs_phase(X, Y, c, s);
#pragma unroll
        for (int t = 0; t < NT; ++t) zc[t] = z[t];
        at += RS_WAVES * step;
        if (st + RS_WAVES < nstep) load(at);
        const double wp = w.w + dl * w.x + dm * w.y;
        const double wc = wp * c, ws = wp * s;
        c0 += wc;
        s0 += ws;
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (t < nt) {
                ac[t] = mfma_f64(wc, zc[t], ac[t]);
                as[t] = mfma_f64(ws, zc[t], as[t]);
                if (src.dip) {
                    const double zg = w.z * zc[t];
                    gc[t] = mfma_f64(c, zg, gc[t]);
                    gs[t] = mfma_f64(s, zg, gs[t]);
                }
            }
    }
    // S(+n), S(-n) of each wavefront (lanes of cos columns: real parts, of sin columns: imaginary
    // parts), then the wavefronts' sums in order; every thread reaches every barrier
    const bool sinc = lane & 8;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        if (t >= nt) break;
        const double n = 8 * (t0 + t) + 1 + (lane & 7);
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double g0 = n * gc[t][v], g1 = n * gs[t][v];
            const double a0 = ac[t][v] + g0, b0 = ac[t][v] - g0;
            const double a1 = row_ror8(as[t][v] + g1), b1 = row_ror8(as[t][v] - g1);
            lds[512 * wv + 64 * v + lane] = sinc ? a0 + a1 : a0 - a1;
            lds[512 * wv + 256 + 64 * v + lane] = sinc ? b1 - b0 : b0 + b1;
        }
        __syncthreads();
        double r = 0.0;
#pragma unroll
        for (int q = 0; q < RS_WAVES; ++q) r += lds[512 * q + tid];
        out[512 * (t0 + t) + tid] = r;
    }
    if (t0 == 0) {
        c0 += __shfl_xor(c0, 16, 64);
        s0 += __shfl_xor(s0, 16, 64);
        c0 += __shfl_xor(c0, 32, 64);
        s0 += __shfl_xor(s0, 32, 64);
        __syncthreads();
        if (lane < 16) {
            lds[32 * wv + lane] = c0;
            lds[32 * wv + 16 + lane] = s0;
        }
        __syncthreads();
        if (tid < 32) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < RS_WAVES; ++q) s += lds[32 * q + tid];
            out[512L * R.ntiles + tid] = s;
        }
    }
}

// Blocks [0, nsb) form the structure factors: block = (set, group of pairs, tile group, chunk),
// chunks fastest, into Spart[set][chunk][group][slot].  The others form the real-space field emu
// of the first set's dipoles, a row per wavefront (both parts need the dipoles alone, so one
// launch holds the two).  With cgblk (the conjugate-gradient solver's partials, cgnb blocks) the
// pass first takes the solver's stopping test for iteration `it` (cg_step; block 0 records the
// scalars) and does nothing once the dipoles have converged.
template <int NT>
__global__ __launch_bounds__(64 * RS_WAVES) void k_rs_sfac(ElecDev P, RsSrcs src, int nsb, int nch, int spc,
                                                           const double2* __restrict__ pht,
                                                           double* __restrict__ Spart, const double* __restrict__ x,
                                                           const double* __restrict__ y, const double* __restrict__ z,
                                                           const int* __restrict__ nbrP, const int* __restrict__ cntP,
                                                           const double2* __restrict__ tens,
                                                           const double* __restrict__ tin, double* __restrict__ emu,
                                                           double* __restrict__ state,
                                                           const double* __restrict__ cgblk, int cgnb, int it)
{
    extern __shared__ double lds[];
    const RsPlan& R = P.rs;
    const double done = state[2];
    CgSums cg = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (cgblk) cg = cg_load(cgnb, cgblk);
    auto go = [&]() {
        if (done != 0.0) return false;
        return !(cgblk && cg_finish(P, cg, it, cgnb, cgblk, state, blockIdx.x == 0 && threadIdx.x < 64));
    };
    int b = blockIdx.x;
    if (b >= nsb) {
        if (!go()) return;
        emu_row<1>(P, (b - nsb) * RS_WAVES + (threadIdx.x >> 6), threadIdx.x & 63, x, y, z, nbrP, cntP, tens, tin,
                   src.s[0].v, emu);
        return;
    }
    // chunks fastest: with 8 chunks (one per XCD, see build_rs) the blocks of an XCD read the
    // same sites, and the groups with the most n, which take longest, start first
    const int ntg = (R.ntiles + NT - 1) / NT;
    const int chunk = b % nch;
    b /= nch;
    const int tg = b % ntg;
    b /= ntg;
    const int g = b % R.ng, set = b / R.ng;
    const long slot = RS_SLOT(R.ntiles);
    rs_sfac_block<NT>(P, src.s[set], spc, g, NT * tg, chunk, pht,
                      Spart + (((long)set * nch + chunk) * R.ng + g) * slot, lds, go);
}

// S(l, m, +n) = v[0] + i v[1] and S(l, m, -n) = v[2] + i v[3] of pair p of a group, n > 0, added
// over the chunks in order: base = the slot of chunk 0, cs = stride from chunk to chunk.
__device__ __forceinline__ void rs_sums(const double* __restrict__ base, long cs, int nch, int p, int n, double (&v)[4])
{
    const double* s = base + 512 * ((n - 1) >> 3) + 64 * (p >> 2) + 16 * (p & 3) + ((n - 1) & 7);
    v[0] = v[1] = v[2] = v[3] = 0.0;
#pragma unroll 4
    for (int ch = 0; ch < nch; ++ch, s += cs) {
        v[0] += s[0];
        v[1] += s[8];
        v[2] += s[256];
        v[3] += s[264];
    }
}

// Reciprocal fields (ewald1p.f:749-769, without the prefactor): a block takes one group of pairs
// and 16 RS_WAVES tpw sites (wavefront w the 16-site tiles w, w + 8, ...).  It first adds the
// group's structure factors over the chunks and lays the weighted amplitudes out in LDS as the
// matrix operands (W of the comment above: H_C, H_S, and both with n W), then each wavefront
// multiplies them with its sites' tables, 4 n at a time, and contracts the 16 pairs' rows.  Set 0
// gives the dipole field, -sum_k k akk (cos Uc + sin Us) with U = S of the dipoles, into
// components 0..2 of Fpart[group][6][n]; set 1 the charge field, U = (Qs, -Qc), into components
// 3..5.  MORE: lists with more than RS_NT tiles of n, whose amplitudes take LDS in turns.
template <bool MORE>
__global__ __launch_bounds__(64 * RS_WAVES, 4) void k_rs_field(ElecDev P, int nch, int tpw, int nsb,
                                                               const double2* __restrict__ pht,
                                                               const double* __restrict__ Spart,
                                                               double* __restrict__ Fpart,
                                                               const double* __restrict__ state)
{
    const double done = state[2];
    __shared__ double W[4][2][8 * RS_NT][16];          // [H_C, H_S, n H_C, n H_S][cos, sin][n][pair]
    __shared__ double W0[2][16];                       // n = 0: [C, S]
    const RsPlan& R = P.rs;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    // site blocks fastest: see k_rs_sfac
    const int sb = blockIdx.x % nsb, g = (blockIdx.x / nsb) % R.ng, set = blockIdx.x / (nsb * R.ng);
    const int row = lane & 15, quad = lane >> 4;
    const int nt = __builtin_amdgcn_readfirstlane(R.pair[16 * g].w);
    const int nn = 8 * R.ntiles + 1;
    const long slot = RS_SLOT(R.ntiles), cs = slot * R.ng;
    const double* base = Spart + ((long)set * nch * R.ng + g) * slot;
    // the amplitudes of tiles [t0, t0 + ntt); every thread of the block takes part (ntt <= RS_NT: one
    // (pair, n) each)
    static_assert(128 * RS_NT <= 64 * RS_WAVES, "");
    // consecutive threads: n of the tile, then pairs, as the sums lie
    const int ap = ((tid >> 3) & 3) + 4 * ((tid >> 5) & 3), an = 8 * (tid >> 7) + (tid & 7);
    double v[4];
    double2 ak;
    auto sums = [&](int t0, int ntt) {
        if (tid < 128 * ntt) {
            rs_sums(base, cs, nch, ap, 8 * t0 + an + 1, v);
            ak = R.ak[(long)(16 * g + ap) * nn + 8 * t0 + an + 1];
        }
    };
    auto amplitudes = [&](int t0, int ntt) {
        if (tid < 128 * ntt) {
            double uc = v[0], us = v[1], dc = v[2], ds = v[3];
            if (set) {
                uc = v[1];
                us = -v[0];
                dc = v[3];
                ds = -v[2];
            }
            uc *= ak.x;
            us *= ak.x;
            dc *= ak.y;
            ds *= ak.y;
            const double fn = 8 * t0 + an + 1;
            W[0][0][an][ap] = uc + dc;
            W[0][1][an][ap] = us - ds;
            W[1][0][an][ap] = us + ds;
            W[1][1][an][ap] = dc - uc;
            W[2][0][an][ap] = fn * (uc - dc);
            W[2][1][an][ap] = fn * (us + ds);
            W[3][0][an][ap] = fn * (us - ds);
            W[3][1][an][ap] = -fn * (uc + dc);
        }
    };
    if (!MORE) sums(0, nt);
    if (wv == RS_WAVES - 1 && lane < 16) {
        double c = 0.0, s = 0.0;
        const double* q = base + 512L * R.ntiles + lane;
        for (int ch = 0; ch < nch; ++ch, q += cs) {
            c += q[0];
            s += q[16];
        }
        const double a = R.ak[(long)(16 * g + lane) * nn].x;
        W0[0][lane] = a * (set ? s : c);
        W0[1][lane] = a * (set ? -c : s);
    }
    double dl[4], dm[4];
    int ox[4], oy[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int4 pr = R.pair[16 * g + quad + 4 * q];
        dl[q] = pr.x;
        dm[q] = pr.y;
        ox[q] = pr.x;
        oy[q] = R.ky + pr.y;
    }
    if (done != 0.0) return;
    if (!MORE) amplitudes(0, nt);
    __syncthreads();
    for (int tl = 0; tl < tpw; ++tl) {
        const int jr = 16 * ((sb * tpw + tl) * RS_WAVES + wv) + row;
        if (!MORE && jr - row >= P.nrow) break;        // (a wavefront's tile is all past the end)
        const bool ok = jr < P.nrow;
        const int j = ok ? jr : P.nrow - 1;
        const double2* p = pht + (long)j * R.kt;
        v4d hc, hs, gc, gs;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            hc[v] = W0[0][quad + 4 * v];
            hs[v] = W0[1][quad + 4 * v];
            gc[v] = gs[v] = 0.0;
        }
        double2 X[4], Y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            X[v] = p[ox[v]];
            Y[v] = p[oy[v]];
        }
        for (int t0 = 0; t0 < nt; t0 += RS_NT) {
            const int ntt = min(RS_NT, nt - t0);
            if (MORE) {
                sums(t0, ntt);
                __syncthreads();
                amplitudes(t0, ntt);
                __syncthreads();
            }
#pragma unroll 2
            for (int q = 0; q < 2 * ntt; ++q) {
                const int nl = 4 * q + quad, n = min(8 * t0 + nl + 1, P.km[2]);
                const double2 z = p[R.kz + n];
                hc = mfma_f64(W[0][0][nl][row], z.x, hc);
                hs = mfma_f64(W[1][0][nl][row], z.x, hs);
                gc = mfma_f64(W[2][0][nl][row], z.x, gc);
                gs = mfma_f64(W[3][0][nl][row], z.x, gs);
                hc = mfma_f64(W[0][1][nl][row], z.y, hc);
                hs = mfma_f64(W[1][1][nl][row], z.y, hs);
                gc = mfma_f64(W[2][1][nl][row], z.y, gc);
                gs = mfma_f64(W[3][1][nl][row], z.y, gs);
            }
        }
        // contract the pairs: components along a*, b*, c*, then Cartesian
        double fa = 0.0, fb = 0.0, fc = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            double c, s;
            rs_phase(X[v], Y[v], c, s);
            const double t = c * hc[v] + s * hs[v];
            fa += dl[v] * t;
            fb += dm[v] * t;
            fc += c * gc[v] + s * gs[v];
        }
        fa += __shfl_xor(fa, 16, 64);
        fb += __shfl_xor(fb, 16, 64);
        fc += __shfl_xor(fc, 16, 64);
        fa += __shfl_xor(fa, 32, 64);
        fb += __shfl_xor(fb, 32, 64);
        fc += __shfl_xor(fc, 32, 64);
        if (ok && quad < 3) {
            const double e = R.rc[3 * quad] * fa + R.rc[3 * quad + 1] * fb + R.rc[3 * quad + 2] * fc;
            Fpart[((long)g * 6 + 3 * set + quad) * P.n + j] = -TWOPI * e;
        }
    }
}

// Sum the field partials over the k chunks and scale (ewald1p.f:941-976): efdd =
// scale * sum + self term; with CHG also efdc = scale * sum (iloop = 1), at the sites that
// can carry a dipole.  Element (component q, site j) = q * nrow + j, 64 per block.
template <bool CHG>
__global__ __launch_bounds__(256) void k_el_kfield_reduce(ElecDev P, const double* __restrict__ Fpart,
                                                          const double* __restrict__ dip, double* __restrict__ efdd,
                                                          double* __restrict__ efdc, const double* __restrict__ state)
{
    if (!CHG && state[2] != 0.0) return;
    const int nrow = P.nrow;
    const int nq = CHG ? 6 : 3;
    const int t = blockIdx.x * 64 + (threadIdx.x & 63);
    const bool valid = t < nq * nrow;
    const int q = valid ? t / nrow : 0, j = valid ? t - q * nrow : 0;
    const double sum = chunk_sum64(Fpart, 6L * P.n, P.fchunks, (long)q * P.n + j, valid);
    if (threadIdx.x >= 64 || !valid) return;
    if (q < 3) {
        const bool pol = site_polr2(P, j) > 1.e-6;
        efdd[3 * j + q] = (pol ? P.scale * sum : 0.0) + P.self_dd * dip[3 * j + q];
    } else {
        efdc[3 * j + q - 3] = P.scale * sum;
    }
}

// ============================================================ solver iteration ======

// emu for a row per WPR wavefronts, blocks of four.  With cgblk (the conjugate-gradient
// solver's partials, cgnb blocks), the solver's stopping test for iteration `it` comes first
// (cg_step; block 0 records the scalars) and the kernel does nothing once the dipoles have
// converged.
template <int WPR>
__global__ __launch_bounds__(256) void k_el_emu(ElecDev P, const double* __restrict__ x, const double* __restrict__ y,
                                                const double* __restrict__ z, const int* __restrict__ nbrP,
                                                const int* __restrict__ cntP, const double2* __restrict__ tens,
                                                const double* __restrict__ tin,
                                                const double* __restrict__ dip, double* __restrict__ emu,
                                                double* __restrict__ state, const double* __restrict__ cgblk, int cgnb,
                                                int it)
{
    if (state[2] != 0.0) return;
    if (cgblk && cg_step(P, it, cgnb, cgblk, state, blockIdx.x == 0 && threadIdx.x < 64)) return;
    constexpr int T = 64 * WPR;
    emu_row<WPR>(P, blockIdx.x * (4 / WPR) + threadIdx.x / T, threadIdx.x % T, x, y, z, nbrP, cntP, tens, tin, dip, emu);
}

// SOR update (iter.f:58-89) and per-block sums of |dmu|^2 and of the dipole count.
__global__ __launch_bounds__(256) void k_el_sor(ElecDev P, const double* __restrict__ efk,
                                                const double* __restrict__ emu, const double* __restrict__ efdd,
                                                const double* __restrict__ efdc, double* __restrict__ dip,
                                                double* __restrict__ blk, const double* __restrict__ state)
{
    if (state[2] != 0.0) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double v[2] = {0.0, 0.0};
    if (i < P.nrow) {
        const double p2 = site_polr2(P, i);
        if (p2 > P.toler) {
            const double oldfac = P.omega, fac = 1.0 - oldfac;
            double dd = 0.0;
            for (int q = 0; q < 3; ++q) {
                const double old = dip[3 * i + q];
                const double nw = oldfac * old + fac * p2 *
                                                      (efk[3 * i + q] + emu[3 * i + q] + efdd[3 * i + q] +
                                                       efdc[3 * i + q] + 0.0) /
                                                      R4PIE0;
                dip[3 * i + q] = nw;
                dd += (nw - old) * (nw - old);
            }
            v[0] = dd;
            v[1] = 1.0;
        }
    }
    block_sum_store(v, blk + 2 * blockIdx.x);
}

// Convergence test (iter.f:95-101): state = [iterations, rms dmu, done, ...].
__global__ __launch_bounds__(64) void k_el_converge(ElecDev P, int nb, const double* __restrict__ blk,
                                                    double* __restrict__ state)
{
    if (state[2] != 0.0) return;
    double s = 0.0, c = 0.0;
    for (int b = threadIdx.x; b < nb; b += 64) {
        s += blk[2 * b];
        c += blk[2 * b + 1];
    }
    s = wsum(s);
    c = wsum(c);
    if (threadIdx.x == 0) {
        if (c == 0.0) c = 1.0;
        const double delta = sqrt(s / c);
        state[0] += 1.0;
        state[1] = delta;
        if (delta <= P.toler) state[2] = 1.0;
    }
}


// ==================================================== conjugate-gradient solver ======
// The induced dipoles solve A mu = E0 with A = D - T, D = r4pie0 / polr2 (per site), T the
// dipole-field operator (emu + efdd) and E0 = efk + efdc.  A is symmetric positive definite
// for Thole-damped dipoles, so preconditioned conjugate gradients reach the SOR fixed point
// of iter.f in far fewer iterations.  The preconditioner M is block-Jacobi over waters: the
// 9 x 9 block of each water's O, H1, H2 dipoles, which holds the strong intramolecular
// couplings (half the iterations of a diagonal preconditioner at liquid density).  The
// stopping test is the reference's: the RMS of the step an SOR update would take from the
// current dipoles, (1 - omega) * rms(polr2 r / r4pie0), against toler (iter.f:95-101).
//
// The iteration is the Chronopoulos-Gear form of preconditioned conjugate gradients
// (A. T. Chronopoulos and C. W. Gear, J. Comput. Appl. Math. 25 (1989) 153-168), in which
// both inner products of an iteration are taken after its vector update, so that one
// iteration is one application of A and one fused update with a single set of block
// partials:
//   n = A m
//   z = n + beta z,  q = m + beta q,  s = w + beta s,  p = u + beta p
//   mu += alpha p,  r -= alpha s,  u -= alpha q,  w -= alpha z,  m = M^-1 w
//   partials of g = r.u and d = w.u, from which cg_step forms the next alpha and beta
// (u = M^-1 r, w = A u, s = A p, q = M^-1 s, z = A q throughout).  It starts from
// r = E0 - A mu0, u = M^-1 r and one extra application of A for w = A u.  T mu, which the
// final passes need, follows mu as T mu += alpha (D p - s).  The scalars need no grid-wide synchronization:
// the first kernel of each iteration sums the update's block partials in every wavefront
// (cg_step) and its first block records them for the update.

// The reciprocal fields of the start dipoles (efdd, with the self term) and of the charges (efdc)
// from their chunk partials, as k_el_kfield_reduce<true>; r = E0 + T mu0 - D mu0 (T mu0 = emu +
// efdd), u = M^-1 r, T mu = T mu0; the first application of A goes to m = u; z, q, s, p start at
// zero.  A block takes CG_WPB waters, a row per lane, as k_cg_update: a quarter of the chunks per
// wavefront, then the first wavefront has the rows.
#define CG_WPB 7
__global__ __launch_bounds__(256) void k_cg_init(ElecDev P, const double* __restrict__ Fpart,
                                                 const double* __restrict__ efk, double* __restrict__ efdc,
                                                 const double* __restrict__ emu, double* __restrict__ efdd,
                                                 const double* __restrict__ dip, const double* __restrict__ minv,
                                                 double* __restrict__ r, double* __restrict__ u, double* __restrict__ m,
                                                 double* __restrict__ z, double* __restrict__ qv,
                                                 double* __restrict__ sv, double* __restrict__ pv,
                                                 double* __restrict__ tmu)
{
    __shared__ double part[4][2][64];
    __shared__ double rs[64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wl = lane / 9, i = lane - 9 * wl;
    const int w = blockIdx.x * CG_WPB + wl;
    const bool act = lane < 9 * CG_WPB && w < P.nw;
    const int o = 9 * w + i, j = 3 * w + i / 3, c = i % 3;
    const double p2 = act ? site_polr2(P, j) : 0.0;
    const bool on = act && p2 > P.toler;
    double sd = 0.0, sc = 0.0;
    if (act) {
        const int c0 = (P.fchunks * wave) / 4, c1 = (P.fchunks * (wave + 1)) / 4;
        const double* f = Fpart + (long)c * P.n + j;
        const long cs = 6L * P.n;
#pragma unroll 4
        for (int ch = c0; ch < c1; ++ch) {
            sd += f[ch * cs];
            sc += f[ch * cs + 3L * P.n];
        }
    }
    part[wave][0][lane] = sd;
    part[wave][1][lane] = sc;
    __syncthreads();
    double rr = 0.0;
    if (wave == 0 && act) {
        sd = ((part[0][0][lane] + part[1][0][lane]) + part[2][0][lane]) + part[3][0][lane];
        sc = ((part[0][1][lane] + part[1][1][lane]) + part[2][1][lane]) + part[3][1][lane];
        const double mu = dip[o];
        const double ed = (p2 > 1.e-6 ? P.scale * sd : 0.0) + P.self_dd * mu, ec = P.scale * sc;
        const double t = emu[o] + ed;
        efdd[o] = ed;
        efdc[o] = ec;
        tmu[o] = t;
        rr = on ? (efk[o] + ec + t) - R4PIE0 * mu / p2 : 0.0;
        r[o] = rr;
        z[o] = 0.0;
        qv[o] = 0.0;
        sv[o] = 0.0;
        pv[o] = 0.0;
    }
    if (wave == 0) rs[lane] = rr;
    __syncthreads();
    if (wave == 0 && act) {
        double uu = 0.0;
        if (on) {
            const double* mi = minv + 45L * w;
#pragma unroll
            for (int k = 0; k < 9; ++k) uu += mi[tri9(i, k)] * rs[9 * wl + k];
        }
        u[o] = uu;
        m[o] = uu;
    }
}

// The vector update of an iteration (INIT: of the start) from n = A m, with A m formed here
// from the real-space field emu and the reciprocal field's chunk partials (efdd = scale *
// sum + self term, as k_el_kfield_reduce).  A block takes CG_WPB waters (63 rows, one per
// lane): its four wavefronts first add a quarter of the field chunks each, in chunk order,
// and the first wavefront adds the quarters in order and updates the rows; the new w of
// each water is shared through LDS for m = M^-1 w.  Block partials (r.u, w.u,
// |polr2 r / r4pie0|^2, dipole count, max |m_i|) per water block.  INIT sets w = A u and
// leaves mu, r, u as they are.
template <bool INIT>
__global__ __launch_bounds__(256) void k_cg_update(ElecDev P, const double* __restrict__ Fpart,
                                                   const double* __restrict__ emu, const double* __restrict__ minv,
                                                   double* __restrict__ m, double* __restrict__ dip,
                                                   double* __restrict__ r, double* __restrict__ u,
                                                   double* __restrict__ wv, double* __restrict__ z,
                                                   double* __restrict__ qv, double* __restrict__ sv,
                                                   double* __restrict__ pv, double* __restrict__ tmu,
                                                   double* __restrict__ blk,
                                                   const double* __restrict__ state)
{
    const double done = state[2];
    const double alpha = INIT ? 0.0 : state[4], beta = INIT ? 0.0 : state[5];
    const int tid = threadIdx.x;
    __shared__ double part[4][64];
    __shared__ double ws[64];
    __shared__ double wmax[4];
    const int lane = tid & 63, wave = tid >> 6;
    const int wl = lane / 9, i = lane - 9 * wl;
    const int w = blockIdx.x * CG_WPB + wl;
    const bool act = lane < 9 * CG_WPB && w < P.nw;
    const int o = act ? 9 * w + i : 0, j = 3 * w + i / 3, c = i % 3;
    const double p2 = act ? site_polr2(P, j) : 0.0;
    const bool on = act && p2 > P.toler;
    // every load of the row is started before the first wait
    double mm = 0.0, em = 0.0, r0 = 0.0, u0 = 0.0, w0 = 0.0, z0 = 0.0, q0 = 0.0, s0 = 0.0, p0 = 0.0, d0 = 0.0, t0 = 0.0;
    double mi[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) mi[k] = 0.0;
    if (wave == 0 && on) {
        mm = m[o];
        em = emu[o];
        r0 = r[o];
        u0 = u[o];
        if (!INIT) {
            w0 = wv[o];
            z0 = z[o];
            q0 = qv[o];
            s0 = sv[o];
            p0 = pv[o];
            d0 = dip[o];
            t0 = tmu[o];
        }
#pragma unroll
        for (int k = 0; k < 9; ++k) mi[k] = minv[45L * w + tri9(i, k)];
    }
    {
        // this wavefront's quarter of the field chunks
        double sum = 0.0;
        if (on && p2 > 1.e-6) {
            const int c0 = (P.fchunks * wave) / 4, c1 = (P.fchunks * (wave + 1)) / 4;
            const double* f = Fpart + (long)c * P.n + j;
            const long cs = 6L * P.n;
#pragma unroll 8
            for (int ch = c0; ch < c1; ++ch) sum += f[ch * cs];
        }
        if (done != 0.0) return;
        part[wave][lane] = sum;
    }
    __syncthreads();
    double rr = 0.0, uu = 0.0, wn = 0.0;
    if (wave == 0 && on) {
        const double sum = ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane];
        const double nv = R4PIE0 * mm / p2 - (em + (p2 > 1.e-6 ? P.scale * sum : 0.0) + P.self_dd * mm);
        if (INIT) {
            wn = nv;
            wv[o] = wn;
            rr = r0;
            uu = u0;
        } else {
            const double zz = nv + beta * z0;
            const double qq = mm + beta * q0;
            const double ss = w0 + beta * s0;
            const double pp = u0 + beta * p0;
            z[o] = zz;
            qv[o] = qq;
            sv[o] = ss;
            pv[o] = pp;
            dip[o] = d0 + alpha * pp;
            tmu[o] = t0 + alpha * (R4PIE0 * pp / p2 - ss);
            rr = r0 - alpha * ss;
            uu = u0 - alpha * qq;
            wn = w0 - alpha * zz;
            r[o] = rr;
            u[o] = uu;
            wv[o] = wn;
        }
    }
    if (wave == 0) ws[lane] = wn;
    __syncthreads();
    double mn = 0.0;
    if (wave == 0 && on) {
#pragma unroll
        for (int k = 0; k < 9; ++k) mn += mi[k] * ws[9 * wl + k];
        m[o] = mn;
    }
    const double zs = p2 * rr / R4PIE0;
    const bool row = wave == 0 && on;
    double v[4] = {rr * uu, wn * uu, row ? zs * zs : 0.0, (row && c == 0) ? 1.0 : 0.0};
    block_sum_store(v, blk + 5 * blockIdx.x);
    // max |m_i| of the block (a maximum: the same in any order)
    double a = fabs(mn);
    for (int o2 = 32; o2 > 0; o2 >>= 1) a = fmax(a, __shfl_xor(a, o2, 64));
    if (lane == 0) wmax[wave] = a;
    __syncthreads();
    if (tid == 0) blk[5 * blockIdx.x + 4] = fmax(fmax(wmax[0], wmax[1]), fmax(wmax[2], wmax[3]));
}

// The whole solve of a small system without reciprocal space in one launch by one block: the first
// application of A (init: to u, as k_cg_update<INIT>), then iterations it0 .. it0 + count - 1 as
// cg_step, emu_row and k_cg_update form them, until the dipoles have converged.  Everything an
// iteration needs stays on the CU: 16 lanes keep the radial factors and separations of a row's
// partners in registers (four each: the at most 61 partners of at most 63 rows), wavefront v the
// vectors of the waters 7 v .. 7 v + 6, and m, its field and the partials pass through LDS, where a
// barrier stands for a launch.  What a later launch continues from is written back.  Bound by
// the latency of the shuffles and barriers of an iteration.
// The solve of 9 waters, two launches to each of its about 17 iterations before: an evaluation
// 265 -> 232 us (of which the two- and three-body terms beside it now take the longer part); of 21
// waters 272 -> 236 us.  With rows passed in turn to 16 wavefronts that read the factors from
// memory each time: 240 us at 9 waters, 283 (268 by single launches) at 16.
#define CG_SOLVE_WATERS 21
__global__ __launch_bounds__(1024) void k_cg_solve(ElecDev P, bool init, int it0, int count,
                                                   const double* __restrict__ x, const double* __restrict__ y,
                                                   const double* __restrict__ z, const int* __restrict__ nbrP,
                                                   const int* __restrict__ cntP, const double2* __restrict__ tens,
                                                   const double* __restrict__ tin, const double* __restrict__ minv,
                                                   double* __restrict__ m, double* __restrict__ dip,
                                                   double* __restrict__ r, double* __restrict__ u,
                                                   double* __restrict__ wv, double* __restrict__ zv,
                                                   double* __restrict__ qv, double* __restrict__ sv,
                                                   double* __restrict__ pv, double* __restrict__ tmu,
                                                   double* __restrict__ blk, double* __restrict__ state)
{
    constexpr int NWV = (CG_SOLVE_WATERS + CG_WPB - 1) / CG_WPB;   // wavefronts with vector rows
    static_assert(16 * 3 * CG_SOLVE_WATERS <= 1024 && 3 * CG_SOLVE_WATERS - 3 <= 64, "");
    __shared__ double lm[9 * CG_SOLVE_WATERS], le[9 * CG_SOLVE_WATERS], lw[NWV][64], lb[5 * NWV], st[16];
    __shared__ double lt[36 * CG_SOLVE_WATERS];
    if (state[2] != 0.0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nb = (P.nw + CG_WPB - 1) / CG_WPB;
    const int wl = lane / 9, i = lane - 9 * wl;
    const int w = wave * CG_WPB + wl;
    const bool act = wave < NWV && lane < 9 * CG_WPB && w < P.nw;
    const int o = act ? 9 * w + i : 0, c = i % 3;
    const double p2 = act ? site_polr2(P, 3 * w + i / 3) : 0.0;
    const bool on = act && p2 > P.toler;
    // the real-space row of these 16 lanes
    const int row = tid >> 4, rl = tid & 15;
    int pj[4];
    double t1[4], t2[4], d[4][3];
    {
        const int np = row < P.nrow ? cntP[row] : 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = rl + 16 * k;
            pj[k] = 0;
            t1[k] = t2[k] = d[k][0] = d[k][1] = d[k][2] = 0.0;
            if (e < np) {
                const long q = (long)row * P.capP + e;
                pj[k] = 3 * nbrP[q];
                t1[k] = tens[q].x;
                t2[k] = tens[q].y;
                (void)sep(P, x, y, z, row, nbrP[q], d[k]);
            }
        }
    }
    // its two excluded partners of the same water, on lanes 0 and 1 (see emu_row)
    int xj = -1, xt = 0;
    if (row < P.nrow && rl < 2) {
        const int rw = row / 3, si = row - 3 * rw, pt = rl < si ? rl : rl + 1;
        const int a = min(si, pt), b = max(si, pt);
        if (site_polr2(P, 3 * rw + pt) > 1.e-6) xj = 3 * (3 * rw + pt);
        xt = 36 * rw + 6 * (a == 0 ? b - 1 : 3);
    }
    for (int e = tid; e < 36 * P.nw; e += 1024) lt[e] = tin[e];
    double mm = 0.0, rr = 0.0, uu = 0.0, wn = 0.0, zz = 0.0, qq = 0.0, ss = 0.0, pp = 0.0, dd = 0.0, tt = 0.0;
    double mi[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) mi[k] = 0.0;
    if (act) {
        mm = m[o];
        lm[o] = mm;
    }
    if (on) {
        rr = r[o];
        uu = u[o];
        zz = zv[o];
        qq = qv[o];
        ss = sv[o];
        pp = pv[o];
        dd = dip[o];
        tt = tmu[o];
        if (!init) wn = wv[o];
#pragma unroll
        for (int k = 0; k < 9; ++k) mi[k] = minv[45L * w + tri9(i, k)];
    }
    if (tid < 16) st[tid] = state[tid];
    if (!init && tid < 5 * nb) lb[tid] = blk[tid];
    __syncthreads();
    for (int it = init ? it0 - 1 : it0; it < it0 + count; ++it) {
        const bool first = it < it0;
        // (the wavefront that records is past its last use of st; the others read it after a barrier)
        if (!first && cg_step(P, it, nb, lb, st, wave == 0)) break;
        {
            double e[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double mx = lm[pj[k]], my = lm[pj[k] + 1], mz = lm[pj[k] + 2];
                const double f = t2[k] * (d[k][0] * mx + d[k][1] * my + d[k][2] * mz);
                e[0] += f * d[k][0] - t1[k] * mx;
                e[1] += f * d[k][1] - t1[k] * my;
                e[2] += f * d[k][2] - t1[k] * mz;
            }
            if (xj >= 0) {
                const double* dt = lt + xt;
                const double mx = lm[xj] * R4PIE0, my = lm[xj + 1] * R4PIE0, mz = lm[xj + 2] * R4PIE0;
                e[0] += dt[0] * mx + dt[1] * my + dt[2] * mz;
                e[1] += dt[1] * mx + dt[3] * my + dt[4] * mz;
                e[2] += dt[2] * mx + dt[4] * my + dt[5] * mz;
            }
            for (int q = 0; q < 3; ++q)
                for (int k = 8; k > 0; k >>= 1) e[q] += __shfl_xor(e[q], k, 16);
            if (rl == 0 && row < P.nrow)
                for (int q = 0; q < 3; ++q) le[3 * row + q] = e[q];
        }
        __syncthreads();
        if (on) {
            const double nv = R4PIE0 * mm / p2 - (le[o] + P.self_dd * mm);
            if (first) {
                wn = nv;
            } else {
                const double alpha = st[4], beta = st[5];
                zz = nv + beta * zz;
                qq = mm + beta * qq;
                ss = wn + beta * ss;
                pp = uu + beta * pp;
                dd += alpha * pp;
                tt += alpha * (R4PIE0 * pp / p2 - ss);
                rr -= alpha * ss;
                uu -= alpha * qq;
                wn -= alpha * zz;
            }
        }
        // the new w of a water's rows, which share a wavefront
        if (wave < NWV) lw[wave][lane] = on ? wn : 0.0;
        __syncthreads();
        if (wave < nb) {
            double mn = 0.0;
            if (on) {
#pragma unroll
                for (int k = 0; k < 9; ++k) mn += mi[k] * lw[wave][9 * wl + k];
                mm = mn;
                lm[o] = mn;
            }
            const double zs = on ? p2 * rr / R4PIE0 : 0.0;
            const double v0 = wsum(rr * uu), v1 = wsum(on ? wn * uu : 0.0), v2 = wsum(zs * zs),
                         v3 = wsum(on && c == 0 ? 1.0 : 0.0);
            double a = fabs(mn);
            for (int o2 = 32; o2 > 0; o2 >>= 1) a = fmax(a, __shfl_xor(a, o2, 64));
            if (lane == 0) {
                lb[5 * wave] = v0;
                lb[5 * wave + 1] = v1;
                lb[5 * wave + 2] = v2;
                lb[5 * wave + 3] = v3;
                lb[5 * wave + 4] = a;
            }
        }
        __syncthreads();
    }
    __syncthreads();
    if (on) {
        m[o] = mm;
        r[o] = rr;
        u[o] = uu;
        wv[o] = wn;
        zv[o] = zz;
        qv[o] = qq;
        sv[o] = ss;
        pv[o] = pp;
        dip[o] = dd;
        tmu[o] = tt;
    }
    if (tid < 5 * nb) blk[tid] = lb[tid];
    if (tid < 16) state[tid] = st[tid];
}


// ================================================================ final passes ======

// Per-k scalars of the final reciprocal pass (ewald1p.f:696-730): akk (Qc^2 + Qs^2),
// akk |summu|^2 and the six omg components; block partials [nb][8].  Also stores, per k,
// the constants the site pass needs in kf[k][16].  The structure factors of mu_x, mu_y, mu_z
// and of the charges (sets 0..3 of Spart) are added over the chunks here.
__global__ __launch_bounds__(256) void k_el_kscal(ElecDev P, const double* __restrict__ kv,
                                                  const double* __restrict__ Spart, double* __restrict__ kf,
                                                  double* __restrict__ blk)
{
    // four lanes per k, a set of structure factors each
    const int k = blockIdx.x * 64 + threadIdx.x / 4, w = threadIdx.x & 3;
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    double mc = 0.0, ms = 0.0;
    if (k < P.K) {
        const RsPlan& R = P.rs;
        const int pos = R.kpos[k], pg = pos >> 8, n = (pos >> 1) & 127;
        const long slot = RS_SLOT(R.ntiles), cs = slot * R.ng;
        const double* base = Spart + ((long)w * R.nchq * R.ng + (pg >> 4)) * slot;
        if (n == 0) {
            const double* q = base + 512L * R.ntiles + (pg & 15);
            for (int ch = 0; ch < R.nchq; ++ch, q += cs) {
                mc += q[0];
                ms += q[16];
            }
        } else {
            double u[4];
            rs_sums(base, cs, R.nchq, pg & 15, n, u);
            mc = (pos & 1) ? u[2] : u[0];
            ms = (pos & 1) ? u[3] : u[1];
        }
    }
    const double Mc[3] = {__shfl(mc, 0, 4), __shfl(mc, 1, 4), __shfl(mc, 2, 4)}, Qc = __shfl(mc, 3, 4);
    const double Ms[3] = {__shfl(ms, 0, 4), __shfl(ms, 1, 4), __shfl(ms, 2, 4)}, Qs = __shfl(ms, 3, 4);
    if (k < P.K && w == 0) {
        const double kx = kv[8 * k], ky = kv[8 * k + 1], kz = kv[8 * k + 2], akk = kv[8 * k + 3];
        const double akv = kv[8 * k + 4];
        const double kk[3] = {kx, ky, kz};
        const double skdmuckrs = kx * Mc[0] + ky * Mc[1] + kz * Mc[2];
        const double skdmuskrs = kx * Ms[0] + ky * Ms[1] + kz * Ms[2];
        const double summu1 = Qc - skdmuskrs, summu2 = Qs + skdmuckrs;
        v[0] = akk * (Qc * Qc + Qs * Qs);
        v[1] = akk * (summu1 * summu1 + summu2 * summu2);
        const double virprs = akv * (summu1 * summu1 + summu2 * summu2);
        const int ia[6] = {0, 1, 2, 0, 0, 1}, ib[6] = {0, 1, 2, 1, 2, 2};
        for (int t = 0; t < 6; ++t)
            v[2 + t] = -virprs * kk[ia[t]] * kk[ib[t]] - 2.0 * akk * kk[ia[t]] * Ms[ib[t]] * summu1 +
                       2.0 * akk * kk[ia[t]] * Mc[ib[t]] * summu2;
        // what the site pass multiplies with the phases of this k, akk taken in
        double* f = kf + 16 * k;
        f[0] = akk * summu1;
        f[1] = akk * summu2;
        f[2] = akk * Qc;
        f[3] = akk * Qs;
        for (int q = 0; q < 3; ++q) {
            f[4 + q] = akk * Mc[q];
            f[7 + q] = akk * Ms[q];
        }
        f[10] = kv[8 * k + 5];   // akv2
    }
    block_sum_store(v, blk + 8 * blockIdx.x);
}

// Final reciprocal pass per site over a chunk of runs (ewald1p.f:550-693, 771-825): forces, ESP
// parts vesp_k / vesp_dc_k, per-atom energy and per-atom stress (without the final prefactors).
// Partials Fpart[chunk][16][n]: f(3), vk, vdck, e, s(9).
//
// With S1 = Qc - k.Ms, S2 = Qs + k.Mc, km = k.mu and the phases c, s of site j, everything follows
// from A = akk (c S1 + s S2) and B = akk (c S2 - s S1):
//   force   -sum k (q B - km A),   vk + vdck = sum A,
//   stress  akk [D_ab T - akv2 k_a k_b T + k_a X_b],  akk T = q A + km B,
//   akk X_b = (s q + c km) akk Mc_b - (c q - s km) akk Ms_b + B mu_b.
// Along a run k = k0 + t g (g = 2 pi c*, t = 0..7): the sums over t carry the moments t^0, t^1
// (and t^2 of akv2 T) only, and are multiplied with k0 once per run and with g once per chunk.
// That leaves 40 FP64 instructions per (k, site) instead of 66, and 6 reads of 16 bytes from LDS
// per (k, wavefront) instead of 9, which had taken the LDS as long as the arithmetic took the
// SIMDs: 512 waters 73.6 -> 50.1 us, 2048 waters 767 -> 479 us (430 us of arithmetic at four
// cycles an instruction).  Slower: two sites per thread (284 registers, one wavefront to a SIMD:
// 61 and 738 us), four wavefronts to a SIMD (spills: 107 and 1226 us), the factors by scalar loads
// (their latency: 99 and 828 us).
__global__ __launch_bounds__(256) void k_el_kfinal(ElecDev P, const int4* __restrict__ runs,
                                                   const int* __restrict__ runk, const double* __restrict__ phc,
                                                   const double* __restrict__ phs, const double* __restrict__ kv,
                                                   const double* __restrict__ kf, const double* __restrict__ chge,
                                                   const double* __restrict__ dip, double* __restrict__ Fpart)
{
    const int j = blockIdx.x * 256 + threadIdx.x;
    const int chunk = blockIdx.y;
    const int r0 = chunk * P.rpc, r1 = min(P.nrun, r0 + P.rpc);
    // the chunk's factors, 12 doubles a k
    extern __shared__ double lds[];
    double2* sk = (double2*)lds;
    const int kb = runk[r0], nk = (r1 < P.nrun ? runk[r1] : P.K) - kb;
    for (int e = threadIdx.x; e < 6 * nk; e += 256) {
        const int kk = e / 6;
        sk[e] = ((const double2*)kf)[8L * (kb + kk) + e - 6 * kk];
    }
    __syncthreads();
    if (j >= P.n) return;
    const int ks = P.kstride;
    const bool pol = site_polr2(P, j) > 1.e-6;
    const double q = chge[j];
    const double mu[3] = {pol ? dip[3 * j] : 0.0, pol ? dip[3 * j + 1] : 0.0, pol ? dip[3 * j + 2] : 0.0};
    const double g[3] = {TWOPI * P.rs.rc[2], TWOPI * P.rs.rc[5], TWOPI * P.rs.rc[8]};
    const double kg = mu[0] * g[0] + mu[1] * g[1] + mu[2] * g[2];
    const double c1 = phc[((long)2 * ks + 1) * P.n + j], s1 = phs[((long)2 * ks + 1) * P.n + j];
    double vk_ = 0.0, va_ = 0.0;
    // sums with k0 (per run) and those left for g
    double F[3] = {0, 0, 0}, R[3] = {0, 0, 0}, Y[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, U[6] = {0, 0, 0, 0, 0, 0};
    double Fg = 0.0, Rg = 0.0, Yg[3] = {0, 0, 0}, Ug[3] = {0, 0, 0}, Ugg = 0.0;
    for (int r = r0; r < r1; ++r) {
        const int4 run = runs[r];
        const int l = run.x, m = run.y, n0 = run.z, cnt = run.w;
        const int k = runk[r];
        const double kx = kv[8L * k], ky = kv[8L * k + 1], kz = kv[8L * k + 2];
        const int am = abs(m), an0 = abs(n0);
        double c, s;
        run_phase(phc[(long)l * P.n + j], phs[(long)l * P.n + j], phc[((long)ks + am) * P.n + j],
                  phs[((long)ks + am) * P.n + j], phc[((long)2 * ks + an0) * P.n + j],
                  phs[((long)2 * ks + an0) * P.n + j], m, n0, c, s);
        const double km0 = mu[0] * kx + mu[1] * ky + mu[2] * kz;
        double f0 = 0.0, f1 = 0.0, b0 = 0.0, b1 = 0.0, u0 = 0.0, u1 = 0.0, u2 = 0.0;
        double y0[3] = {0.0, 0.0, 0.0}, y1[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int t = 0; t < EL_RUN; ++t) {
            if (t >= cnt) break;
            const double2* fl = sk + 6 * (k - kb + t);
            const double2 f01 = fl[0], f23 = fl[1], f45 = fl[2], f67 = fl[3], f89 = fl[4];
            const double f[11] = {f01.x, f01.y, f23.x, f23.y, f45.x, f45.y, f67.x, f67.y, f89.x, f89.y, fl[5].x};
            const double km = km0 + t * kg;
            const double A = c * f[0] + s * f[1], B = c * f[1] - s * f[0];
            const double w = q * B - km * A;
            const double u = (q * A + km * B) * f[10];
            const double a = s * q + c * km, b = c * q - s * km;
            vk_ += c * f[2] + s * f[3];
            va_ += A;
            f0 += w;
            f1 += t * w;
            b0 += B;
            b1 += t * B;
            u0 += u;
            u1 += t * u;
            u2 += (t * t) * u;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double y = a * f[4 + d] - b * f[7 + d];
                y0[d] += y;
                y1[d] += t * y;
            }
            const double cn = c * c1 - s * s1;
            s = s * c1 + c * s1;
            c = cn;
        }
        F[0] += kx * f0;
        F[1] += ky * f0;
        F[2] += kz * f0;
        Fg += f1;
        R[0] += kx * b0;
        R[1] += ky * b0;
        R[2] += kz * b0;
        Rg += b1;
        const double ux = kx * u0, uy = ky * u0, uz = kz * u0;
        U[0] += kx * ux;
        U[1] += kx * uy;
        U[2] += kx * uz;
        U[3] += ky * uy;
        U[4] += ky * uz;
        U[5] += kz * uz;
        Ug[0] += kx * u1;
        Ug[1] += ky * u1;
        Ug[2] += kz * u1;
        Ugg += u2;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            Y[d] += kx * y0[d];
            Y[3 + d] += ky * y0[d];
            Y[6 + d] += kz * y0[d];
            Yg[d] += y1[d];
        }
    }
    double acc[15];
    double D = q * va_;   // sum akk T
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        acc[a] = -(F[a] + g[a] * Fg);
        R[a] += g[a] * Rg;
        D += mu[a] * R[a];
    }
    acc[3] = vk_;
    acc[4] = va_ - vk_;
    acc[5] = q * vk_;
    const int gi[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const double G = U[gi[a][b]] + g[b] * Ug[a] + g[a] * Ug[b] + g[a] * g[b] * Ugg;
            acc[6 + 3 * a + b] = (a == b ? D : 0.0) - G + (Y[3 * a + b] + g[a] * Yg[b]) + mu[b] * R[a];
        }
    double* out = Fpart + (long)chunk * 16 * P.n;
#pragma unroll
    for (int t = 0; t < 15; ++t) out[(long)t * P.n + j] = acc[t];
}

// Sums of the final pass's site partials over the k chunks: ksum[t][j] for the 15 site
// quantities t of k_el_kfinal, 64 elements (t, j) per block.
__global__ __launch_bounds__(256) void k_el_ksum(ElecDev P, const double* __restrict__ Fpart,
                                                 double* __restrict__ ksum)
{
    const long e = (long)blockIdx.x * 64 + (threadIdx.x & 63);
    const bool valid = e < 15L * P.n;
    const double v = chunk_sum64(Fpart, 16L * P.n, P.kchunks, e, valid);
    if (threadIdx.x < 64 && valid) ksum[e] = v;
}

// Real-space pair terms of one row (ewald2p.f:118-600; nthole = 4, lacs, lads): forces,
// per-atom energy, ESP parts, and the row's force-matrix contraction W_i (real partners
// only; for an M-site row the partner sums sum_j F and sum_j F (x) x_j, from which the
// M-row redistribution builds W of O, H1, H2).  Each pair is seen from both of its rows,
// so block partials carry half of each pair's energy, virial and stress.  One wavefront
// per site; partials [n][8]: energy, virial, stress (xx xy xz yy yz zz).
//
// Bound by FP64 arithmetic.  The smeared charge-charge energy (exp(-x) - x^1/4 Gamma(3/4)
// Q(3/4, x)) / r, x = ascc u^4, is the dear part (the reference's continued fraction: tens of
// divisions) and below 1e-26 of 1 / r from x = PAIR_XNEAR on, under a hundred-thousandth of the
// last place of erfc(alpha r) / r at any real cut-off, so it is left out there: that leaves the
// partners within 2.3 (H-H) to 3.9 A (O-O), a few per row, which are gathered in LDS and taken
// 64 at a time instead of one or two lanes of each step.  With one exp less, the powers from
// the host's table and the sums in 25 exchanges: 365 -> 107 us for a 701-water cluster, 46 -> 30
// at 512 waters, 161 -> 94 at 2 048.
#define PAIR_XNEAR 60.0
__global__ __launch_bounds__(64) void k_el_pairs(ElecDev P, const double* __restrict__ x,
                                                 const double* __restrict__ y, const double* __restrict__ z,
                                                 const double* __restrict__ chge, const double* __restrict__ dip,
                                                 const double* __restrict__ tab, const int* __restrict__ nbrA,
                                                 const int* __restrict__ cntA, double g34, double gln34,
                                                 double* __restrict__ f2, double* __restrict__ e2,
                                                 double* __restrict__ vr, double* __restrict__ vdcr,
                                                 double* __restrict__ w2, double* __restrict__ fmsum,
                                                 double* __restrict__ fmx, double* __restrict__ blk)
{
    __shared__ double2 near[128];                      // (x, qj / r) of near partners waiting
    __shared__ double sums[24];
    const int i = blockIdx.x;
    const int lane = threadIdx.x;
    if (i >= P.n) return;
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const double qi = chge[i];
    const int ti = site_type(P, i);
    const bool poli = site_polr2(P, i) > 1.e-6;
    const double mi[3] = {dip[3 * i], dip[3 * i + 1], dip[3 * i + 2]};
    const double xi[3] = {x[i], y[i], z[i]};
    const bool mrow = i >= P.nreal;
    // [0..2] force, [3] energy / 2, [4] vr, [5] vdcr, [6..14] W, [15..20] stress, [21..23] fm; without
    // R4PIE0 until the end
    double v[24];
#pragma unroll
    for (int t = 0; t < 24; ++t) v[t] = 0.0;
    double smq = 0.0;                                  // sum of q_j sm
    int nnear = 0;
    auto smear = [&](int cnt) {
        if (lane < cnt) {
            const double2 p = near[lane];
            smq += (exp(-p.x) - sqrt(sqrt(p.x)) * g34 * gammq_nr(0.75, p.x, gln34)) * p.y;
        }
    };
    const int na = cntA[i];
    for (int base = 0; base < na; base += 64) {
        const int s = base + lane;
        const int j = s < na ? nbrA[(long)i * P.capA + s] : i;
        double d[3] = {0.0, 0.0, 0.0};
        double rsq = P.rcut * P.rcut;
        if (s < na) rsq = sep(P, x, y, z, i, j, d);
        const bool in = s < na && P.rcut * P.rcut > rsq;
        double xc = PAIR_XNEAR, qr = 0.0;
        if (in) {
            const double rrr = sqrt(rsq);
            double bbb[4];
            table_interp(P, tab, rrr, bbb);
            const double rri = 1.0 / rrr, rsqi = rri * rri;
            const double r3i = rri * rsqi, r5i = r3i * rsqi;
            const double qj = chge[j];
            const double u = rrr * P.bbi[ti][site_type(P, j)];
            const double u4 = (u * u) * (u * u);
            const double espdum = bbb[0] + rri;
            xc = P.ascc * u4;
            qr = qj * rri;
            const double dumd = exp(-P.ascd * u4);
            const double dumc = P.ascc == P.ascd ? dumd : exp(-xc);
            const double cicj = qi * qj;
            double ffac = cicj * (r3i * (1.0 - dumc) + bbb[1]);
            const double mj[3] = {dip[3 * j], dip[3 * j + 1], dip[3 * j + 2]};
            const double rdmui = mi[0] * d[0] + mi[1] * d[1] + mi[2] * d[2];
            const double rdmuj = mj[0] * d[0] + mj[1] * d[1] + mj[2] * d[2];
            const double dumd2 = (1.0 + (4.0 / 3.0) * (P.ascd * u4)) * dumd;
            const double b1 = bbb[1] + r3i * (1.0 - dumd);
            ffac -= (qj * rdmui - qi * rdmuj) * (3.0 * r5i * (1.0 - dumd2) + bbb[2]);
            double dfi = b1 * qj, dfj = -b1 * qi;
            if (poli && site_polr2(P, j) > 1.e-6) {
                const double dpidpj = mi[0] * mj[0] + mi[1] * mj[1] + mi[2] * mj[2];
                const double rr2 = rdmui * rdmuj;
                const double arob4 = P.athole * u4;
                const double dum1 = exp(-arob4);
                const double dum2 = (1.0 + (4.0 / 3.0) * arob4) * dum1;
                const double c3 = 3.0 * r5i * (1.0 - dum2) + bbb[2];
                // 4 a dum1 / b^4 = 4 arob4 dum1 / r^4
                const double dum34 = 4.0 * arob4 * dum1 * (rsqi * rsqi);
                ffac += dpidpj * (3.0 * r5i * (1.0 - dum1) + bbb[2] - rri * dum34) -
                        rr2 * (15.0 * (rsqi * r5i) * (1.0 - dum2) + bbb[3] - dum34 * (4.0 * arob4 - 1.0) * r3i);
                dfi += c3 * rdmuj;
                dfj += c3 * rdmui;
            }
            double fv[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                fv[q] = ffac * d[q] + dfi * mi[q] + dfj * mj[q];
                v[q] += fv[q];
            }
            v[3] += cicj * espdum;
            v[4] += qj * espdum;
            v[5] += rdmuj * b1;
            v[15] += d[0] * fv[0];
            v[16] += d[0] * fv[1];
            v[17] += d[0] * fv[2];
            v[18] += d[1] * fv[1];
            v[19] += d[1] * fv[2];
            v[20] += d[2] * fv[2];
            if (j < P.nreal) {
                // raw separations, or the partner's position for an M-site row
                const double xr[3] = {mrow ? x[j] : xi[0] - x[j], mrow ? y[j] : xi[1] - y[j], mrow ? z[j] : xi[2] - z[j]};
#pragma unroll
                for (int a = 0; a < 3; ++a) {
#pragma unroll
                    for (int b = 0; b < 3; ++b) v[6 + 3 * a + b] += fv[a] * xr[b];
                    v[21 + a] += fv[a];
                }
            }
        }
        const bool isnear = xc < PAIR_XNEAR;
        const unsigned long long bn = __ballot(isnear);
        if (isnear) near[nnear + __popcll(bn & below)] = make_double2(xc, qr);
        nnear += __popcll(bn);
        __syncthreads();
        if (nnear >= 64) {
            smear(64);
            const double2 rest = near[64 + lane];
            __syncthreads();
            near[lane] = rest;
            nnear -= 64;
            __syncthreads();
        }
    }
    smear(nnear);
    v[4] -= smq;
    v[3] = 0.5 * (v[3] - qi * smq);
#pragma unroll
    for (int t = 15; t < 21; ++t) v[t] *= 0.5;
    int k;
    const double t = R4PIE0 * wave_sum24(v, lane, k);
    if (k < 24) sums[k] = t;
    __syncthreads();
    if (lane < 3) f2[3 * i + lane] = sums[lane];
    if (lane == 3) e2[i] = sums[3];
    if (lane == 4) vr[i] = sums[4];
    if (lane == 5) vdcr[i] = sums[5];
    if (lane >= 6 && lane < 15) (mrow ? fmx : w2)[9 * i + lane - 6] = sums[lane];
    if (lane >= 15 && lane < 21) blk[8 * i + 2 + lane - 15] = sums[lane];
    if (lane >= 21 && lane < 24 && mrow) fmsum[3 * i + lane - 21] = sums[lane];
    // the virial is minus the trace of the stress (both halved)
    if (lane == 24) blk[8 * i] = sums[3];
    if (lane == 25) blk[8 * i + 1] = -(sums[15] + sums[18] + sums[20]);
}

// The end of an evaluation, four lanes per water (lane a: site O, H1, H2, M), 16 waters per
// wavefront.  In turn: the site's reciprocal results from the final pass's sums ksum, with the
// prefactors (ewald1p.f:941-1001; null: no reciprocal space); its polarization energy
// (coulomb_polar.f:58-103); the excluded pairs with the other three sites (ewald3p.f:80-391, every
// pair seen from both of its sites); the ESP (forces.f:876-880); the charge-derivative forces on
// O, H1, H2 (qdforce.f90:70-566; the charges do not depend on M); and the site forces and the
// per-real-atom outputs of the heat-current decomposition, with the M site's share moved onto
// O, H1, H2 (dlpoly_cmd.f:2583-2606, heatcurrent.f90:302-555): fout (3 per site; M forces moved
// when distribute != 0), eout (energy ew1p + ew2p + ew3p + polar), sout (ew1p stress), wout
// (force-matrix contraction; columns of real atoms only, diagonal entries skipped,
// heatcurrent.f90:541-555, 711-719).  emu + efdd is the dipoles' own field (efdd null: emu holds
// both).  Block partials [24]: polar, q^2, excluded pairs (energy, virial, stress 6), qd (virial,
// stress 6), the angular terms of the per-atom qd stresses (qdforce.f90:504-531, the ones recorded
// without HEAT_STRESS; 6).
// Bound by one lane's latency: six launches of one thread per water or site before (polar 4, sums 5,
// excluded pairs 18, ESP 5, qd 26, outputs 9 us at 512 waters), 16.7 us as one.
__global__ __launch_bounds__(64) void k_el_water_final(
    ElecDev P, int distribute, const double* __restrict__ x, const double* __restrict__ y, const double* __restrict__ z,
    const double* __restrict__ chge, const double* __restrict__ dip, const double* __restrict__ dg,
    const double* __restrict__ ksum, const double* __restrict__ efk, const double* __restrict__ efdc,
    const double* __restrict__ emu, const double* __restrict__ efdd, const double* __restrict__ f2,
    const double* __restrict__ e2, const double* __restrict__ vr, const double* __restrict__ vdcr,
    const double* __restrict__ w2, const double* __restrict__ fmsum, const double* __restrict__ fmx,
    double* __restrict__ e1, double* __restrict__ vesp, double* __restrict__ fout, double* __restrict__ eout,
    double* __restrict__ sout, double* __restrict__ wout, double* __restrict__ blk)
{
    const int lane = threadIdx.x, a = lane & 3;
    const int wr = blockIdx.x * 16 + (lane >> 2);
    const bool live = wr < P.nw;
    const int w = live ? wr : P.nw - 1;                // (lanes past the last water repeat it, unused)
    const int i = a < 3 ? 3 * w + a : P.nreal + w;
    const double wt = a == 0 ? 1.0 - P.gamma : 0.5 * P.gamma;
    double red[24];
#pragma unroll
    for (int t = 0; t < 24; ++t) red[t] = 0.0;
    // the water's sites
    double xs[4][3], qs[4], mus[4][3];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const int j = b < 3 ? 3 * w + b : P.nreal + w;
        xs[b][0] = x[j];
        xs[b][1] = y[j];
        xs[b][2] = z[j];
        qs[b] = chge[j];
#pragma unroll
        for (int q = 0; q < 3; ++q) mus[b][q] = dip[3 * j + q];
    }
    const double xi[3] = {x[i], y[i], z[i]}, qi = chge[i];
    const double mi[3] = {dip[3 * i], dip[3 * i + 1], dip[3 * i + 2]};
    const double p2 = site_polr2(P, i);
    // reciprocal space
    double f[3], vk = 0.0, vd = 0.0, e = 0.0, st[9];
    double kz[15];
#pragma unroll
    for (int t = 0; t < 15; ++t) kz[t] = ksum ? ksum[(long)t * P.n + i] : 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) f[q] = P.scale * kz[q] + f2[3 * i + q];
    vk = kz[3] * P.scale;
    vd = kz[4] * P.scale;
    const double er = -R4PIE0 * P.alpha * qi * qi / SQRPI + P.scal1 * kz[5];
#pragma unroll
    for (int t = 0; t < 9; ++t) st[t] = -(P.scal1 * kz[6 + t]);
    red[1] = qi * qi;
    // polarization
    if (p2 > 1.e-6) {
        double t = 0.0, m2 = 0.0;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const double own = efdd ? emu[3 * i + q] + efdd[3 * i + q] : emu[3 * i + q];
            t += mi[q] * (efk[3 * i + q] + efdc[3 * i + q] + 0.5 * own);
            m2 += mi[q] * mi[q];
        }
        red[0] = R4PIE0 * m2 / p2 / 2.0 - t;
    }
    e = er + e2[i] + red[0];
    // excluded pairs: F = force on this site from site b
    double vc = 0.0, W[9], FM[3] = {0.0, 0.0, 0.0};    // FM: force on M from this real site
#pragma unroll
    for (int t = 0; t < 9; ++t) W[t] = 0.0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        if (b == a) continue;
        const int j = b < 3 ? 3 * w + b : P.nreal + w;
        double d[3] = {xi[0] - xs[b][0], xi[1] - xs[b][1], xi[2] - xs[b][2]};
        image_vec(P.g, d[0], d[1], d[2]);
        const double rsq = norm2_nc(d[0], d[1], d[2]);
        const double rrr = sqrt(rsq);
        const double rri = 1.0 / rrr, rsqi = rri * rri;
        const double r3i = rri * rsqi, r5i = r3i * rsqi;
        double bbb[4];
        bfun_direct(P.alpha, rrr, rsqi, bbb);
        const double qj = qs[b], cicj = qi * qj;
        const double rdmui = mi[0] * d[0] + mi[1] * d[1] + mi[2] * d[2];
        const double rdmuj = mus[b][0] * d[0] + mus[b][1] * d[1] + mus[b][2] * d[2];
        double ffac = cicj * bbb[1] - (qj * rdmui - qi * rdmuj) * bbb[2];
        double dfi = bbb[1] * qj, dfj = -bbb[1] * qi;
        if (p2 > 1.e-6 && site_polr2(P, j) > 1.e-6) {
            const double dpidpj = mi[0] * mus[b][0] + mi[1] * mus[b][1] + mi[2] * mus[b][2];
            const double rr2 = rdmui * rdmuj;
            const double ath = (a == 0 || b == 0) ? P.athole12 : P.athole13;
            const double u = rrr * P.bbi[site_type(P, i)][site_type(P, j)];
            const double arob4 = ath * (u * u) * (u * u);
            const double dum1 = exp(-arob4);
            const double dum2 = (1.0 + (4.0 / 3.0) * arob4) * dum1;
            const double c3 = 3.0 * r5i * (1.0 - dum2) + bbb[2];
            const double dum34 = 4.0 * arob4 * dum1 * (rsqi * rsqi);
            ffac += dpidpj * (3.0 * r5i * (1.0 - dum1) + bbb[2] - rri * dum34) -
                    rr2 * (15.0 * (rsqi * r5i) * (1.0 - dum2) + bbb[3] - dum34 * (4.0 * arob4 - 1.0) * r3i);
            dfi += c3 * rdmuj;
            dfj += c3 * rdmui;
        }
        double F[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            F[q] = R4PIE0 * (ffac * d[q] + dfi * mi[q] + dfj * mus[b][q]);
            f[q] += F[q];
        }
        const double eh = 0.5 * cicj * bbb[0] * R4PIE0;
        e += eh;
        vc += R4PIE0 * (qj * bbb[0] + rdmuj * bbb[1]);
        red[2] += eh;
        red[4] += 0.5 * d[0] * F[0];
        red[5] += 0.5 * d[0] * F[1];
        red[6] += 0.5 * d[0] * F[2];
        red[7] += 0.5 * d[1] * F[1];
        red[8] += 0.5 * d[1] * F[2];
        red[9] += 0.5 * d[2] * F[2];
        if (b < 3) {
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int q = 0; q < 3; ++q) W[3 * p + q] += F[p] * (xi[q] - xs[b][q]);
        } else {
#pragma unroll
            for (int q = 0; q < 3; ++q) FM[q] = -F[q];
        }
    }
    red[3] = -(red[4] + red[7] + red[9]);
    // the M row's entries moved to O, H1, H2 (the M lane's own W is not used)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const double G[3] = {__shfl(FM[0], b, 4), __shfl(FM[1], b, 4), __shfl(FM[2], b, 4)};
        if (b == a) continue;
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int q = 0; q < 3; ++q) W[3 * p + q] += wt * G[p] * (xi[q] - xs[b][q]);
    }
    // ESP
    const double ve = vk + vr[i] + -2.0 * R4PIE0 * qi * P.alpha / SQRPI + vc + vd + vdcr[i];
    const double vt1 = __shfl(ve, 1, 4), vt2 = __shfl(ve, 2, 4), vt3 = __shfl(ve, 3, 4);
    // charge derivatives
    {
        const double* G = dg + 6 * w;   // dp1dr1, dp1dr2, dp2dr1, dp2dr2, dp1dcos, dp2dcos
        double r1v[3] = {xs[1][0] - xs[0][0], xs[1][1] - xs[0][1], xs[1][2] - xs[0][2]};
        double r2v[3] = {xs[2][0] - xs[0][0], xs[2][1] - xs[0][1], xs[2][2] - xs[0][2]};
        double r3v[3] = {xs[1][0] - xs[2][0], xs[1][1] - xs[2][1], xs[1][2] - xs[2][2]};
        image_vec(P.g, r1v[0], r1v[1], r1v[2]);
        image_vec(P.g, r2v[0], r2v[1], r2v[2]);
        image_vec(P.g, r3v[0], r3v[1], r3v[2]);
        const double r1 = sqrt(r1v[0] * r1v[0] + r1v[1] * r1v[1] + r1v[2] * r1v[2]);
        const double r2 = sqrt(r2v[0] * r2v[0] + r2v[1] * r2v[1] + r2v[2] * r2v[2]);
        const double rdot = r1v[0] * r2v[0] + r1v[1] * r2v[1] + r1v[2] * r2v[2];
        const double r1i = 1.0 / r1, r2i = 1.0 / r2;
        const double cost = rdot * (r1i * r2i);
        const double r3 = sqrt(r1 * r1 + r2 * r2 - 2.0 * r1 * r2 * cost);
        const double sint = sqrt(1.0 - cost * cost);
        const double cott = cost / sint, rdi = 1.0 / rdot;
        const double tmp = P.gamma / 2.0 / (1.0 - P.gamma);
        if (a < 3) {
            const int col = P.compat_qd ? P.nw + w : P.nreal + w;
            double xc[3] = {0.0, 0.0, 0.0};
            if (col < P.nreal) {
                xc[0] = x[col];
                xc[1] = y[col];
                xc[2] = z[col];
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                // derivatives of r1, r2 and theta by this site
                const double a1 = r1v[q] * r1i, a2 = r2v[q] * r2i;
                const double t1 = cott * (a1 * r1i - r2v[q] * rdi), t2 = cott * (a2 * r2i - r1v[q] * rdi);
                const double d1 = a == 0 ? -a1 : a == 1 ? a1 : 0.0;
                const double d2 = a == 0 ? -a2 : a == 2 ? a2 : 0.0;
                const double dt = a == 0 ? -t1 - t2 : a == 1 ? t1 : t2;
                const double dp1 = G[0] * d1 + G[1] * d2 - sint * G[4] * dt;
                const double dp2 = G[2] * d1 + G[3] * d2 - sint * G[5] * dt;
                const double dq1 = dp1 * (tmp + 1.0) + dp2 * tmp;
                const double dq2 = dp2 * (tmp + 1.0) + dp1 * tmp;
                const double F1 = -dq1 * vt1, F2 = -dq2 * vt2, F3 = (dq1 + dq2) * vt3;
                f[q] += F1 + F2 + F3;
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    if (a != 1) W[3 * q + r] += F1 * (xi[r] - xs[1][r]);
                    if (a != 2) W[3 * q + r] += F2 * (xi[r] - xs[2][r]);
                    if (col < P.nreal && col != i) W[3 * q + r] += F3 * (xi[r] - xc[r]);
                }
            }
        }
        // this site's charge in the virial and stress
        const double g0 = a == 1 ? G[0] + (G[0] + G[2]) * tmp : a == 2 ? G[2] + (G[0] + G[2]) * tmp
                        : a == 3 ? -(G[0] + G[2]) / (1.0 - P.gamma) : 0.0;
        const double g1 = a == 1 ? G[1] + (G[1] + G[3]) * tmp : a == 2 ? G[3] + (G[1] + G[3]) * tmp
                        : a == 3 ? -(G[1] + G[3]) / (1.0 - P.gamma) : 0.0;
        const double gc = a == 1 ? G[4] + (G[4] + G[5]) * tmp : a == 2 ? G[5] + (G[4] + G[5]) * tmp
                        : a == 3 ? -(G[4] + G[5]) / (1.0 - P.gamma) : 0.0;
        const double rr3i = 1.0 / sqrt(r3v[0] * r3v[0] + r3v[1] * r3v[1] + r3v[2] * r3v[2]);
        const double c12 = (r1 - r2 * cost) * r1i * r2i * r1i, c13 = (r2 - r1 * cost) * r1i * r2i * r2i;
        const double c23 = -r3 * r1i * r2i * rr3i;
        const int sa[6] = {0, 0, 0, 1, 1, 2}, sb[6] = {0, 1, 2, 1, 2, 2};
        double dc[6];
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            const double p1 = r1v[sa[t]] * r1v[sb[t]], p2r = r2v[sa[t]] * r2v[sb[t]], p3 = r3v[sa[t]] * r3v[sb[t]];
            dc[t] = c12 * p1 + c13 * p2r + c23 * p3;
            red[11 + t] = -ve * (g0 * r1i * p1 + g1 * r2i * p2r + gc * dc[t]);
            red[17 + t] = ve * gc * dc[t];
        }
        red[10] = ve * (r1 * g0 + r2 * g1 + gc * (dc[0] + dc[3] + dc[5]));
    }
    // outputs, the M site's share moved onto the real atoms
    double fm[3], sm[9];
#pragma unroll
    for (int q = 0; q < 3; ++q) fm[q] = __shfl(f[q], 3, 4);
#pragma unroll
    for (int t = 0; t < 9; ++t) sm[t] = __shfl(st[t], 3, 4);
    const double em = __shfl(e, 3, 4);
    if (live) {
        e1[i] = er;
        vesp[i] = ve;
        if (a < 3) {
            const int m = P.nreal + w;
            eout[i] = e + wt * em;
#pragma unroll
            for (int q = 0; q < 3; ++q) fout[3 * i + q] = distribute ? f[q] + wt * fm[q] : f[q];
#pragma unroll
            for (int t = 0; t < 9; ++t) sout[9 * i + t] = st[t] + wt * sm[t];
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    wout[9 * i + 3 * p + q] = w2[9 * i + 3 * p + q] + W[3 * p + q] +
                                              wt * (fmsum[3 * m + p] * xi[q] - fmx[9 * m + 3 * p + q]);
        } else {
#pragma unroll
            for (int q = 0; q < 3; ++q) fout[3 * i + q] = distribute ? 0.0 : f[q];
        }
    } else {
#pragma unroll
        for (int t = 0; t < 24; ++t) red[t] = 0.0;
    }
    int k;
    const double t = wave_sum24(red, lane, k);
    if (k < 24 && (lane & 1) == 0) blk[24L * blockIdx.x + k] = t;
}

// Fixed-order sums of block partials: set b has nb[b] blocks of stride[b] values, of which
// nv[b] are summed into out[off[b] ..].  One block of 256 threads per (set, value), listed
// in sv[]: thread t adds blocks t, t + 256, ..., then the wavefront sums and the four wave
// sums are added in order.
struct SumSets {
    const double* blk[7];
    int nb[7], stride[7], nv[7], off[7];
    int nsv;
    unsigned char sv[64][2];   // (set, value) of each block
};
__global__ __launch_bounds__(256) void k_el_sum_sets(SumSets S, double* __restrict__ out)
{
    __shared__ double ws[4];
    const int b = S.sv[blockIdx.x][0], q = S.sv[blockIdx.x][1];
    double s = 0.0;
    for (int k = threadIdx.x; k < S.nb[b]; k += 256) s += S.blk[b][(long)k * S.stride[b] + q];
    s = wsum(s);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[S.off[b] + q] = ((ws[0] + ws[1]) + ws[2]) + ws[3];
}

// Zero a double array (graph-safe replacement for a memset node).
__global__ void k_el_zero(double* __restrict__ p, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// ============================================================ host launchers ======

namespace {
inline int ceil_div(long a, long b) { return (int)((a + b - 1) / b); }
// dynamic LDS of the reciprocal-space passes (bytes)
inline size_t rs_lds(int spc) { return sizeof(double) * std::max(512L * RS_WAVES, 4L * spc); }

// The real-space field of dip: four wavefronts to a row where rows are long (a cluster's hold
// every other polarizable site; 300 waters 8.7 -> 7.3 us, 701 waters 28.7 -> 23.4), one where a
// block per row costs more than it shortens (2048-water box, 305 partners: 15.2 against 22.6).
void launch_emu(const ElecBuffers& E, const ElecDev& P, const double* dip, double* state, const double* cgblk, int cgnb,
                int it, hipStream_t s)
{
    if (P.capP >= 512 && P.g.imcon == 0)
        hipLaunchKernelGGL(k_el_emu<4>, dim3(P.nrow), dim3(256), 0, s, P, E.x, E.y, E.z, E.nbrP, E.cntP, E.tens, E.tin,
                           dip, E.emu, state, cgblk, cgnb, it);
    else
        hipLaunchKernelGGL(k_el_emu<1>, dim3(ceil_div(P.nrow, 4)), dim3(256), 0, s, P, E.x, E.y, E.z, E.nbrP, E.cntP,
                           E.tens, E.tin, dip, E.emu, state, cgblk, cgnb, it);
}

// Structure factors of nset sets of weights over nch chunks of spc sites; with emu also the
// real-space field of set 0 (dipoles).  Tiles of n per block: as many as the list needs, up to 4
// (more are spread over blocks; each costs 16 accumulator registers).
template <int NT>
void rs_launch_sfac_t(const ElecBuffers& E, const ElecDev& P, const RsSrcs& src, int nset, int nch, int spc, bool emu,
                      double* state, const double* cgblk, int cgnb, int it, hipStream_t s)
{
    const int nsb = P.rs.ng * ceil_div(P.rs.ntiles, NT) * nch * nset;
    hipLaunchKernelGGL(k_rs_sfac<NT>, dim3(nsb + (emu ? ceil_div(P.nrow, RS_WAVES) : 0)), dim3(64 * RS_WAVES), rs_lds(spc),
                       s, P, src, nsb, nch, spc, E.pht, E.Spart, E.x, E.y, E.z, E.nbrP, E.cntP, E.tens, E.tin, E.emu, state, cgblk,
                       cgnb, it);
}
void rs_launch_sfac(const ElecBuffers& E, const ElecDev& P, const RsSrcs& src, int nset, int nch, int spc, bool emu,
                    double* state, const double* cgblk, int cgnb, int it, hipStream_t s)
{
    auto f = P.rs.ntiles == 1   ? rs_launch_sfac_t<1>
             : P.rs.ntiles == 2 ? rs_launch_sfac_t<2>
             : P.rs.ntiles == 3 ? rs_launch_sfac_t<3>
                                : rs_launch_sfac_t<4>;
    f(E, P, src, nset, nch, spc, emu, state, cgblk, cgnb, it, s);
}
// The fields of nset sets of structure factors summed over nch chunks: 16-site tiles per
// wavefront so that there are about two blocks per CU (each block first adds its group's chunks).
void rs_launch_field(const ElecBuffers& E, const ElecDev& P, int nset, int nch, hipStream_t s)
{
    const int tiles = ceil_div(P.nrow, 16 * RS_WAVES);
    const int tpw = std::max(1L, std::min((long)tiles, (long)tiles * P.rs.ng / 448));
    const int nsb = ceil_div(tiles, tpw);
    auto k = P.rs.ntiles > RS_NT ? k_rs_field<true> : k_rs_field<false>;
    hipLaunchKernelGGL(k, dim3(nsb * P.rs.ng * nset), dim3(64 * RS_WAVES), 0, s, P, nch, tpw, nsb, E.pht, E.Spart,
                       E.Fpart, E.state);
}
}

// The sites and charges (and with cg the preconditioner), the neighbour rows (and with ksum the
// phase tables).
int el_launch_setup(ElecBuffers& E, const ElecDev& P, CellList& cells, bool cg, bool ksum, hipStream_t s)
{
    const int nwb = ceil_div(P.nw, 64), nph = ksum ? ceil_div(P.n + RS_PAD, 64) : 0;
    hipLaunchKernelGGL(k_el_waters, dim3(cg ? 2 * nwb : nwb), dim3(64), 0, s, P, nwb, E.x, E.y, E.z, E.chge, E.dg,
                       E.dip, E.cg_minv);
    if (P.cells.on) {
        const int rc = cells_build(cells, P.n, E.x, E.y, E.z, 1, s);
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_el_nbr, dim3(nph + P.n), dim3(64), 0, s, P, nph, E.x, E.y, E.z, E.nbrA, E.cntA, E.nbrP, E.cntP,
                       E.err, E.phc, E.phs, E.pht);
    return (int)hipGetLastError();
}

// after the neighbour counts were checked by the host
// The reciprocal field of the dipoles mu at the first n sites (particle mesh) into
// Fpart[c * P.n + j] as a k-sum partial (times kap), for the chunk-sum readers with one chunk
// (scale_state > 0: mu spread times the power of two in state[scale_state], see SpSpec)
static void el_spme_dipole_field(ElecBuffers& E, const ElecSpme& sp, int n, const double* mu, const double* state,
                                 hipStream_t s, int scale_state = 0)
{
    SpSpec spec{};
    spec.ngr = 1;
    spec.mu_on[0] = 1;
    spec.comp[0] = -1;
    spec.scale_state = scale_state;
    double2* g = sp.B->grid;
    sp_launch_spread(*sp.B, *sp.G, n, nullptr, mu, spec, g, true, state, s);
    sp_launch_convolve(*sp.B, *sp.G, g, 1, true, state, s);
    sp_launch_field(*sp.B, *sp.G, n, g, 1, sp.kap, E.Fpart, E.n, state, s, scale_state);
}

static inline ElecDev one_chunk(const ElecDev& P)
{
    ElecDev Q = P;
    Q.fchunks = 1;
    Q.K = 0;
    return Q;
}

// The charge fields and dipole tensors of every row, then the reciprocal fields of the start
// dipoles and of the charges as partials (Fpart); the real-space field of the start dipoles; for
// SOR also the sums of the partials (the conjugate-gradient start forms its own).
int el_launch_prep(ElecBuffers& E, const ElecDev& P, bool cg, const ElecSpme* sp, hipStream_t s)
{
    hipLaunchKernelGGL(k_el_prep, dim3(P.n), dim3(64), 0, s, P, E.x, E.y, E.z, E.chge, E.tab, E.nbrA, E.cntA, E.tens,
                       E.tin, E.efk);
    if (sp && !sp->B) {
        // no reciprocal space (an isolated cluster): zero fields, in the layout of the k-sum
        // field partials (one chunk), so that the reductions form efdd (the self term is 0
        // without an Ewald split) and efdc
        el_launch_zero(E.Fpart, 6L * P.n, s);
    } else if (sp) {
        // particle mesh: splines of every site, then the fields of the start dipoles (grid 0)
        // and of the charges (grid 1) at every site, in the layout of the k-sum field partials
        sp_launch_prep(*sp->B, *sp->G, P.n, E.x, E.y, E.z, s);
        SpSpec spec{};
        spec.ngr = 2;
        spec.mu_on[0] = 1;
        spec.comp[0] = -1;
        spec.q_on[1] = 1;
        spec.comp[1] = -1;
        double2* g = sp->B->grid;
        sp_launch_spread(*sp->B, *sp->G, P.n, E.chge, E.dip, spec, g, true, nullptr, s);
        sp_launch_convolve(*sp->B, *sp->G, g, 2, true, nullptr, s);
        sp_launch_field(*sp->B, *sp->G, P.n, g, 2, sp->kap, E.Fpart, P.n, nullptr, s);
    } else {
        // structure factors of the start dipoles and of the charges, and the iloop = 1 fields
        rs_launch_sfac(E, P, {{{E.dip, 3, 1, P.n, 1}, {E.chge, 1, 0, P.n, 0}}}, 2, P.rs.nchq, P.rs.spcq, true, E.state, nullptr,
                       0, 0, s);
        rs_launch_field(E, P, 2, P.rs.nchq, s);
    }
    if (sp) launch_emu(E, P, E.dip, E.state, nullptr, 0, 0, s);
    if (!cg)
        hipLaunchKernelGGL(k_el_kfield_reduce<true>, dim3(ceil_div(6L * P.nrow, 64)), dim3(256), 0, s,
                           sp ? one_chunk(P) : P, E.Fpart, E.dip, E.efdd, E.efdc, E.state);
    return (int)hipGetLastError();
}

int el_launch_iteration(ElecBuffers& E, const ElecDev& P, int first, const ElecSpme* sp, hipStream_t s)
{
    if (!first && sp && !sp->B) {
        // no reciprocal space: efdd keeps the preparation's zeros
    } else if (!first && sp) {
        el_spme_dipole_field(E, *sp, P.nrow, E.dip, E.state, s);
        hipLaunchKernelGGL(k_el_kfield_reduce<false>, dim3(ceil_div(3L * P.nrow, 64)), dim3(256), 0, s, one_chunk(P),
                           E.Fpart, E.dip, E.efdd, E.efdc, E.state);
    } else if (!first) {
        // reciprocal dipole field from the current dipoles (the first iteration's came
        // with the charge field)
        rs_launch_sfac(E, P, {{{E.dip, 3, 1, P.nrow, 1}}}, 1, P.rs.nch, P.rs.spc, true, E.state, nullptr, 0, 0, s);
        rs_launch_field(E, P, 1, P.rs.nch, s);
        hipLaunchKernelGGL(k_el_kfield_reduce<false>, dim3(ceil_div(3L * P.nrow, 64)), dim3(256), 0, s, P, E.Fpart, E.dip,
                           E.efdd, E.efdc, E.state);
    }
    // (the first iteration's came with the preparation)
    if (!first && sp) launch_emu(E, P, E.dip, E.state, nullptr, 0, 0, s);
    const int nb = ceil_div(P.nrow, 256);
    hipLaunchKernelGGL(k_el_sor, dim3(nb), dim3(256), 0, s, P, E.efk, E.emu, E.efdd, E.efdc, E.dip, E.blk, E.state);
    hipLaunchKernelGGL(k_el_converge, dim3(1), dim3(64), 0, s, P, nb, E.blk, E.state);
    return (int)hipGetLastError();
}

// The dipole-field operator applied to the solver's m (emu: real-space rows; Fpart: the
// reciprocal field's partials), for the k-sum: structure factors (taking the stopping test
// of iteration `it` first when `check`) and emu in one launch, then the field.
static void el_cg_apply_ksum(ElecBuffers& E, const ElecDev& P, bool check, int it, hipStream_t s)
{
    rs_launch_sfac(E, P, {{{E.cg_m, 3, 1, P.nrow, 1}}}, 1, P.rs.nch, P.rs.spc, true, E.state, check ? E.cgblk : nullptr,
                   ceil_div(P.nw, CG_WPB), it, s);
    rs_launch_field(E, P, 1, P.rs.nch, s);
}

// The same for the particle mesh (emu first, with the stopping test when `check`) and for no
// reciprocal space (emu alone; the preparation's zero field partials stand)
static void el_cg_apply_other(ElecBuffers& E, const ElecDev& P, const ElecSpme& sp, bool check, int it, hipStream_t s)
{
    const int nbw = ceil_div(P.nw, CG_WPB);
    launch_emu(E, P, E.cg_m, E.state, check ? E.cgblk : nullptr, nbw, it, s);
    if (sp.B) el_spme_dipole_field(E, sp, P.nrow, E.cg_m, E.state, s, 9);
}

static void el_cg_update(ElecBuffers& E, const ElecDev& P, const ElecSpme* sp, bool init, hipStream_t s)
{
    const int nbw = ceil_div(P.nw, CG_WPB);
    const ElecDev Q = sp ? one_chunk(P) : P;
    if (init)
        hipLaunchKernelGGL(k_cg_update<true>, dim3(nbw), dim3(256), 0, s, Q, E.Fpart, E.emu, E.cg_minv, E.cg_m, E.dip,
                           E.cg_r, E.cg_u, E.cg_w, E.cg_z, E.cg_q, E.cg_s, E.cg_p, E.cg_tmu, E.cgblk, E.state);
    else
        hipLaunchKernelGGL(k_cg_update<false>, dim3(nbw), dim3(256), 0, s, Q, E.Fpart, E.emu, E.cg_minv, E.cg_m, E.dip,
                           E.cg_r, E.cg_u, E.cg_w, E.cg_z, E.cg_q, E.cg_s, E.cg_p, E.cg_tmu, E.cgblk, E.state);
}

// The one-launch solve takes what its block holds: evaluations of 5 to 21 waters take 230 to 240 us
// with it and 265 to 273 us with launches per iteration, which larger systems need for their width.
static inline bool one_launch_solve(const ElecDev& P, const ElecSpme* sp)
{
    return sp && !sp->B && P.nw <= CG_SOLVE_WATERS;
}

static void el_cg_solve(ElecBuffers& E, const ElecDev& P, bool init, int it0, int count, hipStream_t s)
{
    hipLaunchKernelGGL(k_cg_solve, dim3(1), dim3(1024), 0, s, P, init, it0, count, E.x, E.y, E.z, E.nbrP, E.cntP, E.tens,
                       E.tin, E.cg_minv, E.cg_m, E.dip, E.cg_r, E.cg_u, E.cg_w, E.cg_z, E.cg_q, E.cg_s, E.cg_p, E.cg_tmu,
                       E.cgblk, E.state);
}

// Iteration `it` (0-based): the stopping test and scalars from the last update's partials,
// n = A m (real-space rows, structure factors, reciprocal field), then the vector update.
int el_launch_cg_iteration(ElecBuffers& E, const ElecDev& P, int it, const ElecSpme* sp, hipStream_t s)
{
    if (one_launch_solve(P, sp)) {
        el_cg_solve(E, P, false, it, 1, s);
        return (int)hipGetLastError();
    }
    if (sp) el_cg_apply_other(E, P, *sp, true, it, s);
    else el_cg_apply_ksum(E, P, true, it, s);
    el_cg_update(E, P, sp, false, s);
    return (int)hipGetLastError();
}

// conjugate-gradient start: residual of the start dipoles (their fields came with the
// charge fields of the preparation), u = M^-1 r, and
// the first application of A, to u, for w = A u
int el_launch_cg_start(ElecBuffers& E, const ElecDev& P, int iters, const ElecSpme* sp, hipStream_t s)
{
    hipLaunchKernelGGL(k_cg_init, dim3(ceil_div(P.nw, CG_WPB)), dim3(256), 0, s, sp ? one_chunk(P) : P, E.Fpart, E.efk,
                       E.efdc, E.emu, E.efdd, E.dip, E.cg_minv, E.cg_r, E.cg_u, E.cg_m, E.cg_z, E.cg_q, E.cg_s, E.cg_p,
                       E.cg_tmu);
    if (one_launch_solve(P, sp)) {
        el_cg_solve(E, P, true, 0, iters, s);
        return (int)hipGetLastError();
    }
    if (!sp) el_cg_apply_ksum(E, P, false, 0, s);
    else el_cg_apply_other(E, P, *sp, false, 0, s);
    el_cg_update(E, P, sp, true, s);
    for (int it = 0; it < iters; ++it) {
        const int rc = el_launch_cg_iteration(E, P, it, sp, s);
        if (rc) return rc;
    }
    return (int)hipGetLastError();
}

// `reps` launches of the dipole structure-factor pass over the current dipoles, bracketed
// by events on the stream (timing only: the partials it writes are rewritten by every
// evaluation before use)
int el_time_sfac(ElecBuffers& E, const ElecDev& P, int reps, hipEvent_t a, hipEvent_t b, hipStream_t s)
{
    (void)hipEventRecord(a, s);
    for (int r = 0; r < reps; ++r)
        rs_launch_sfac(E, P, {{{E.dip, 3, 1, P.nrow, 1}}}, 1, P.rs.nch, P.rs.spc, false, E.zero_state, nullptr, 0, 0, s);
    (void)hipEventRecord(b, s);
    return (int)hipGetLastError();
}

int el_launch_final(ElecBuffers& E, const ElecDev& P, int distribute, double g34, double gln34, int refresh,
                    const ElecSpme* sp, hipStream_t s)
{
    // k-sum: one partial per 64 k; particle mesh: one per 4 sites (k_sp_elec_final's blocks)
    const int nwb = ceil_div(P.nw, 16), nkb = !sp ? ceil_div(P.K, 64) : sp->B ? ceil_div(P.n, 4) : 0;
    double* b_ks = E.blk;                        // [nkb][8]
    double* b_p2 = b_ks + 8L * nkb;              // [n][8]
    double* b_w = b_p2 + 8L * P.n;               // [nwb][24]
    if (sp && sp->B) {
        // particle mesh: grids 0..4 hold q + mu, q, and mu_x, mu_y, mu_z as charges; the
        // stress kernels of grid 0 go to grids 5..10; every per-site quantity of the k-sum
        // site pass then comes from one gather (k_sp_elec_final), in the k-sum pass's units
        SpSpec spec{};
        spec.ngr = 5;
        spec.q_on[0] = 1;
        spec.mu_on[0] = 1;
        spec.q_on[1] = 1;
        spec.comp[0] = spec.comp[1] = -1;
        for (int b = 0; b < 3; ++b) spec.comp[2 + b] = (signed char)b;
        SpmeBuffers& B = *sp->B;
        const SpmeGeom& G = *sp->G;
        double2* g = B.grid;
        sp_launch_spread(B, G, P.n, E.chge, E.dip, spec, g, true, nullptr, s);
        sp_launch_fft(B, G, g, 5, false, nullptr, s, true);
        sp_launch_influence_stress(B, G, g, g + 5 * B.ng_cap, s);
        sp_launch_influence(B, G, g + B.ng_cap, 4, false, nullptr, s);
        sp_launch_fft(B, G, g, 11, true, nullptr, s, false);
        sp_launch_elec_final(B, G, P.n, E.chge, E.dip, g, sp->kap, E.ksum, b_ks, s);
    }
    if (!sp) {
        // structure factors of mu_x, mu_y, mu_z of the converged dipoles and of the charges
        rs_launch_sfac(E, P,
                       {{{E.dip, 3, 0, P.nrow, 1}, {E.dip + 1, 3, 0, P.nrow, 1}, {E.dip + 2, 3, 0, P.nrow, 1},
                         {E.chge, 1, 0, P.n, 0}}}, 4, P.rs.nchq, P.rs.spcq, false, E.zero_state, nullptr, 0, 0, s);
        hipLaunchKernelGGL(k_el_kscal, dim3(nkb), dim3(256), 0, s, P, E.kv, E.Spart, E.kf, b_ks);
        hipLaunchKernelGGL(k_el_kfinal, dim3(ceil_div(P.n, 256), P.kchunks), dim3(256),
                           sizeof(double2) * 6 * EL_RUN * P.rpc, s, P, (const int4*)E.runs, E.runk, E.phc, E.phs, E.kv, E.kf, E.chge, E.dip, E.Fpart);
        hipLaunchKernelGGL(k_el_ksum, dim3(ceil_div(15L * P.n, 64)), dim3(256), 0, s, P, E.Fpart, E.ksum);
    }
    hipLaunchKernelGGL(k_el_pairs, dim3(P.n), dim3(64), 0, s, P, E.x, E.y, E.z, E.chge, E.dip, E.tab, E.nbrA, E.cntA,
                       g34, gln34, E.f2, E.e2, E.vr, E.vdcr, E.w2, E.fmsum, E.fmx, b_p2);
    // the dipoles' own field: carried along by the conjugate-gradient solver as T mu; the SOR path
    // keeps that of its last iteration, as the reference does
    hipLaunchKernelGGL(k_el_water_final, dim3(nwb), dim3(64), 0, s, P, distribute, E.x, E.y, E.z, E.chge, E.dip, E.dg,
                       sp && !sp->B ? nullptr : E.ksum, E.efk, E.efdc, refresh ? E.cg_tmu : E.emu,
                       refresh ? nullptr : E.efdd, E.f2, E.e2, E.vr, E.vdcr, E.w2, E.fmsum, E.fmx, E.e1, E.vesp, E.fsite,
                       E.eout, E.sout, E.wout, b_w);
    // scalars: [0] eng_polar, [1..8] k sums (engc, engdum, omg6), [9] sum q^2, [11..18] pairs
    // (energy, virial, stress6), [19..26] excluded pairs, [28..34] qd (virial, stress6),
    // [35..40] angular per-atom qd stresses
    SumSets ss{};
    const double* sb[7] = {b_ks, b_p2, b_w, b_w + 1, b_w + 2, b_w + 10, b_w + 17};
    const int snb[7] = {nkb, P.n, nwb, nwb, nwb, nwb, nwb}, sst[7] = {8, 8, 24, 24, 24, 24, 24};
    const int snv[7] = {8, 8, 1, 1, 8, 7, 6}, soff[7] = {1, 11, 0, 9, 19, 28, 35};
    ss.nsv = 0;
    for (int q = 0; q < 7; ++q) {
        ss.blk[q] = sb[q];
        ss.nb[q] = snb[q];
        ss.stride[q] = sst[q];
        ss.nv[q] = snv[q];
        ss.off[q] = soff[q];
        for (int v = 0; v < snv[q]; ++v) {
            ss.sv[ss.nsv][0] = (unsigned char)q;
            ss.sv[ss.nsv][1] = (unsigned char)v;
            ++ss.nsv;
        }
    }
    hipLaunchKernelGGL(k_el_sum_sets, dim3(ss.nsv), dim3(256), 0, s, ss, E.scal);
    return (int)hipGetLastError();
}

void el_launch_zero(double* p, long n, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_el_zero, dim3(ceil_div(n, 256)), dim3(256), 0, s, p, n);
}

__global__ void k_el_add(double* __restrict__ dst, const double* __restrict__ src, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] += src[i];
}

// dst[i] += src[i], i < n
void el_launch_add(double* dst, const double* src, long n, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_el_add, dim3(ceil_div(n, 256)), dim3(256), 0, s, dst, src, n);
}

__global__ void k_el_copy(double* __restrict__ dst, const double* __restrict__ src, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

__global__ void k_el_pack(const double* __restrict__ state, const int* __restrict__ err,
                          const double* __restrict__ scal, const int* __restrict__ spflag, double* __restrict__ out)
{
    const int t = threadIdx.x;
    if (t >= EL_PK_N) return;
    double v;
    if (t < EL_PK_ERR) v = state[t - EL_PK_ST];
    else if (t < EL_PK_SCAL) v = (double)err[0];
    else if (t < EL_PK_SPF) v = scal[t - EL_PK_SCAL];
    else v = spflag ? (double)spflag[t - EL_PK_SPF] : 0.0;
    out[t] = v;
}

void el_launch_pack(const double* state, const int* err, const double* scal, const int* spflag, double* out,
                    hipStream_t s)
{
    hipLaunchKernelGGL(k_el_pack, dim3(1), dim3(64), 0, s, state, err, scal, spflag, out);
}

// Up to EL_NSEG copies dst_k[i] = src_k[i], i < n_k (a null source clears dst_k) in one
// launch, segment k in blockIdx.y: the small copies around an evaluation as one graph node.
struct ElCopySegs {
    double* dst[EL_NSEG];
    const double* src[EL_NSEG];
    long n[EL_NSEG];
};

__global__ void k_el_copy_segs(ElCopySegs S)
{
    const int k = blockIdx.y;
    double* __restrict__ d = S.dst[k];
    const double* __restrict__ src = S.src[k];
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < S.n[k]; i += (long)gridDim.x * blockDim.x)
        d[i] = src ? src[i] : 0.0;
}

void el_launch_copy_segs(int nseg, double* const* dst, const double* const* src, const long* n, hipStream_t s)
{
    ElCopySegs S{};
    long nmax = 0;
    for (int k = 0; k < nseg; ++k) {
        S.dst[k] = dst[k];
        S.src[k] = src[k];
        S.n[k] = n[k];
        nmax = n[k] > nmax ? n[k] : nmax;
    }
    if (nseg <= 0 || nmax <= 0) return;
    const long blocks = ceil_div(nmax, 256) < 1024 ? ceil_div(nmax, 256) : 1024;
    hipLaunchKernelGGL(k_el_copy_segs, dim3(blocks, nseg), dim3(256), 0, s, S);
}

// dst[i] = src[i], i < n (a kernel rather than a copy call, so that a captured graph holds
// only kernel nodes)
void el_launch_copy(double* dst, const double* src, long n, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_el_copy, dim3(ceil_div(n, 256)), dim3(256), 0, s, dst, src, n);
}
