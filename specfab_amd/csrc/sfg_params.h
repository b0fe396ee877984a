// Per-parcel operator parameters from the kinematics: the 23 operator weights
// theta, the 15 weights omega of Gamma0 <D> and the diagonal s_l (REG + CDRX).
#pragma once
#include "generated/sfg_moment_maps.h"
#include "sfg_device.h"
#include "sfg_kernels.h"

namespace sfg {

struct ParcelParams {
    double D[9], W[9], tau[9];
    double g0, lam, rate;    // DDRX and CDRX rates; reg_nu |D|
    double tv[6], sv[6], c;  // Mandel vectors of tau and tau.tau, 5 Gamma0 / (tau:tau)
};

__device__ inline void parcel_kinematics(const ParamArgs& a, int64_t p, ParcelParams& q) {
    double G[9];
    for (int i = 0; i < 9; i++) G[i] = a.ugrad[p * 9 + i];
    sym_skew(G, q.D, q.W);
    for (int i = 0; i < 9; i++) q.tau[i] = a.tau ? a.tau[p * 9 + i] : q.D[i];
    q.g0 = (a.procs & 2) && a.gam0 ? a.gam0[p] : 0.0;
    q.lam = ((a.procs & 4) && a.lam) ? a.lam[p] : 0.0;
    q.rate = 0.0;
    if (a.procs & 8) {
        double fro = 0;
        for (int i = 0; i < 9; i++) fro += q.D[i] * q.D[i];
        q.rate = a.reg_nu * sqrt(fro);
    }
    if (a.procs & 2) {
        const double s2 = sqrt(2.0);
        const double* tau = q.tau;
        double tsq[9];
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++) {
                double s = 0;
                for (int k = 0; k < 3; k++) s += tau[3 * i + k] * tau[3 * k + j];
                tsq[3 * i + j] = s;
            }
        const double norm = tsq[0] + tsq[4] + tsq[8];
        const double tv[6] = {tau[0], tau[4], tau[8], s2 * tau[5], s2 * tau[2], s2 * tau[1]};
        const double sv[6] = {tsq[0], tsq[4], tsq[8], s2 * tsq[5], s2 * tsq[2], s2 * tsq[1]};
        for (int i = 0; i < 6; i++) q.tv[i] = tv[i], q.sv[i] = sv[i];
        q.c = q.g0 * 5.0 / norm;
    }
}

__device__ inline void parcel_theta(const ParamArgs& a, const ParcelParams& q, double* th) {
    for (int i = 0; i < NPAR_K; i++) th[i] = 0.0;
    if (a.procs & 1) {
        cplx qe[5], qo[3];
        d_lrot_weights(q.D, q.W, a.iota, a.zeta, nullptr, nullptr, nullptr, nullptr, qe, qo);
        th[0] = qe[2].re; th[1] = qe[3].re; th[2] = qe[3].im; th[3] = qe[4].re; th[4] = qe[4].im;
        th[5] = qo[1].re; th[6] = qo[2].re; th[7] = qo[2].im;
    }
    if (a.procs & 2) {
        cplx g[15];
        d_ddrx_weights(q.tau, g);
        // theta = Gamma0 * (Re/Im g(l, m >= 0)), k index of (l,m): l=0 -> 0, l=2 -> 3+m, l=4 -> 10+m
        th[8] = q.g0 * g[0].re;
        th[9] = q.g0 * g[3].re;
        th[10] = q.g0 * g[4].re; th[11] = q.g0 * g[4].im;
        th[12] = q.g0 * g[5].re; th[13] = q.g0 * g[5].im;
        th[14] = q.g0 * g[10].re;
        for (int m = 1; m <= 4; m++) {
            th[13 + 2 * m] = q.g0 * g[10 + m].re;
            th[14 + 2 * m] = q.g0 * g[10 + m].im;
        }
    }
}

// <D> = 5 [ (tau.tau):a2 - tau:a4:tau ] / (tau:tau), src/dynamics.f90:402-422,
// with a2v = A2 x / x0 + I/3, a4v = A4 x / x0  =>  Gamma0 <D> = (omega . x) / x0
__device__ inline double parcel_omega(const ParamArgs& a, const ParcelParams& q, int i0) {
    double d1 = 0, d2 = 0;
    for (int i = 0; i < 6; i++) {
        d1 += q.sv[i] * a.A2[i * 15 + i0];
        double r = 0;
        for (int j = 0; j < 6; j++) r += a.A4[(6 * i + j) * 15 + i0] * q.tv[j];
        d2 += q.tv[i] * r;
    }
    const double om = q.c * (d1 - d2);
    return i0 == 0 ? om + q.c * ((q.sv[0] + q.sv[1] + q.sv[2]) / 3.0) : om;
}

// The same for a constant i0: the column i0 of the maps folds to literals and its
// zeros (five in six) drop out, so that nothing is loaded.
template <int I0>
__device__ __forceinline__ double parcel_omega_const(const ParcelParams& q) {
    double e[15] = {}, a2[6], a4[6][6];
    e[I0] = 1.0;
    moment_maps(e, a2, a4);
    double d1 = 0, d2 = 0;
#pragma unroll
    for (int i = 0; i < 6; i++) {
        if (a2[i] != 0.0) d1 += q.sv[i] * a2[i];
        double r = 0;
#pragma unroll
        for (int j = 0; j < 6; j++)
            if (a4[i][j] != 0.0) r += a4[i][j] * q.tv[j];
        d2 += q.tv[i] * r;
    }
    const double om = q.c * (d1 - d2);
    return I0 == 0 ? om + q.c * ((q.sv[0] + q.sv[1] + q.sv[2]) / 3.0) : om;
}

__device__ inline double parcel_sl(const ParamArgs& a, const ParcelParams& q, int b) {
    const int l = 2 * b;
    double v = -q.rate * a.reg_shape[b];
    if (a.procs & 4) v += q.lam * (-(double)(l * (l + 1)));
    return v;
}

}  // namespace sfg
