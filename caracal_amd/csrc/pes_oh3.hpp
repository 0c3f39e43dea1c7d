// OH + H2 surface of Schatz and Elgersma (Chem. Phys. Lett. 73, 21 (1980)) in
// the POTLIB form the reference evaluates (egrad_oh3, src/egrad_oh3.f:33-190;
// pot_oh3 and its three-body, four-body and H2O routines, :249-598; the
// constants of BLOCK DATA PTPACM_oh3, :620-633, all written with a D
// exponent).  One lane per bead, FP64.
//
// Atoms O, H1 (hydroxyl), H2, H3; distances R1 = O-H1, R2 = O-H2, R3 = O-H3,
// R4 = H1-H2, R5 = H1-H3, R6 = H2-H3.  V = three Morse pairs + LEPS over
// (R2, R3, R6) + H2O terms over (R1, R2, R4) and (R1, R3, R5) + a four-body
// Gaussian over (R2, R3, R4, R5) - 2 DE2 + DE3.
//
// The reference's routines share one derivative array: where an H2O switching
// factor is exactly zero (0.5 gamma s >= 43, an O-H distance beyond 37.6 bohr)
// the H2O routine leaves that entry unset and the previous routine's value
// stands in its place (src/egrad_oh3.f:590-594).  `shared` below carries that
// array so the device gives the reference's forces there too.
#pragma once
#include "quad.hpp"

namespace cam {
namespace oh3 {

constexpr double kDe[3] = {0.148201, 0.0275690, 0.151548};
constexpr double kBeta[3] = {1.260580, 0.924180, 1.068620};
constexpr double kRe[3] = {1.863300, 2.907700, 1.428600};
constexpr double kSato = 0.10;
constexpr double kGam[3] = {2.399700, 1.058350, 2.399700};
constexpr double kReOH = 1.808090, kReHH = 2.861590;
constexpr double kCon[7] = {-.0015920, 0.026963, 0.0014689, 0.080011, 0.085816, -0.063179, 0.101380};
constexpr double kAlp[4] = {4.773, 7.14, 2.938, 5.28};
constexpr double kLam[4] = {0.10, 0.10, 0.20, 0.03};
constexpr double kAcon[2] = {0.10, 0.009};

// LEPS over (r0, r1, r2): pair 1's Morse constants for the two O-H
// distances, pair 3's for H-H.
__device__ inline double leps(double r0, double r1, double r2, double *dedr)
{
    const double rr[3] = {r0, r1, r2};
    double x[3], exch[3], b[3], energy = 0.0;
    constexpr double z = kSato, zpo = 1.0 + z, op3z = 1.0 + 3.0 * z, top3z = 2.0 * op3z, zp3 = z + 3.0,
                     tzp3 = 2.0 * zp3;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int k = i == 2 ? 2 : 0;
        const double do4z = kDe[k] / 4.0 / zpo;
        b[i] = kBeta[k] * do4z * 2.0;
        x[i] = exp(-kBeta[k] * (rr[i] - kRe[k]));
        const double coul = do4z * (zp3 * x[i] - top3z) * x[i];
        exch[i] = do4z * (op3z * x[i] - tzp3) * x[i];
        energy = energy + coul;
    }
    const double d12 = exch[0] - exch[1], d23 = exch[1] - exch[2], d31 = exch[2] - exch[0];
    const double rad = sqrt(d12 * d12 + d23 * d23 + d31 * d31);
    const double s2 = sqrt(2.0);
    energy = energy - rad / s2;
    const double s = exch[0] + exch[1] + exch[2];
#pragma unroll
    for (int i = 0; i < 3; ++i)
        dedr[i] = b[i] * x[i] * ((3.0 * exch[i] - s) / s2 * (op3z * x[i] - zp3) / rad - zp3 * x[i] + op3z);
    return energy;
}

// H2O term over (r_OH, r_OH', r_HH'); dedr holds the shared array on entry.
__device__ inline double h2o(double r0, double r1, double r2, double *dedr)
{
    double s[3], q[3], dq[3];
    s[0] = r0 - kReOH;
    s[2] = r1 - kReOH;
    s[1] = r2 - kReHH;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double x = 0.5 * kGam[i] * s[i];
        if (x >= 43.0) {
            q[i] = 0.0;
            dq[i] = 0.0;
        } else {
            q[i] = x >= 15.0 ? 2.0 / (1.0 + exp(2.0 * x)) : 1.0 - tanh(x);
            const double ch = cosh(x);
            dq[i] = -0.5 * kGam[i] / (ch * ch);
        }
    }
    const double *c = kCon;
    const double p = c[0] + c[1] * (s[0] + s[2]) + c[2] * s[1] + 0.5 * c[3] * (s[0] * s[0] + s[2] * s[2]) +
                     0.5 * c[4] * s[1] * s[1] + c[5] * s[1] * (s[0] + s[2]) + c[6] * s[0] * s[2];
    const double e = q[0] * q[1] * q[2] * p;
    const double dp[3] = {c[1] + c[3] * s[0] + c[5] * s[1] + c[6] * s[2], c[2] + c[4] * s[1] + c[5] * (s[0] + s[2]),
                          c[1] + c[3] * s[2] + c[5] * s[1] + c[6] * s[0]};
#pragma unroll
    for (int i = 0; i < 3; ++i)
        if (q[i] != 0.0) dedr[i] = e * (dq[i] / q[i] + (dp[i] / p));
    const double t = dedr[1];
    dedr[1] = dedr[2];
    dedr[2] = t;
    return e;
}

__device__ inline double four_body(const double *r, double *dedr)
{
    const double e1 = r[0] - kAlp[0], e2 = r[1] - kAlp[0], e3 = r[2] - kAlp[2], e4 = r[3] - kAlp[2];
    const double f1 = r[0] - kAlp[1], f2 = r[1] - kAlp[1], f3 = r[2] - kAlp[3], f4 = r[3] - kAlp[3];
    const double t1 =
        exp(-kLam[0] * (e1 * e1) - kLam[0] * (e2 * e2) - kLam[2] * (e3 * e3) - kLam[2] * (e4 * e4)) * kAcon[0];
    const double t2 =
        exp(-kLam[1] * (f1 * f1) - kLam[1] * (f2 * f2) - kLam[3] * (f3 * f3) - kLam[3] * (f4 * f4)) * kAcon[1];
    dedr[0] = -2.0 * (t1 * kLam[0] * e1 + t2 * kLam[1] * f1);
    dedr[1] = -2.0 * (t1 * kLam[0] * e2 + t2 * kLam[1] * f2);
    dedr[2] = -2.0 * (t1 * kLam[2] * e3 + t2 * kLam[3] * f3);
    dedr[3] = -2.0 * (t1 * kLam[2] * e4 + t2 * kLam[3] * f4);
    return t1 + t2;
}

// V and dV/dR of the six distances, summed in the reference's order.
__device__ inline double pot(const double *r, double *dvdr)
{
    auto morse = [](int k, double rr, double &dv) {
        const double ex = exp(-kBeta[k] * (rr - kRe[k]));
        const double u = 1.0 - ex;
        dv = 2.0 * kBeta[k] * kDe[k] * u * ex;
        return kDe[k] * (u * u);
    };
    double d0, d3, d4;
    double v = morse(0, r[0], d0) + morse(1, r[3], d3) + morse(1, r[4], d4);
    dvdr[0] = d0;
    dvdr[3] = d3;
    dvdr[4] = d4;
    double sh[4];
    v = v + leps(r[1], r[2], r[5], sh);
    dvdr[1] = sh[0];
    dvdr[2] = sh[1];
    dvdr[5] = sh[2];
    v = v + h2o(r[0], r[1], r[3], sh);
    dvdr[0] = dvdr[0] + sh[0];
    dvdr[1] = dvdr[1] + sh[1];
    dvdr[3] = dvdr[3] + sh[2];
    v = v + h2o(r[0], r[2], r[4], sh);
    dvdr[0] = dvdr[0] + sh[0];
    dvdr[2] = dvdr[2] + sh[1];
    dvdr[4] = dvdr[4] + sh[2];
    const double r4[4] = {r[1], r[2], r[3], r[4]};
    v = v + four_body(r4, sh);
    dvdr[1] = dvdr[1] + sh[0];
    dvdr[2] = dvdr[2] + sh[1];
    dvdr[3] = dvdr[3] + sh[2];
    dvdr[4] = dvdr[4] + sh[3];
    return v - 2.0 * kDe[1] + kDe[2];
}

// One bead: x = (O, H1, H2, H3) xyz, g the same layout.  The chain rule adds
// each distance's term in the reference's order (O: R1 R2 R3; H1: R1 R4 R5;
// H2: R2 R4 R6; H3: R3 R5 R6), with u = dV/dR * dx / R.
__device__ inline void egrad_bead(const double *x, double &v, double *g)
{
    constexpr int pa[6] = {1, 2, 3, 2, 3, 3}, pb[6] = {0, 0, 0, 1, 1, 2};
    double d[6][3], r[6], dvdr[6];
#pragma unroll
    for (int m = 0; m < 6; ++m) {
#pragma unroll
        for (int c = 0; c < 3; ++c) d[m][c] = x[3 * pa[m] + c] - x[3 * pb[m] + c];
        r[m] = sqrt(d[m][0] * d[m][0] + d[m][1] * d[m][1] + d[m][2] * d[m][2]);
    }
    v = pot(r, dvdr);
    constexpr int terms[4][3] = {{0, 1, 2}, {0, 3, 4}, {1, 3, 5}, {2, 4, 5}};
#pragma unroll
    for (int at = 0; at < 4; ++at)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            double acc = 0.0;
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                const int m = terms[at][t];
                const double u = dvdr[m] * d[m][c] / r[m];
                acc = pa[m] == at ? acc + u : acc - u;
            }
            g[3 * at + c] = acc;
        }
}

// One bead on a quad of lanes: lane i owns atom i (O, H1, H2, H3).  The
// exponentials and hyperbolic functions, most of the one-lane time, go one
// distance to a lane in two rounds: R1, R2, R3, R4 on lanes 0..3, then R6, the
// two four-body Gaussians and R5; each switching factor of the H2O terms is
// evaluated once (R1's stands in both).  The combination of the terms, a few
// dozen products, is repeated on every lane.  x = this lane's atom, V on every
// lane, g = dV/dx of this lane's atom.
__device__ inline void egrad_quad(const double *x, double &v, double *g)
{
    using quad::bcast;
    using quad::dpp;
    using quad::perm;
    const int i = threadIdx.x & 3;
    double d1[3], d2[3], r1 = 0.0, r2 = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        d1[c] = dpp<perm(1, 2, 3, 2)>(x[c]) - dpp<perm(0, 0, 0, 1)>(x[c]);
        d2[c] = bcast<3>(x[c]) - dpp<perm(2, 1, 1, 1)>(x[c]);
        r1 += d1[c] * d1[c];
        r2 += d2[c] * d2[c];
    }
    r1 = sqrt(r1);
    r2 = sqrt(r2);
    const double R1 = bcast<0>(r1), R2 = bcast<1>(r1), R3 = bcast<2>(r1), R4 = bcast<3>(r1), R5 = bcast<3>(r2);
    // one switching factor at s = r - re: value and derivative over value (0, 0 where it vanishes)
    auto factor = [](double gam, double s, double &q, double &w) {
        const double y = 0.5 * gam * s;
        q = w = 0.0;
        if (y < 43.0) {
            q = y >= 15.0 ? 2.0 / (1.0 + exp(2.0 * y)) : 1.0 - tanh(y);
            const double ch = cosh(y);
            w = -0.5 * gam / (ch * ch) / q;
        }
    };
    double q1, w1, q2, w2;
    const bool hh = i == 3;
    const double x1 = exp(-(hh ? kBeta[1] : kBeta[0]) * (r1 - (hh ? kRe[1] : kRe[0])));
    factor(hh ? kGam[1] : kGam[0], r1 - (hh ? kReHH : kReOH), q1, w1);
    // four-body Gaussians over (R2, R3, R4, R5): the first on lane 1, the second on lane 2
    const bool g1 = i == 1;
    const double ao = g1 ? kAlp[0] : kAlp[1], ah = g1 ? kAlp[2] : kAlp[3];
    const double lo = g1 ? kLam[0] : kLam[1], lh = g1 ? kLam[2] : kLam[3];
    const double f2 = R2 - ao, f3 = R3 - ao, f4 = R4 - ah, f5 = R5 - ah;
    const double gauss = -lo * (f2 * f2) - lo * (f3 * f3) - lh * (f4 * f4) - lh * (f5 * f5);
    const double arg = i == 0 ? -kBeta[2] * (r2 - kRe[2]) : hh ? -kBeta[1] * (r2 - kRe[1]) : gauss;
    const double x2 = exp(arg);
    factor(kGam[1], R5 - kReHH, q2, w2);               // the same on every lane

    // Morse pairs R1, R4, R5
    auto morse = [](int k, double ex, double &dv) {
        const double u = 1.0 - ex;
        dv = 2.0 * kBeta[k] * kDe[k] * u * ex;
        return kDe[k] * (u * u);
    };
    double dv[6];
    v = morse(0, bcast<0>(x1), dv[0]) + morse(1, bcast<3>(x1), dv[3]) + morse(1, bcast<3>(x2), dv[4]);
    // LEPS over R2, R3, R6
    double sh[3];
    {
        constexpr double z = kSato, zpo = 1.0 + z, op3z = 1.0 + 3.0 * z, top3z = 2.0 * op3z, zp3 = z + 3.0,
                         tzp3 = 2.0 * zp3;
        const double e[3] = {bcast<1>(x1), bcast<2>(x1), bcast<0>(x2)};
        double exch[3], energy = 0.0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double do4z = kDe[j == 2 ? 2 : 0] / 4.0 / zpo;
            energy += do4z * (zp3 * e[j] - top3z) * e[j];
            exch[j] = do4z * (op3z * e[j] - tzp3) * e[j];
        }
        const double d12 = exch[0] - exch[1], d23 = exch[1] - exch[2], d31 = exch[2] - exch[0];
        const double rad = sqrt(d12 * d12 + d23 * d23 + d31 * d31), irad = 1.0 / rad;
        const double s2 = sqrt(2.0), s = exch[0] + exch[1] + exch[2];
        v = v + (energy - rad / s2);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int k = j == 2 ? 2 : 0;
            const double b = kBeta[k] * (kDe[k] / 4.0 / zpo) * 2.0;
            sh[j] = b * e[j] * ((3.0 * exch[j] - s) / s2 * (op3z * e[j] - zp3) * irad - zp3 * e[j] + op3z);
        }
        dv[1] = sh[0];
        dv[2] = sh[1];
        dv[5] = sh[2];
    }
    // H2O terms over (R1, R2, R4) and (R1, R3, R5); sh is the shared array
    auto h2o = [&](double s0, double s2, double s1, const double *q, const double *w) {
        const double *c = kCon;
        const double p = c[0] + c[1] * (s0 + s2) + c[2] * s1 + 0.5 * c[3] * (s0 * s0 + s2 * s2) + 0.5 * c[4] * s1 * s1 +
                         c[5] * s1 * (s0 + s2) + c[6] * s0 * s2;
        const double e = q[0] * q[1] * q[2] * p, ip = 1.0 / p;
        const double dp[3] = {c[1] + c[3] * s0 + c[5] * s1 + c[6] * s2, c[2] + c[4] * s1 + c[5] * (s0 + s2),
                              c[1] + c[3] * s2 + c[5] * s1 + c[6] * s0};
#pragma unroll
        for (int j = 0; j < 3; ++j) sh[j] = q[j] != 0.0 ? e * (w[j] + dp[j] * ip) : sh[j];
        const double t = sh[1];
        sh[1] = sh[2];
        sh[2] = t;
        return e;
    };
    const double qo = bcast<0>(q1), wo = bcast<0>(w1);
    {
        const double q[3] = {qo, bcast<3>(q1), bcast<1>(q1)}, w[3] = {wo, bcast<3>(w1), bcast<1>(w1)};
        v = v + h2o(R1 - kReOH, R2 - kReOH, R4 - kReHH, q, w);
        dv[0] = dv[0] + sh[0];
        dv[1] = dv[1] + sh[1];
        dv[3] = dv[3] + sh[2];
    }
    {
        const double q[3] = {qo, q2, bcast<2>(q1)}, w[3] = {wo, w2, bcast<2>(w1)};
        v = v + h2o(R1 - kReOH, R3 - kReOH, R5 - kReHH, q, w);
        dv[0] = dv[0] + sh[0];
        dv[2] = dv[2] + sh[1];
        dv[4] = dv[4] + sh[2];
    }
    {
        const double t1 = bcast<1>(x2) * kAcon[0], t2 = bcast<2>(x2) * kAcon[1];
        dv[1] -= 2.0 * (t1 * kLam[0] * (R2 - kAlp[0]) + t2 * kLam[1] * (R2 - kAlp[1]));
        dv[2] -= 2.0 * (t1 * kLam[0] * (R3 - kAlp[0]) + t2 * kLam[1] * (R3 - kAlp[1]));
        dv[3] -= 2.0 * (t1 * kLam[2] * (R4 - kAlp[2]) + t2 * kLam[3] * (R4 - kAlp[3]));
        dv[4] -= 2.0 * (t1 * kLam[2] * (R5 - kAlp[2]) + t2 * kLam[3] * (R5 - kAlp[3]));
        v = v + (t1 + t2);
    }
    v = v - 2.0 * kDe[1] + kDe[2];
    // the lane's distances' terms, gathered by atom in the reference's order
    const double u1 = (i == 0 ? dv[0] : i == 1 ? dv[1] : i == 2 ? dv[2] : dv[3]) / r1;
    const double u2 = (i == 0 ? dv[5] : dv[4]) / r2;
    const double s1 = i == 0 ? -1.0 : 1.0, s2 = i <= 1 ? -1.0 : 1.0, s3 = i <= 2 ? -1.0 : 1.0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double F1 = u1 * d1[c], F2 = u2 * d2[c];
        const double a = dpp<perm(0, 0, 1, 2)>(F1);
        const double b1 = dpp<perm(1, 3, 3, 3)>(F1), c1 = bcast<2>(F1), c2 = dpp<perm(0, 3, 0, 0)>(F2);
        g[c] = s1 * a + s2 * (i == 3 ? F2 : b1) + s3 * (i == 0 ? c1 : c2);
    }
}

}  // namespace oh3
}  // namespace cam
