// Nose-Hoover chain thermostat shared by the trajectory engine and the box.
#pragma once

#include <hip/hip_runtime.h>

namespace cam {

// a / q from iq = 1/q: the product corrected by its own remainder, so within a
// rounding of the quotient, in three dependent operations instead of a division.
__device__ __forceinline__ double nhc_quot(double a, double q, double iq)
{
    const double r = a * iq;
    return fma(fma(-q, r, a), iq, r);
}

// The Nose-Hoover chain of one system (a trajectory, or a box) over half a
// time step (src/nhc.f90:35-169): four thermostats with velocities vnh and masses qnh,
// nc = 5 substeps of the 3-stage Suzuki-Yoshida factorisation, on the
// centroid-momenta kinetic energy eksum.  Returns the factor that scales
// every momentum.  ekt is the chain's kT.
//
// One lane, one dependent chain of 15 stages.  Bound by its latency: eight
// divisions and seven exponentials a stage took 9.2 us.  Divisions by the
// masses go through their reciprocals, and the exponentials of the way back
// through the chain are those of the way in (their velocities have not
// changed): 7.5 us, launch included.
__device__ inline double nhc_chain(double *vnh, const double *qnh, double eksum, double ekt, int nfree, double dt)
{
    const double w0 = 1.0 / (2.0 - 1.2599210498948731648);      // 2 - cbrt(2)
    const double dtc = dt / 5.0;
    const double i0 = 1.0 / qnh[0], i1 = 1.0 / qnh[1], i2 = 1.0 / qnh[2], i3 = 1.0 / qnh[3];
    const double nkt = (double)nfree * ekt;
    double v0 = vnh[0], v1 = vnh[1], v2 = vnh[2], v3 = vnh[3], scale = 1.0;
    for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double dts = (j == 1 ? 1.0 - 2.0 * w0 : w0) * dtc;
            const double dt2 = 0.5 * dts, dt4 = 0.25 * dts, dt8 = 0.125 * dts;
            v3 = v3 + nhc_quot(qnh[2] * v2 * v2 - ekt, qnh[3], i3) * dt4;
            const double e3 = exp(-v3 * dt8);
            v2 = e3 * (v2 * e3 + nhc_quot(qnh[1] * v1 * v1 - ekt, qnh[2], i2) * dt4);
            const double e2 = exp(-v2 * dt8);
            v1 = e2 * (v1 * e2 + nhc_quot(qnh[0] * v0 * v0 - ekt, qnh[1], i1) * dt4);
            const double e1 = exp(-v1 * dt8);
            v0 = e1 * (v0 * e1 + nhc_quot(2.0 * eksum - nkt, qnh[0], i0) * dt4);
            const double e0 = exp(-v0 * dt2);
            scale = scale * e0;
            eksum = eksum * e0 * e0;
            v0 = e1 * (v0 * e1 + nhc_quot(2.0 * eksum - nkt, qnh[0], i0) * dt4);
            v1 = e2 * (v1 * e2 + nhc_quot(qnh[0] * v0 * v0 - ekt, qnh[1], i1) * dt4);
            v2 = e3 * (v2 * e3 + nhc_quot(qnh[1] * v1 * v1 - ekt, qnh[2], i2) * dt4);
            v3 = v3 + nhc_quot(qnh[2] * v2 * v2 - ekt, qnh[3], i3) * dt4;
        }
    vnh[0] = v0;
    vnh[1] = v1;
    vnh[2] = v2;
    vnh[3] = v3;
    return scale;
}

}  // namespace cam
