// The reaction coordinate (calc_xi BIMOLEC, src/calc_xi.f90:63-523) of one
// trajectory's centroid evaluated by a group of lanes of one wave, for the
// step kernels, where it sits between the beads' forces and the second half
// kick of every step and everything waits for it.  One lane evaluating it
// alone (with indexed atoms as blends over all of them) took 11 us of a 21 us
// H3 window step: a serial chain of some thousand FP64 operations.  Here the
// distances are one lane each, the coordinates one lane each, and an atom is
// an index into LDS.
//
// Both dividing surfaces are sums over distances R_j = P_a - P_b between two
// points (an atom, or the centre of mass of a reactant):
//   s = sum_j wt_j (|R_j| - ref_j),
// the bonds (breaking +1/n, forming -1/n) in s1, the pairs of reactant
// centres (-1/terms, ref = r_inf) in s0.  With P_a - P_b = sum_at B_j[at] x_at
// the gradient is sum_j wt_j B_j[at] R_j / |R_j|, and the Hessian times a
// vector v is sum_j wt_j B_j[at] (|R_j|^2 u_j - R_j (R_j . u_j)) / |R_j|^3
// with u_j = sum_at B_j[at] v_at.
#pragma once
#include "step_common.hpp"

namespace cam {

// Host-built (engine.hip), one per engine, copied to LDS by every block.
constexpr int kXiMax = 2 * CAM_MAX_BONDS + CAM_MAX_REAC * (CAM_MAX_REAC - 1) / 2;
struct XiTable {
    int nd, nbond, n_reac, pad;                  // distances, the first nbond of them bonds
    int pa[kXiMax], pb[kXiMax];                  // 3 * point: atoms, then reactant centres from natoms on
    double wt[kXiMax], ref[kXiMax];
    double B[kXiMax][CAM_MAX_ATOMS];
    double fw[CAM_MAX_REAC][CAM_MAX_ATOMS];      // mass fractions of the reactants' atoms
    double inv_mass[CAM_MAX_ATOMS];
};

// Orders this wave's LDS accesses; the lanes of a group belong to one wave.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int NA>
struct XiGroup {
    static constexpr int N = 3 * NA, GL = N <= 16 ? 16 : 32;     // lanes of a group: one per coordinate
    static_assert(N <= GL && kXiMax <= GL && 3 * CAM_MAX_REAC <= GL, "a lane per coordinate and per distance");
    struct Work {                                // a group's LDS
        double pts[3 * (NA + CAM_MAX_REAC)];     // the centroid (written by the caller), then the centres
        double R[kXiMax][3], rinv[kXiMax], val[kXiMax], w[kXiMax][3];
        double v[N];
    };

    // Sum over the group's lanes, the same bits on all of them.
    __device__ static __forceinline__ double sum(double x)
    {
        for (int o = GL / 2; o > 0; o >>= 1) x += __shfl_xor(x, o, GL);
        return x;
    }

    // s0 and s1 on every lane and their derivatives by coordinate i on lane i
    // (0 on lanes past the last coordinate), at the positions in w.pts.
    __device__ static __forceinline__ void surfaces(const XiTable &t, Work &w, int i, double &s0, double &s1,
                                                    double &ds0, double &ds1)
    {
        wave_sync();
        if (i < 3 * t.n_reac) {
            double c = 0.0;
#pragma unroll
            for (int at = 0; at < NA; ++at) c = fma(t.fw[i / 3][at], w.pts[3 * at + i % 3], c);
            w.pts[N + i] = c;
        }
        wave_sync();
        if (i < t.nd) {
            double R[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) R[d] = w.R[i][d] = w.pts[t.pa[i] + d] - w.pts[t.pb[i] + d];
            const double r = sqrt(R[0] * R[0] + R[1] * R[1] + R[2] * R[2]);
            w.rinv[i] = 1.0 / r;
            w.val[i] = (r - t.ref[i]) * t.wt[i];
        }
        wave_sync();
        s0 = s1 = ds0 = ds1 = 0.0;
        const int at = i < N ? i / 3 : 0, d = i % 3;
        for (int j = 0; j < t.nd; ++j) {
            const double g = i < N ? t.wt[j] * t.B[j][at] * (w.R[j][d] * w.rinv[j]) : 0.0;
            if (j < t.nbond) {
                s1 += w.val[j];
                ds1 += g;
            } else {
                s0 += w.val[j];
                ds0 += g;
            }
        }
    }

    // Products of the Hessians of s0 and s1 with the vector w.v (written by
    // the caller), component i on lane i, at the distances of the last
    // surfaces().
    __device__ static __forceinline__ void hess_vec(const XiTable &t, Work &w, int i, double &h0, double &h1)
    {
        wave_sync();
        if (i < t.nd) {
            double u[3] = { 0.0, 0.0, 0.0 };
#pragma unroll
            for (int at = 0; at < NA; ++at)
#pragma unroll
                for (int d = 0; d < 3; ++d) u[d] = fma(t.B[i][at], w.v[3 * at + d], u[d]);
            const double R0 = w.R[i][0], R1 = w.R[i][1], R2 = w.R[i][2], ri = w.rinv[i];
            const double rr = R0 * R0 + R1 * R1 + R2 * R2, ru = R0 * u[0] + R1 * u[1] + R2 * u[2];
            const double f = t.wt[i] * (ri * ri * ri);
            w.w[i][0] = (rr * u[0] - R0 * ru) * f;
            w.w[i][1] = (rr * u[1] - R1 * ru) * f;
            w.w[i][2] = (rr * u[2] - R2 * ru) * f;
        }
        wave_sync();
        h0 = h1 = 0.0;
        const int at = i < N ? i / 3 : 0, d = i % 3;
        for (int j = 0; j < t.nd; ++j) {
            const double h = i < N ? t.B[j][at] * w.w[j][d] : 0.0;
            if (j < t.nbond) h1 += h;
            else h0 += h;
        }
    }

    // umbrella mode 0 (src/umbrella.f90:109-173; umbrella_bias has the
    // formulas): xi of mode 1 on every lane, the two parts of the bias
    // gradient of coordinate i on lane i.  w.pts holds the centroid.
    __device__ static __forceinline__ void bias(const XiTable &t, Work &w, int i, double beta, double k_force,
                                                double xi_ideal, double &xi1, double &gk, double &gh)
    {
        double s0, s1, ds0, ds1;
        surfaces(t, w, i, s0, s1, ds0, ds1);
        const double D = s0 - s1, inv_D = 1.0 / D, inv_D2 = inv_D * inv_D;
        xi1 = s0 * inv_D;
        const double dxi = (s0 * ds1 - s1 * ds0) * inv_D2;
        gk = k_force * (xi1 - xi_ideal) * dxi;
        const double v = i < N ? dxi * t.inv_mass[i / 3] : 0.0;
        if (i < N) w.v[i] = v;
        double h0, h1;
        hess_vec(t, w, i, h0, h1);
        const double fs2 = sum(dxi * v), ds0v = sum(ds0 * v), ds1v = sum(ds1 * v);
        const double cross = s0 * ds1v - s1 * ds0v;
        const double f = -1.0 / (beta * fs2) * inv_D2 * inv_D;
        gh = ((s0 * h1 + ds0 * ds1v - ds1 * ds0v - s1 * h0) * D - 2.0 * cross * (ds0 - ds1)) * f;
    }
};

}  // namespace cam
