// Removal of the overall translation and rotation of a ring polymer after a
// step (src/transrot.f90:36-237), shared by the step kernels and the
// one-wave-per-trajectory kernel of the split schedule.
//
// With the reference's total mass M' = nbeads sum(m) (sum over beads and
// atoms, times nbeads once more, src/transrot.f90:62-72): vtot = sum(p) / M',
// xt = sum(m q) / M', the angular momentum L = sum(q x p) - M' xt x vtot, the
// inertia tensor about xt, and p -= m (vtot + omega x (q - xt)) with I omega =
// L.  The reference divides momenta into velocities and multiplies back; the
// products cancel here, which differs in rounding only.
#pragma once
#include <hip/hip_runtime.h>

namespace cam {

// omega = I^-1 L for the symmetric tensor I = {xx, xy, xz, yy, yz, zz}, by
// symmetric elimination with the largest remaining diagonal element as the
// pivot (of a positive tensor the largest element is on the diagonal, the one
// the reference's full pivoting takes, src/invert.f90).  Every index is a
// compile-time constant and the exchanges are selects, so nothing goes to
// scratch memory.
__device__ __forceinline__ void inertia_solve(const double *I, const double *L, double *omega)
{
    double a00 = I[0], a01 = I[1], a02 = I[2], a11 = I[3], a12 = I[4], a22 = I[5];
    double b0 = L[0], b1 = L[1], b2 = L[2];
    auto swap_if = [](bool c, double &x, double &y) {
        const double t = c ? y : x;
        y = c ? x : y;
        x = t;
    };
    const int p = a22 > a00 && a22 > a11 ? 2 : a11 > a00 ? 1 : 0;
    swap_if(p == 1, a00, a11);
    swap_if(p == 1, a02, a12);
    swap_if(p == 1, b0, b1);
    swap_if(p == 2, a00, a22);
    swap_if(p == 2, a01, a12);
    swap_if(p == 2, b0, b2);
    const double i0 = 1.0 / a00;
    const double l1 = a01 * i0, l2 = a02 * i0;
    a11 = fma(-l1, a01, a11);
    a12 = fma(-l1, a02, a12);
    a22 = fma(-l2, a02, a22);
    b1 = fma(-l1, b0, b1);
    b2 = fma(-l2, b0, b2);
    const bool s = a22 > a11;
    swap_if(s, a11, a22);
    swap_if(s, a01, a02);
    swap_if(s, b1, b2);
    const double i1 = 1.0 / a11;
    const double l3 = a12 * i1;
    a22 = fma(-l3, a12, a22);
    b2 = fma(-l3, b1, b2);
    double x2 = b2 / a22;
    double x1 = (b1 - a12 * x2) * i1;
    double x0 = (b0 - a01 * x1 - a02 * x2) * i0;
    swap_if(s, x1, x2);
    swap_if(p == 1, x0, x1);
    swap_if(p == 2, x0, x2);
    omega[0] = x0;
    omega[1] = x1;
    omega[2] = x2;
}

// The first sums {sum p, sum m q}(6) of one atom of one bead added to v.
__device__ __forceinline__ void transrot_sums1(const double *q, const double *p, double m, double *v)
{
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        v[d] += p[d];
        v[3 + d] += q[d] * m;
    }
}

// The second sums {q x p (3), m (q - xt)(q - xt) (6)} of one atom of one bead
// added to v; xt the centre.
__device__ __forceinline__ void transrot_sums2(const double *q, const double *p, double m, const double *xt, double *v)
{
    v[0] += q[1] * p[2] - q[2] * p[1];
    v[1] += q[2] * p[0] - q[0] * p[2];
    v[2] += q[0] * p[1] - q[1] * p[0];
    const double x = q[0] - xt[0], y = q[1] - xt[1], z = q[2] - xt[2];
    const double mx = x * m, my = y * m, mz = z * m;
    v[3] += x * mx;
    v[4] += x * my;
    v[5] += x * mz;
    v[6] += y * my;
    v[7] += y * mz;
    v[8] += z * mz;
}

// vtot, xt (the first sums over M') and omega from the second sums.
__device__ __forceinline__ void transrot_omega(const double *vtot, const double *xt, const double *s2, double totmass,
                                               double *omega)
{
    double L[3];
    L[0] = s2[0] - (xt[1] * vtot[2] - xt[2] * vtot[1]) * totmass;
    L[1] = s2[1] - (xt[2] * vtot[0] - xt[0] * vtot[2]) * totmass;
    L[2] = s2[2] - (xt[0] * vtot[1] - xt[1] * vtot[0]) * totmass;
    const double I[6] = { s2[6] + s2[8], -s2[4], -s2[5], s2[3] + s2[8], -s2[7], s2[3] + s2[6] };
    inertia_solve(I, L, omega);
}

// p -= m (vtot + omega x (q - xt)) of one atom of one bead.
__device__ __forceinline__ void transrot_apply(const double *q, double *p, double m, const double *vtot,
                                               const double *xt, const double *omega)
{
    const double x = q[0] - xt[0], y = q[1] - xt[1], z = q[2] - xt[2];
    p[0] -= m * (vtot[0] + (omega[1] * z - omega[2] * y));
    p[1] -= m * (vtot[1] + (omega[2] * x - omega[0] * z));
    p[2] -= m * (vtot[2] + (omega[0] * y - omega[1] * x));
}

}  // namespace cam
