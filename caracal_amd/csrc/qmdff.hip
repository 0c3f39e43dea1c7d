// The reference's QMDFF force field on the device (ff_eg + ff_nonb + ff_hb as
// src/gradient.f90:341-348 calls them for one QMDFF), for nbeads replicas of
// one structure at once: the box engine's force field for QMDFF boxes.
//
// Kernels of one evaluation (positions and gradients [bead][atom][3]):
//   qm_terms_kernel   everything that does not depend on other terms, a role
//                     per block:
//     pairs of atoms of different molecules (dispersion, repulsion, Coulomb;
//       src/ff_nonb.f90:198-332, :453-509): one wave per atom i; the atoms j
//       within the cutoff are queued and evaluated 64 at a time (qinter); every
//       pair is evaluated from both sides, so no atomics are needed;
//     intermolecular hydrogen bonds (src/ff_hb.f90:198-276): every donor bond
//       A-H against every acceptor atom j of another molecule, once from the
//       acceptor's side (its gradient and the energy) and once from the
//       donor's (the A and H gradients), one wave each;
//     the slots of bonds, bends, torsions, nci pairs and listed hydrogen bonds,
//       one lane each;
//   qm_gather_kernel  four lanes per (bead, atom): the bonded terms, the nci
//                     pairs and the listed hydrogen bonds the atom takes part
//                     in (a term is evaluated once per atom it moves and its
//                     energy counted at its first atom), plus the partials
//                     above, in a fixed order;
//   qm_reduce_kernel  per-bead energies from the block partials in a fixed
//                     order.
// Results are bitwise reproducible run to run.  Arithmetic follows the
// reference routine by routine, quirks included (abdamp's single-precision
// constant, the unsigned torsion angle, q q / r^2 Coulomb gradients for the
// Zahn energy, eabhag's minimum image on the A-H vector only, hydrogen-bond
// thresholds in default-REAL literals).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <vector>

#include "qmdff.hpp"
#include "quad.hpp"

namespace cam {

constexpr int kQTile = 256;         // lanes per block; j atoms per LDS tile
constexpr int kQWaves = kQTile / 64;    // waves per block: atoms i of an intermolecular block
constexpr int kQSplit = 8;          // parts of the j range that are summed on their own
constexpr int kQMaxElem = 16;       // distinct elements of one force field
constexpr int kQImageCap = 64;      // minimum-image iterations (the reference loops until inside)

struct QDev {
    int n, ne, nbond, nangl, ntors, nnci, nhb, ndon, nacc;
    int periodic, zahn, inter;          // inter: more than one molecule
    double box[3], box2[3], ibox[3];
    double coul_cut, vdw_cut, cut_low, zahn_a, zahn_par;
    double eps1[6], eps2[6];
    const int *elem;                    // n: element slot 0..ne-1
    const int *mol;                     // n: molecule number
    const double *q;                    // n
    const double *c6;                   // n * n, [i][j]: the row of atom i holds the C6 its pairs use
    const double *r0, *r06, *sr42, *zab, *alpha;   // ne * ne: [slot_i][slot_j]
    const double *rad;                  // ne (bohr)
    const int *bond, *angl, *tors, *nci, *hb;      // 0-based atoms
    const double *vbond, *vangl, *vtors, *vhb;
    const int *rptr, *rcode;            // per atom: the term slots (and hydrogen-bond parts) it takes part in
    int sbase[5], nslot;                // first slot of bonds, bends, torsions, nci pairs, listed H-bonds
    const int *don, *acc;               // donor bonds (A, H) and acceptor atoms
    const double *don_lim, *acc_lim;    // hydrogen-bond distance thresholds
    const double *hbc;                  // n: hbpara(10, 5, q) * scalehb
    const double *scal;                 // n: scalehb of the atom's element
};

// term codes of the per-atom lists: kind << 28 | role << 26 | index
enum { kTBond = 0, kTAngle = 1, kTTors = 2, kTNci = 3, kTHbList = 4, kTHbAcc = 5, kTHbDon = 6 };

struct QmdffDev {
    QDev d{};
    std::vector<void *> allocs;
    double *gpart = nullptr, *epart = nullptr, *gacc = nullptr, *eacc = nullptr, *gdon = nullptr;
    double *gslot = nullptr, *eslot = nullptr;
    int cap_beads = 0;
};

namespace {

__device__ inline void qimg(const QDev &f, double *d)
{
    if (!f.periodic) return;
#pragma unroll
    for (int c = 0; c < 3; ++c)
        for (int it = 0; it < kQImageCap && fabs(d[c]) > f.box2[c]; ++it) d[c] = d[c] - copysign(f.box[c], d[c]);
}

__device__ inline void qsub(const double *x, int a, int b, double *d)
{
    d[0] = x[3 * a] - x[3 * b];
    d[1] = x[3 * a + 1] - x[3 * b + 1];
    d[2] = x[3 * a + 2] - x[3 * b + 2];
}

__device__ inline void qcross(const double *a, const double *b, double *c)
{
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
}

__device__ inline double qnorm(double *r, bool normalise)
{
    const double sp = (r[0] * r[0] + r[1] * r[1]) + r[2] * r[2];
    const double rn = sqrt(sp);
    if (normalise && fabs(rn) > 1e-14) {
        const double o = 1.0 / rn;
        r[0] = o * r[0];
        r[1] = o * r[1];
        r[2] = o * r[2];
    }
    return rn;
}

__device__ inline double qdot(const double *a, const double *b) { return (a[0] * b[0] + a[1] * b[1]) + a[2] * b[2]; }

// abdamp (src/abdamp.f90:36-51)
__device__ inline void qabdamp(const QDev &f, int ea, int eb, double r2, double &damp, double &ddamp)
{
    const double c = (double)(3.0f * 3.5710642f);
    const double s = f.rad[ea] + f.rad[eb];
    const double rcut = c * (s * s);
    const double rr = (r2 / rcut) * (r2 / rcut);
    damp = 1.0 / (1.0 + rr);
    ddamp = -2.0 * 2 * rr / (r2 * ((1.0 + rr) * (1.0 + rr)));
}

// bond stretch m, gradient on its atom of the given role (src/ff_eg.f90:87-163)
__device__ void qbond(const QDev &f, const double *x, int m, int role, double &e, double *gv)
{
    const int i = f.bond[2 * m], j = f.bond[2 * m + 1];
    double rb[3];
    qsub(x, i, j, rb);
    qimg(f, rb);
    const double r2 = (rb[0] * rb[0] + rb[1] * rb[1]) + rb[2] * rb[2];
    const double r = sqrt(r2);
    const double rij = f.vbond[3 * m], kij = f.vbond[3 * m + 1], aai = f.vbond[3 * m + 2];
    const double aai2 = aai / 2;
    const double p1 = pow(rij / r, aai), p2 = pow(rij / r, aai2);
    e = kij * (1.0 + p1 - 2.0 * p2);
    const double fac = aai * kij * (-p1 + p2) / r2;
    const double sgn = role == 0 ? 1.0 : -1.0;
    for (int c = 0; c < 3; ++c) gv[c] = sgn * (fac * rb[c]);
}

// bend m (src/ff_eg.f90:167-299): vertex angl[0]; roles 0 vertex, 1 and 2 the outer atoms
__device__ void qangle(const QDev &f, const double *x, int m, int role, double &e, double *gv)
{
    const int j = f.angl[3 * m], i = f.angl[3 * m + 1], k = f.angl[3 * m + 2];
    const double c0 = f.vangl[2 * m], kijk = f.vangl[2 * m + 1];
    double vab[3], vcb[3], vp[3], deda[3], dedc[3];
    qsub(x, i, j, vab);
    qsub(x, k, j, vcb);
    qimg(f, vab);
    qimg(f, vcb);
    const double rab2 = (vab[0] * vab[0] + vab[1] * vab[1]) + vab[2] * vab[2];
    const double rcb2 = (vcb[0] * vcb[0] + vcb[1] * vcb[1]) + vcb[2] * vcb[2];
    qcross(vcb, vab, vp);
    const double tp = (vp[0] * vp[0] + vp[1] * vp[1]) + vp[2] * vp[2];
    const double rp = (tp > 0.0 ? sqrt(tp) : 0.0) + 1e-14;
    const double rimp = qdot(vab, vcb);
    const double al = rab2 > 0.0 ? sqrt(rab2) : 0.0, bl = rcb2 > 0.0 ? sqrt(rcb2) : 0.0;
    double cosa = (al > 0.0 && bl > 0.0) ? rimp / (al * bl) : 0.0;
    cosa = fmin(1.0, fmax(-1.0, cosa));
    const double theta = acos(cosa);
    double dij, d2ij, djk, d2jk;
    qabdamp(f, f.elem[i], f.elem[j], rab2, dij, d2ij);
    qabdamp(f, f.elem[k], f.elem[j], rcb2, djk, d2jk);
    const double damp = dij * djk;
    double ea, deddt;
    if (3.1415926535897932384626433832795029 - c0 < 1e-6) {
        const double dt = theta - c0;
        ea = kijk * (dt * dt);
        deddt = 2.0 * kijk * dt;
    } else {
        const double dc = cosa - cos(c0);
        ea = kijk * (dc * dc);
        deddt = 2.0 * kijk * sin(theta) * (cos(c0) - cosa);
    }
    e = ea * damp;
    qcross(vab, vp, deda);
    const double rm1 = -deddt / (rab2 * rp);
    qcross(vcb, vp, dedc);
    const double rm2 = deddt / (rcb2 * rp);
    for (int c = 0; c < 3; ++c) {
        const double a = deda[c] * rm1, cc = dedc[c] * rm2;
        const double t1 = ea * d2ij * djk * vab[c], t2 = ea * d2jk * dij * vcb[c];
        if (role == 1) gv[c] = a * damp + t1;
        else if (role == 0) gv[c] = -(a + cc) * damp - t1 - t2;
        else gv[c] = cc * damp + t2;
    }
}

// torsion or out-of-plane term m (src/ff_eg.f90:303-619, src/valijkl.f90,
// src/dphidr.f90, src/omega.f90, src/domegadr.f90); roles 0..3 = i, j, k, l
__device__ void qtors(const QDev &f, const double *x, int m, int role, double &e, double *gv)
{
    const int *t = f.tors + 6 * m;
    const double *vt = f.vtors + 14 * m;
    const int i = t[0], j = t[1], k = t[2], l = t[3], nt = t[4];
    const double phi0 = vt[0];
    const double PI = 3.1415926535897932384626433832795029, PI2 = 6.28318530717958623199592693708837;
    const double SPI = 1.77245385090551599275151910313925;
    double vab[3], vcb[3], vdc[3], dd[3];
    double et = 0.0, dij = 0.0;
    if (t[5] != 2) {
        qsub(x, i, j, vab);
        qsub(x, j, k, vcb);
        qsub(x, k, l, vdc);
        qimg(f, vab);
        qimg(f, vcb);
        qimg(f, vdc);
        double dpij, d2ij, dpjk, d2jk, dpkl, d2kl;
        qabdamp(f, f.elem[i], f.elem[j], (vab[0] * vab[0] + vab[1] * vab[1]) + vab[2] * vab[2], dpij, d2ij);
        qabdamp(f, f.elem[k], f.elem[j], (vcb[0] * vcb[0] + vcb[1] * vcb[1]) + vcb[2] * vcb[2], dpjk, d2jk);
        qabdamp(f, f.elem[k], f.elem[l], (vdc[0] * vdc[0] + vdc[1] * vdc[1]) + vdc[2] * vdc[2], dpkl, d2kl);
        const double damp = dpjk * dpij * dpkl;
        // valijkl: the unsigned dihedral
        double ra[3], rb[3], rc[3], na[3], nb[3];
        qsub(x, j, i, ra);
        qsub(x, k, j, rb);
        qsub(x, l, k, rc);
        qimg(f, ra);
        qimg(f, rb);
        qimg(f, rc);
        qcross(ra, rb, na);
        qcross(rb, rc, nb);
        double nau[3] = { na[0], na[1], na[2] }, nbu[3] = { nb[0], nb[1], nb[2] };
        qnorm(nau, true);
        qnorm(nbu, true);
        double sab = qdot(nau, nbu);
        if (fabs(fabs(sab) - 1.0) < 1e-14) sab = copysign(1.0, sab);
        const double phi = acos(sab);
        // dphidr, only the row of this role
        const double cosphi = cos(phi), sinphi = sin(phi);
        const double nan_ = qnorm(na, false), nbn = qnorm(nb, false);
        const double nenner = nan_ * nbn * sinphi;
        if (fabs(nenner) < 1e-14) {
            dd[0] = dd[1] = dd[2] = 0.0;
        } else {
            const double on = 1.0 / nenner;
            double u[3], v[3], w[3], z[3];
            if (role == 0) {
                qcross(na, rb, u);
                qcross(nb, rb, v);
                for (int c = 0; c < 3; ++c) dd[c] = on * (cosphi * nbn / nan_ * u[c] - v[c]);
            } else if (role == 1) {
                double rapb[3] = { ra[0] + rb[0], ra[1] + rb[1], ra[2] + rb[2] };
                qcross(rapb, na, u);     // rapba
                qcross(nb, rc, v);       // rbc
                qcross(na, rc, w);       // rac
                qcross(rapb, nb, z);     // rapbb
                for (int c = 0; c < 3; ++c)
                    dd[c] = on * (cosphi * (nbn / nan_ * u[c] + nan_ / nbn * v[c]) - (w[c] + z[c]));
            } else if (role == 2) {
                double rbpc[3] = { rb[0] + rc[0], rb[1] + rc[1], rb[2] + rc[2] };
                qcross(na, ra, u);       // raa
                qcross(rbpc, nb, v);     // rbpcb
                qcross(nb, ra, w);       // rba
                qcross(rbpc, na, z);     // rbpca
                for (int c = 0; c < 3; ++c)
                    dd[c] = on * (cosphi * (nbn / nan_ * u[c] + nan_ / nbn * v[c]) - (w[c] + z[c]));
            } else {
                qcross(nb, rb, u);       // rbb
                qcross(na, rb, v);       // rab
                for (int c = 0; c < 3; ++c) dd[c] = on * (cosphi * nan_ / nbn * u[c] - v[c]);
            }
        }
        int mm = 2;
        for (int it = 0; it < nt; ++it) {
            const double rn = vt[mm];
            const double dphi1 = phi - phi0, dphi2 = phi + phi0 - PI2;
            const double c1 = rn * dphi1 + vt[mm + 1], c2 = rn * dphi2 + vt[mm + 1];
            const double x1cos = cos(c1), x2cos = cos(c2), x1sin = sin(c1), x2sin = sin(c2);
            const double phipi = phi - PI;
            const double ef = erf(phipi);
            const double ea1 = vt[mm + 2] * (1.0 + x1cos), ea2 = vt[mm + 2] * (1.0 + x2cos);
            et = et + 0.5 * (1.0 - ef) * ea1 + (0.5 + 0.5 * ef) * ea2;
            const double expo = exp(-(phipi * phipi)) / SPI;
            dij = dij - expo * ea1 - 0.5 * (1.0 - ef) * vt[mm + 2] * x1sin * rn + expo * ea2 -
                  (0.5 + 0.5 * ef) * vt[mm + 2] * x2sin * rn;
            mm = mm + 3;
        }
        et = et * vt[1];
        dij = dij * vt[1] * damp;
        double t1[3], t2[3], t3[3];
        for (int c = 0; c < 3; ++c) {
            t1[c] = et * d2ij * dpjk * dpkl * vab[c];
            t2[c] = et * d2jk * dpij * dpkl * vcb[c];
            t3[c] = et * d2kl * dpij * dpjk * vdc[c];
        }
        for (int c = 0; c < 3; ++c) {
            if (role == 0) gv[c] = dij * dd[c] + t1[c];
            else if (role == 1) gv[c] = dij * dd[c] - t1[c] + t2[c];
            else if (role == 2) gv[c] = dij * dd[c] + t3[c] - t2[c];
            else gv[c] = dij * dd[c] - t3[c];
        }
        e = et * damp;
    } else {
        qsub(x, j, i, vab);
        qsub(x, j, k, vcb);
        qsub(x, j, l, vdc);
        qimg(f, vab);
        qimg(f, vcb);
        qimg(f, vdc);
        double dpij, d2ij, dpjk, d2jk, dpjl, d2jl;
        qabdamp(f, f.elem[i], f.elem[j], (vab[0] * vab[0] + vab[1] * vab[1]) + vab[2] * vab[2], dpij, d2ij);
        qabdamp(f, f.elem[k], f.elem[j], (vcb[0] * vcb[0] + vcb[1] * vcb[1]) + vcb[2] * vcb[2], dpjk, d2jk);
        qabdamp(f, f.elem[j], f.elem[l], (vdc[0] * vdc[0] + vdc[1] * vdc[1]) + vdc[2] * vdc[2], dpjl, d2jl);
        const double damp = dpjk * dpij * dpjl;
        // omega and domegadr
        double re[3], rd[3], rv[3], rn[3];
        qsub(x, i, j, re);
        qsub(x, k, j, rd);
        qsub(x, l, i, rv);
        qimg(f, re);
        qimg(f, rd);
        qimg(f, rv);
        qcross(re, rd, rn);
        double rnu[3] = { rn[0], rn[1], rn[2] }, rvu[3] = { rv[0], rv[1], rv[2] };
        qnorm(rnu, true);
        qnorm(rvu, true);
        const double om = asin(qdot(rnu, rvu));
        const double sinom = sin(om);
        const double rvn = qnorm(rv, false), rnn = qnorm(rn, false);
        const double nenner = rnn * rvn * cos(om);
        if (fabs(nenner) > 1e-14) {
            const double on = 1.0 / nenner;
            double u[3], v[3];
            double rdme[3] = { rd[0] - re[0], rd[1] - re[1], rd[2] - re[2] };
            if (role == 0) {
                qcross(rd, rv, u);       // rdv
                qcross(rd, rn, v);       // rdn
                for (int c = 0; c < 3; ++c) dd[c] = on * (u[c] - rn[c] - sinom * (rvn / rnn * v[c] - rnn / rvn * rv[c]));
            } else if (role == 1) {
                qcross(rv, rdme, u);     // rvdme
                qcross(rn, rdme, v);     // rndme
                for (int c = 0; c < 3; ++c) dd[c] = on * (u[c] - sinom * rvn / rnn * v[c]);
            } else if (role == 2) {
                qcross(rv, re, u);       // rve
                qcross(rn, re, v);       // rne
                for (int c = 0; c < 3; ++c) dd[c] = on * (u[c] - sinom * rvn / rnn * v[c]);
            } else {
                for (int c = 0; c < 3; ++c) dd[c] = on * (rn[c] - sinom * rnn / rvn * rv[c]);
            }
        } else {
            dd[0] = dd[1] = dd[2] = 0.0;
        }
        const double rnt = vt[2];
        if (rnt > 1e-6) {
            const double c1 = (om - phi0) + PI;
            et = (1.0 + cos(c1)) * vt[1];
            dij = -sin(c1) * vt[1] * damp;
        } else {
            const double dc = cos(om) - cos(phi0);
            et = vt[1] * (dc * dc);
            dij = 2.0 * vt[1] * sin(om) * (cos(phi0) - cos(om)) * damp;
        }
        double t1[3], t2[3], t3[3];
        for (int c = 0; c < 3; ++c) {
            t1[c] = et * d2ij * dpjk * dpjl * vab[c];
            t2[c] = et * d2jk * dpij * dpjl * vcb[c];
            t3[c] = et * d2jl * dpij * dpjk * vdc[c];
        }
        for (int c = 0; c < 3; ++c) {
            if (role == 0) gv[c] = dij * dd[c] - t1[c];
            else if (role == 1) gv[c] = dij * dd[c] + t1[c] + t2[c] + t3[c];
            else if (role == 2) gv[c] = dij * dd[c] - t2[c];
            else gv[c] = dij * dd[c] - t3[c];
        }
        e = et * damp;
    }
}

// Dispersion and repulsion of the pair (a, b) scaled by s, gradient on a for
// d = x_a - x_b (src/ff_nonb.f90:118-175, :228-320); T is the arithmetic, t
// the element tables (of QDev, or their copy in LDS) and pe the pair's place.
struct QTables {
    const double *r0, *r06, *sr42, *zab, *alpha;
};

template <typename T>
__device__ inline void qdisp_rep(const QTables &f, int pe, double c6d, const T *d, T r2, T r, T s, T &e, T *ga)
{
    const T R0 = (T)f.r0[pe];
    const T c6 = (T)c6d;
    const T r4 = r2 * r2, r6 = r4 * r2;
    const T r06 = (T)f.r06[pe];
    const T t6 = r6 + r06, t8 = r6 * r2 + r06 * R0 * R0;
    const T c6t6 = c6 / t6, c6t8 = c6 / t8;
    T t27 = (T)f.sr42[pe] * c6t8;
    e = -(c6t6 + t27) * s;
    T drij = s * (c6t6 * (T)6.0 * r4 / t6 + (T)8.0 * t27 * r6 / t8);
    for (int c = 0; c < 3; ++c) ga[c] = d[c] * drij;
    if (r < (T)25) {
        const T xz = (T)f.zab[pe], alpha = (T)f.alpha[pe];
        t27 = xz * exp(-alpha * r);
        const T oner = (T)1.0 / r;
        e = e + t27 * oner * s;
        drij = s * t27 * (alpha * r + (T)1.0) * oner / r2;
        for (int c = 0; c < 3; ++c) ga[c] = ga[c] - d[c] * drij;
    }
}

// Coulomb of the pair (src/ff_nonb.f90:400-509); false outside the cutoff
template <typename T>
__device__ inline bool qcoulomb(const QDev &f, double qa, double qb, const T *d, T r2, T r, T scale, T &e, T *ga)
{
    T sw = (T)1.0;
    if (f.periodic) {
        if (r > (T)f.coul_cut) return false;
        if (!f.zahn && r > (T)f.cut_low) {
            const T xv = (r - (T)f.cut_low) / ((T)f.coul_cut - (T)f.cut_low);
            sw = (T)exp(1.0) * exp((T)1.0 / (xv - (T)1.0));
        }
    }
    if (r > (T)f.coul_cut) return false;
    const T oner = (T)1.0 / r;
    if (f.zahn)
        e = (T)qa * (T)qb * ((erfc((T)f.zahn_a * r) * oner) - (T)f.zahn_par * (r - (T)f.coul_cut));
    else
        e = (T)qa * (T)qb * oner * scale * sw;
    const T drij = e / r2;
    for (int c = 0; c < 3; ++c) ga[c] = -d[c] * drij;
    return true;
}

// nci pair m, gradient on its atom of the given role (src/ff_nonb.f90:88-193, :400-449)
__device__ void qnci(const QDev &f, const double *x, int m, int role, double &e, double *gv)
{
    const int i1 = f.nci[3 * m], i2 = f.nci[3 * m + 1], nk = f.nci[3 * m + 2] - 1;
    double d[3];
    qsub(x, i1, i2, d);
    qimg(f, d);
    const double r2 = (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2];
    const double r = sqrt(r2);
    const double vdw = f.periodic ? f.vdw_cut : 10.0 / 0.52917721092;
    double ga[3] = { 0.0, 0.0, 0.0 }, gc[3];
    e = 0.0;
    if (!(f.periodic && r > vdw))
        qdisp_rep<double>({ f.r0, f.r06, f.sr42, f.zab, f.alpha }, f.elem[i1] * f.ne + f.elem[i2],
                          f.c6[(size_t)i1 * f.n + i2], d, r2, r, f.eps2[nk], e, ga);
    double ec;
    if (qcoulomb<double>(f, f.q[i1], f.q[i2], d, r2, r, f.eps1[nk], ec, gc)) {
        e = e + ec;
        for (int c = 0; c < 3; ++c) ga[c] = ga[c] + gc[c];
    }
    const double sgn = role == 0 ? 1.0 : -1.0;
    for (int c = 0; c < 3; ++c) gv[c] = sgn * ga[c];
}

// eabhag (src/eabhag.f90): energy and the gradient of all three atoms.  PART
// kHbAcceptor: only the energy and ga are used, kHbDonor: only gb and gh.
// Those two state which product of a sum is rounded: left to the compiler it
// is one or the other with what else is in the kernel, and the bits with it.
enum { kHbListed = 0, kHbAcceptor = 1, kHbDonor = 2 };

template <int PART>
__device__ double qeabhag(const QDev &f, const double *x, int A, int B, int H, double ca, double cb, double *ga,
                          double *gb, double *gh)
{
    const double longcut = 8.0, alp7 = 12.0, alp3 = 6.0;
    double drah[3], drbh[3], drab[3], dg[3], dg2[3];
    qsub(x, A, H, drah);
    qsub(x, B, H, drbh);
    qsub(x, A, B, drab);
    qimg(f, drah);
    const double rab2 = (drab[0] * drab[0] + drab[1] * drab[1]) + drab[2] * drab[2];
    const double rab = sqrt(rab2);
    const double rah2 = (drah[0] * drah[0] + drah[1] * drah[1]) + drah[2] * drah[2];
    const double rah = sqrt(rah2);
    const double rbh2 = (drbh[0] * drbh[0] + drbh[1] * drbh[1]) + drbh[2] * drbh[2];
    const double rbh = sqrt(rbh2);
    const double ratio = pow(rab / longcut, alp7);
    double rdampl = 1.0 / (1.0 + ratio);
    rdampl = rdampl / rab2 / rab;
    double aprod, cosabh;
    if (rah2 > rbh2) {
        aprod = 1.0 / rbh / rab;
        cosabh = -qdot(drbh, drab) * aprod;
    } else {
        aprod = 1.0 / rah / rab;
        cosabh = qdot(drah, drab) * aprod;
    }
    double aterm = 0.5 * (cosabh + 1.0);
    double apref = pow(aterm, alp3 - 1);
    aterm = aterm * apref;
    apref = alp3 * 0.5 * apref;
    const double rah4 = rah2 * rah2, rbh4 = rbh2 * rbh2;
    const double denom = 1.0 / (PART == kHbListed     ? rah4 + rbh4
                                : PART == kHbAcceptor ? fma(rah2, rah2, rbh4)
                                                      : fma(rbh2, rbh2, rah4));
    const double da = (ca * rah4 + cb * rbh4) * denom;
    const double eabh = -da * rdampl * aterm;
    if (eabh > -1e-8) {
        for (int c = 0; c < 3; ++c) ga[c] = gb[c] = gh[c] = 0.0;
        return 0.0;
    }
    double gi = 4.0 * (ca - cb) * rah2 * rbh4 * denom * denom;
    gi = -gi * rdampl * aterm;
    double gib = 4.0 * (cb - ca) * rbh2 * rah4 * denom * denom;
    gib = -gib * rdampl * aterm;
    double gd = rdampl * rdampl * rab * (3.0 + (3.0 + alp7) * ratio);
    gd = gd * da * aterm;
    const double ge = -da * rdampl * apref;
    if constexpr (PART == kHbListed) {
        for (int c = 0; c < 3; ++c) ga[c] = gi * drah[c];
        for (int c = 0; c < 3; ++c) gb[c] = gib * drbh[c];
        for (int c = 0; c < 3; ++c) gh[c] = -ga[c] - gb[c];
        for (int c = 0; c < 3; ++c) {
            dg[c] = gd * drab[c];
            ga[c] = ga[c] + dg[c];
            gb[c] = gb[c] - dg[c];
        }
    } else {
        for (int c = 0; c < 3; ++c) {
            const double gbh = gib * drbh[c];
            ga[c] = fma(gd, drab[c], gi * drah[c]);
            gb[c] = fma(-gd, drab[c], gbh);
            gh[c] = fma(-gi, drah[c], -gbh);
        }
    }
    if (rah2 > rbh2) {
        for (int c = 0; c < 3; ++c) {
            dg[c] = fma(-aprod, drbh[c], -(cosabh * drab[c] / rab2));
            dg2[c] = fma(aprod, drab[c], cosabh * drbh[c] / rbh2);
            ga[c] = fma(ge, dg[c], ga[c]);
            gh[c] = fma(ge, dg2[c], gh[c]);
            gb[c] = fma(-ge, dg2[c], fma(-ge, dg[c], gb[c]));
        }
    } else {
        for (int c = 0; c < 3; ++c) {
            dg[c] = fma(-aprod, drah[c], cosabh * drab[c] / rab2);
            dg2[c] = fma(-aprod, drab[c], cosabh * drah[c] / rah2);
            gb[c] = fma(ge, dg[c], gb[c]);
            gh[c] = fma(ge, dg2[c], gh[c]);
            ga[c] = fma(-ge, dg2[c], fma(-ge, dg[c], ga[c]));
        }
    }
    return eabh;
}

// Listed hydrogen bond m (src/ff_hb.f90:60-86); roles 0 = A, 1 = B, 2 = H
__device__ void qhblist(const QDev &f, const double *x, int m, int role, double &e, double *gv)
{
    const int a = f.hb[3 * m], b = f.hb[3 * m + 1], h = f.hb[3 * m + 2];
    double d[3], ga[3], gb[3], gh[3];
    qsub(x, a, b, d);
    qimg(f, d);
    const double r = sqrt((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]);
    e = 0.0;
    gv[0] = gv[1] = gv[2] = 0.0;
    if (r > 15.0) return;
    e = qeabhag<kHbListed>(f, x, a, b, h, f.vhb[2 * m], f.vhb[2 * m + 1], ga, gb, gh);
    const double *s = role == 0 ? ga : role == 1 ? gb : gh;
    for (int c = 0; c < 3; ++c) gv[c] = s[c];
}

// Whether the intermolecular hydrogen bond of donor bond dn and acceptor slot
// ac, eabhag(j, A, H), counts (src/ff_hb.f90:198-276)
__device__ bool qhbnear(const QDev &f, const double *x, int dn, int ac)
{
    const int A = f.don[2 * dn], H = f.don[2 * dn + 1], j = f.acc[ac];
    if (f.mol[H] == f.mol[j]) return false;
    double d[3];
    qsub(x, A, j, d);
    qimg(f, d);
    const double r = sqrt((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]);
    if (r > 15.0) return false;
    const double cpar = f.scal[A] * f.scal[j];
    if (!(cpar > 1e-6)) return false;
    qsub(x, A, H, d);
    qimg(f, d);
    const double ri = sqrt((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]);
    qsub(x, j, H, d);
    qimg(f, d);
    const double rj = sqrt((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2]);
    return ri < f.don_lim[dn] || rj < f.acc_lim[ac];
}

// ---------------------------------------------------------------------------

// Sums of an atom's pair terms: FP64, compensated where the terms are binary32.
template <typename T>
struct QAcc {
    double s = 0.0;
    __device__ void add(T v) { s = s + (double)v; }
    __device__ double get() const { return s; }
};
template <>
struct QAcc<float> {
    double s = 0.0, c = 0.0;
    __device__ void add(float v)
    {
        const double y = (double)v - c;
        const double t = s + y;
        c = (t - s) - y;
        s = t;
    }
    __device__ double get() const { return s; }
};

// a + b, never fused with the product that a or b is.
template <typename T>
__device__ __forceinline__ T qadd(T a, T b)
{
#pragma clang fp contract(off)
    return a + b;
}

// Intermolecular pairs of atom i (one wave) with every other atom of a bead.
//
// A fifth of the atoms of the 51 bohr ethanol box lies within the 19 bohr
// cutoff.  With a lane per atom i and the block's 64 or 256 atoms walking all j
// together, nearly every j was inside for some lane, so every lane went
// through the whole pair (262 us for 1125 atoms x 16 beads).  Here the lanes
// stand for 64 atoms j: the distance check is a small part of a pair's work,
// those inside are queued, and the pair runs with the lanes full.
//
// The j range is summed in eighths, each in the order of j, and the gather adds
// the eighths in order: these are the sums, and the pair's are the operations,
// of lanes that walk an eighth each.  Summed over the lanes, or with 1/r and
// 1/t6 from reciprocal estimates (115 us a force call of 16 beads instead of
// 148), forces move by an ulp, which a torsion next to planar (1/sin phi) makes
// 1e-9 of the momenta in 50 steps.  A step takes eight atoms of every eighth,
// so that a batch holds some of each and the additions, which wait for each
// other, are few in a row: four lanes per eighth add the batch's terms from LDS
// (with the atoms taken in order, 28 in a row instead of 8, a call took 160 us).
struct QTile {
    double x[3][kQTile];                // j atoms of the tile
    int mol[kQTile];
    unsigned short queue[kQWaves][kQSplit][64];    // per wave and eighth: accepted atoms, from the eighth's first
    double res[kQWaves][67 * 4];        // per wave: the terms of a batch, [component][lane] (binary32 ones exact)
    double tab[5][kQMaxElem * kQMaxElem];
    double e[kQWaves];
};

// A wave's LDS queue is its own and its LDS accesses are in order: no barrier,
// only no reordering by the compiler.
__device__ __forceinline__ void qwave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// gpart: [eighth][bead][atom][3], here at this bead; stride between eighths.
template <typename T>
__device__ void qinter(const QDev &f, const double *__restrict__ x, int blk, QTile &s, double *gpart, size_t stride,
                       double *epart)
{
    const int n = f.n, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = blk * kQWaves + wave;
    const bool act = i < n;
    const int ii = act ? i : n - 1;
    const double xi0 = x[3 * ii], xi1 = x[3 * ii + 1], xi2 = x[3 * ii + 2];
    const int mi = f.mol[ii], ei = f.elem[ii] * f.ne;
    const double qi = f.q[ii];
    const double *c6 = f.c6 + (size_t)ii * n;
    for (int k = tid; k < f.ne * f.ne; k += kQTile) {
        s.tab[0][k] = f.r0[k];
        s.tab[1][k] = f.r06[k];
        s.tab[2][k] = f.sr42[k];
        s.tab[3][k] = f.zab[k];
        s.tab[4][k] = f.alpha[k];
    }
    const T vdw = f.periodic ? (T)f.vdw_cut : (T)(10.0 / 0.52917721092);
    // the queue holds every pair either cutoff takes; a NaN distance is kept
    const double rmax = f.vdw_cut > f.coul_cut ? f.vdw_cut : f.coul_cut;
    const double cut2 = f.periodic ? rmax * rmax * (1.0 + 1e-6) : INFINITY;
    const int chunk = (n + kQSplit - 1) / kQSplit;
    // of a step: eighth and place; of the sums: eighth and component (3: energy)
    const int sp = lane >> 3, comp = lane & 7;
    double *res = s.res[wave];
    QAcc<T> acc;
    int queued = 0, mine = 0;                      // in the wave's queues, and in this lane's eighth
    auto pairs = [&]() {
        // a lane per queued atom, one eighth after the other
        int start = 0, from = 0, q = 0, first = 0;
#pragma unroll
        for (int k = 1; k < kQSplit; ++k) {
            start += __builtin_amdgcn_readlane(mine, 8 * (k - 1));
            first = sp >= k ? start : first;       // of this lane's eighth
            q = lane >= start ? k : q;             // the eighth of this lane's atom
            from = lane >= start ? start : from;
        }
        const bool on = lane < queued;
        const int j = on ? q * chunk + s.queue[wave][q][lane - from] : 0;
        double dd[3] = { xi0 - x[3 * j], xi1 - x[3 * j + 1], xi2 - x[3 * j + 2] };
        qimg(f, dd);
        const T d[3] = { (T)dd[0], (T)dd[1], (T)dd[2] };
        const T r2 = (d[0] * d[0] + d[1] * d[1]) + d[2] * d[2];
        const T r = sqrt(r2);
        T ga[3] = { (T)0, (T)0, (T)0 }, e = (T)0;
        if (!(f.periodic && r > vdw))
            qdisp_rep<T>({ s.tab[0], s.tab[1], s.tab[2], s.tab[3], s.tab[4] }, ei + f.elem[j], c6[j], d, r2, r, (T)1.0, e,
                         ga);
        T ec, gc[3];
        if (qcoulomb<T>(f, qi, f.q[j], d, r2, r, (T)1.0, ec, gc)) {
            e = qadd(e, ec);
            for (int c = 0; c < 3; ++c) ga[c] = qadd(ga[c], gc[c]);
        }
        for (int c = 0; c < 3; ++c) res[67 * c + lane] = (double)ga[c];
        res[67 * 3 + lane] = (double)e;
        qwave_fence();
        if (comp < 4)
            for (int k = 0; k < mine; k += 4) {    // 4 reads at a time; only the additions wait
                const double *v = res + 67 * comp + first + k;
                double t[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) t[u] = v[u];
#pragma unroll
                for (int u = 0; u < 4; ++u) acc.add(k + u < mine ? (T)t[u] : (T)0);    // + 0 changes neither sum
            }
        qwave_fence();
        queued = mine = 0;
    };
    for (int t0 = 0; t0 < chunk; t0 += kQTile / kQSplit) {
        __syncthreads();
        const int jt = (tid >> 5) * chunk + t0 + (tid & 31);
        if (t0 + (tid & 31) < chunk && jt < n) {
            for (int c = 0; c < 3; ++c) s.x[c][tid] = x[3 * jt + c];
            s.mol[tid] = f.mol[jt];
        }
        __syncthreads();
        if (!act) continue;                        // the whole wave
        for (int u0 = 0; u0 < kQTile / kQSplit && t0 + u0 < chunk; u0 += 8) {
            const int jj = t0 + u0 + comp, u = 32 * sp + u0 + comp;
            const bool there = jj < chunk && sp * chunk + jj < n;
            const int uu = there ? u : 0;
            bool in = there && s.mol[uu] != mi;                   // not i's own molecule (nor i)
            double d[3] = { xi0 - s.x[0][uu], xi1 - s.x[1][uu], xi2 - s.x[2][uu] };
            if (f.periodic)                                       // a nearest image in one step; the pair has its own
                for (int c = 0; c < 3; ++c) d[c] = fma(-f.box[c], rint(d[c] * f.ibox[c]), d[c]);
            in = in && !((d[0] * d[0] + d[1] * d[1]) + d[2] * d[2] > cut2);
            const unsigned long long m = __ballot(in);
            if (queued + __popcll(m) > 64) pairs();
            const unsigned eighth = (unsigned)(m >> (8 * sp)) & 0xFFu;
            if (in) s.queue[wave][sp][mine + __popc(eighth & ((1u << comp) - 1u))] = (unsigned short)jj;
            mine += __popc(eighth);
            queued += __popcll(m);
            qwave_fence();
        }
    }
    if (queued > 0) pairs();
    if (act && comp < 3) gpart[sp * stride + 3 * i + comp] = acc.get();
    double ee = act && comp == 3 ? acc.get() : 0.0;
    for (int o = 32; o > 0; o >>= 1) ee += __shfl_xor(ee, o);
    if (lane == 0) s.e[wave] = 0.5 * ee;           // every pair counted from both sides
    __syncthreads();
    if (tid == 0) *epart = ((s.e[0] + s.e[1]) + s.e[2]) + s.e[3];
}

// Every (term, atom) slot of the bonded terms, nci pairs and listed hydrogen
// bonds: the term's gradient on that atom, and its energy at the slot of its
// first atom (block sums in a fixed order).  Slots are contiguous per kind.
__device__ void qslot(const QDev &f, const double *__restrict__ x, int blk, double *sred, double *gslot, double *eslot)
{
    const int sl = blk * kQTile + threadIdx.x;
    double e = 0.0;
    if (sl < f.nslot) {
        double et = 0.0, gv[3] = { 0.0, 0.0, 0.0 };
        int kind = 4;
        while (kind > 0 && sl < f.sbase[kind]) --kind;
        const int roles = kind == 0 ? 2 : kind == 1 ? 3 : kind == 2 ? 4 : kind == 3 ? 2 : 3;
        const int idx = (sl - f.sbase[kind]) / roles, role = (sl - f.sbase[kind]) % roles;
        switch (kind) {
        case kTBond: qbond(f, x, idx, role, et, gv); break;
        case kTAngle: qangle(f, x, idx, role, et, gv); break;
        case kTTors: qtors(f, x, idx, role, et, gv); break;
        case kTNci: qnci(f, x, idx, role, et, gv); break;
        default: qhblist(f, x, idx, role, et, gv); break;
        }
        double *o = gslot + (size_t)sl * 3;
        o[0] = gv[0];
        o[1] = gv[1];
        o[2] = gv[2];
        if (role == 0) e = et;
    }
    for (int o = 32; o > 0; o >>= 1) e = e + __shfl_xor(e, o);
    if ((threadIdx.x & 63) == 0) sred[threadIdx.x >> 6] = e;
    __syncthreads();
    if (threadIdx.x == 0) *eslot = ((sred[0] + sred[1]) + sred[2]) + sred[3];
}

// Intermolecular hydrogen bonds, one wave per acceptor against all donor bonds
// (gradient of the acceptor and energy) or, DON, per donor bond against all
// acceptors (gradients of A and H); butterfly sums, a fixed order.
//
// A tenth of the pairs lies within the 15 bohr of the term, so a few lanes of
// each 64 had a bond and the wave went through all of it for them, once per 64
// partners.  Now those that count are queued and evaluated together, and the
// blocks come first in the grid, as the waves with the longest chains: 15 of
// the 130 us of a force call of 1125 atoms x 16 beads.  Two or four acceptors
// to a wave fill the evaluations better, but the longer chains cost more (7
// and 23 us).
//
// The terms of a batch go to LDS, and the lane that the partner's number names
// (mod 64) adds its own in their order: the sums of lanes that stride over the
// partners, whatever the batches were (3 us of the call).
template <bool DON>
__device__ void qhb(const QDev &f, const double *__restrict__ x, int own, QTile &s, double *gout, double *eout)
{
    const int lane = threadIdx.x & 63, n2 = DON ? f.nacc : f.ndon;
    if (own >= (DON ? f.ndon : f.nacc)) return;
    int *queue = reinterpret_cast<int *>(s.queue[threadIdx.x >> 6]);     // 63 + 64 at most
    static_assert(sizeof s.queue[0] >= 128 * sizeof(int), "");
    double *res = s.res[threadIdx.x >> 6];
    double sum[6] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
    int count = 0;
    // sum[at..at + nv - 1] += v of the terms whose partner is this lane's, places `mine` of the batch
    auto own_terms = [&](unsigned long long mine, int at, int nv, const double *v) {
        for (int c = 0; c < nv; ++c) res[4 * lane + c] = v[c];
        qwave_fence();
        for (; mine; mine &= mine - 1) {
            const double *r = res + 4 * __builtin_ctzll(mine);
            for (int c = 0; c < nv; ++c) sum[at + c] = sum[at + c] + r[c];
        }
        qwave_fence();
    };
    for (int o0 = 0; o0 < n2; o0 += 64) {
        const int o = o0 + lane;
        const bool in = o < n2 && qhbnear(f, x, DON ? own : o, DON ? o : own);
        const unsigned long long m = __ballot(in);
        if (in) queue[count + __popcll(m & ((1ull << lane) - 1ull))] = o;
        count += __popcll(m);
        qwave_fence();
        const bool last = o0 + 64 >= n2;
        while (count >= 64 || (last && count > 0)) {
            const int k = min(count, 64);
            const int other = queue[lane < k ? lane : 0], rest = queue[64 + lane];
            const int dn = DON ? own : other, A = f.don[2 * dn], H = f.don[2 * dn + 1];
            const int j = f.acc[DON ? other : own];
            double gj[3], ga[3], gh[3];
            const double e = qeabhag<DON ? kHbDonor : kHbAcceptor>(f, x, j, A, H, f.hbc[j], f.hbc[A], gj, ga, gh);
            unsigned long long mine = 0;
            for (int t = 0; t < k; ++t)
                mine |= (unsigned long long)((__builtin_amdgcn_readlane(other, t) & 63) == lane) << t;
            if (DON) {
                own_terms(mine, 0, 3, ga);
                own_terms(mine, 3, 3, gh);
            } else {
                const double v[4] = { gj[0], gj[1], gj[2], e };
                own_terms(mine, 0, 4, v);
            }
            count -= k;
            if (lane < count) queue[lane] = rest;
            qwave_fence();
        }
    }
    for (int c = 0; c < (DON ? 6 : 4); ++c)
        for (int t = 32; t > 0; t >>= 1) sum[c] = sum[c] + __shfl_xor(sum[c], t);
    if (lane != 0) return;
    for (int c = 0; c < (DON ? 6 : 3); ++c) gout[(size_t)(DON ? 6 : 3) * own + c] = sum[c];
    if (!DON) eout[own] = sum[3];
}

// Blocks of one bead (blockIdx.y): in this order nacc and ndon of the hydrogen
// bonds, nslot of the slots, ninter of the intermolecular pairs.  One launch:
// the hydrogen-bond and slot blocks, 17 to 25 us each as kernels of their own
// that fill a part of the chip, run beside the pairs.
struct QBlocks {
    int ninter, nacc, ndon, nslot;
};

// Built without machine-level loop-invariant code motion (see the Makefile):
// with it the constants of exp and erfc were held in 128 registers across the
// loops and others spilled inside them (151 us a call, 132 without).  Five
// waves per SIMD, the most that the LDS allows, cost 52 bytes of spills in the
// slots: an FP64 call of 1125 atoms x 16 beads takes 148 us, 161 at four.
template <typename T>
__global__ __launch_bounds__(kQTile) __attribute__((amdgpu_waves_per_eu(5))) void qm_terms_kernel(
    QDev f, QBlocks nb, const double *__restrict__ xall, double *gpart, double *epart, double *gacc, double *eacc,
    double *gdon, double *gslot, double *eslot)
{
    __shared__ QTile s;
    const int b = blockIdx.y, wave = threadIdx.x >> 6;
    const double *x = xall + (size_t)b * f.n * 3;
    int k = blockIdx.x;
    if (k < nb.nacc) {
        qhb<false>(f, x, k * kQWaves + wave, s, gacc + (size_t)b * f.nacc * 3, eacc + (size_t)b * f.nacc);
        return;
    }
    k -= nb.nacc;
    if (k < nb.ndon) {
        qhb<true>(f, x, k * kQWaves + wave, s, gdon + (size_t)b * f.ndon * 6, nullptr);
        return;
    }
    k -= nb.ndon;
    if (k < nb.nslot) {
        qslot(f, x, k, s.e, gslot + (size_t)b * f.nslot * 3, eslot + (size_t)b * nb.nslot + k);
        return;
    }
    k -= nb.nslot;
    qinter<T>(f, x, k, s, gpart + (size_t)b * f.n * 3, (size_t)gridDim.y * f.n * 3, epart + (size_t)b * nb.ninter + k);
}

// Four lanes per (bead, atom): its term slots and hydrogen-bond parts, every
// fourth of the list loaded by a lane (the loads of a list entry wait for its
// code, so one lane's list was a chain of some twenty memory latencies: 16 us,
// now 9.0) and added by all four in the list's order, then the eighths of
// the intermolecular sum; the acceptors' energies.
__global__ __launch_bounds__(256) void qm_gather_kernel(QDev f, const double *gslot, const double *gpart,
                                                        const double *gacc, const double *eacc, const double *gdon,
                                                        double *gout, double *egather)
{
    __shared__ double sred[4];
    const int i = blockIdx.x * 64 + (threadIdx.x >> 2), sub = threadIdx.x & 3, b = blockIdx.y;
    const bool act = i < f.n;
    double g[3] = { 0.0, 0.0, 0.0 }, e = 0.0;
    if (act) {
        const int end = f.rptr[i + 1];
        for (int k0 = f.rptr[i]; k0 < end; k0 += 4) {          // the same trips on all four lanes
            double v[3] = { 0.0, 0.0, 0.0 };
            if (k0 + sub < end) {
                const int code = f.rcode[k0 + sub];
                const int kind = code >> 28, payload = code & 0x0FFFFFFF;
                const double *src;
                if (kind == kTHbAcc) {
                    src = gacc + ((size_t)b * f.nacc + payload) * 3;
                    e = e + eacc[(size_t)b * f.nacc + payload];
                } else if (kind == kTHbDon) {
                    const int role = payload >> 26, dn = payload & 0x03FFFFFF;
                    src = gdon + ((size_t)b * f.ndon + dn) * 6 + (role == 1 ? 0 : 3);
                } else {
                    src = gslot + ((size_t)b * f.nslot + payload) * 3;
                }
                for (int c = 0; c < 3; ++c) v[c] = src[c];
            }
            for (int c = 0; c < 3; ++c)                        // past the end: + 0
                g[c] = (((g[c] + quad::bcast<0>(v[c])) + quad::bcast<1>(v[c])) + quad::bcast<2>(v[c])) +
                       quad::bcast<3>(v[c]);
        }
        if (gout && sub < 3) {
            double own = sub == 0 ? g[0] : sub == 1 ? g[1] : g[2];
            const size_t o = ((size_t)b * f.n + i) * 3 + sub, stride = (size_t)gridDim.y * f.n * 3;
            if (f.inter)
#pragma unroll
                for (int s = 0; s < kQSplit; ++s) own = own + gpart[s * stride + o];
            gout[o] = own;
        }
    }
    for (int o = 32; o > 0; o >>= 1) e = e + __shfl_xor(e, o);
    if ((threadIdx.x & 63) == 0) sred[threadIdx.x >> 6] = e;
    __syncthreads();
    if (threadIdx.x == 0) egather[(size_t)b * gridDim.x + blockIdx.x] = ((sred[0] + sred[1]) + sred[2]) + sred[3];
}

// One wave per bead: lanes over each list of block sums, then a butterfly (a
// fixed order).
__global__ __launch_bounds__(64) void qm_reduce_kernel(const double *eslot, int nsl, const double *epart, int ninter,
                                                       const double *egather, int ngather, double *e)
{
    const int b = blockIdx.x, lane = threadIdx.x;
    double s = 0.0;
    for (int k = lane; k < nsl; k += 64) s = s + eslot[(size_t)b * nsl + k];
    for (int k = lane; k < ngather; k += 64) s = s + egather[(size_t)b * ngather + k];
    for (int k = lane; k < ninter; k += 64) s = s + epart[(size_t)b * ninter + k];
    for (int o = 32; o > 0; o >>= 1) s = s + __shfl_xor(s, o);
    if (lane == 0) e[b] = s;
}

template <typename Tv>
int upload(QmdffDev *q, const std::vector<Tv> &v, const Tv **out)
{
    *out = nullptr;
    if (v.empty()) return CAM_OK;
    void *p = nullptr;
    CAM_HIP(hipMalloc(&p, v.size() * sizeof(Tv)));
    q->allocs.push_back(p);
    CAM_HIP(hipMemcpy(p, v.data(), v.size() * sizeof(Tv), hipMemcpyHostToDevice));
    *out = static_cast<const Tv *>(p);
    return CAM_OK;
}

}  // namespace

void qmdff_free(QmdffDev *q)
{
    if (!q) return;
    for (void *p : q->allocs) (void)hipFree(p);
    double *bufs[] = { q->gpart, q->epart, q->gacc, q->eacc, q->gdon, q->gslot, q->eslot };
    for (double *p : bufs)
        if (p) (void)hipFree(p);
    delete q;
}

int qmdff_natoms(const QmdffDev *q) { return q->d.n; }

int qmdff_build(const cam_qmdff_desc *in, QmdffDev **out)
{
    *out = nullptr;
    const int n = in->natoms;
    std::unique_ptr<QmdffDev> q(new QmdffDev());
    QDev &d = q->d;
    d.n = n;
    d.nbond = in->nbond;
    d.nangl = in->nangl;
    d.ntors = in->ntors;
    d.nnci = in->nnci;
    d.nhb = in->nhb;
    d.periodic = in->periodic != 0;
    d.zahn = in->zahn != 0;
    for (int c = 0; c < 3; ++c) {
        d.box[c] = in->box[c];
        d.box2[c] = 0.5 * in->box[c];
        d.ibox[c] = 1.0 / in->box[c];
    }
    d.coul_cut = in->coul_cut;
    d.vdw_cut = in->vdw_cut;
    d.cut_low = in->cut_low;
    d.zahn_a = in->zahn_a;
    d.zahn_par = in->zahn_par;
    for (int k = 0; k < 6; ++k) {
        d.eps1[k] = in->eps1[k];
        d.eps2[k] = in->eps2[k];
    }
    // element slots
    std::vector<int> zs;
    for (int i = 0; i < n; ++i)
        if (std::find(zs.begin(), zs.end(), in->at[i]) == zs.end()) zs.push_back(in->at[i]);
    CAM_CHECK_ARG((int)zs.size() <= kQMaxElem, "more than %d elements", kQMaxElem);
    const int ne = (int)zs.size();
    d.ne = ne;
    std::vector<int> elem(n), mol(n);
    std::vector<double> scal(n), hbc(n);
    for (int i = 0; i < n; ++i) {
        elem[i] = (int)(std::find(zs.begin(), zs.end(), in->at[i]) - zs.begin());
        mol[i] = (int)in->molnum[i];
        scal[i] = in->scalehb[in->at[i] - 1];
        const double eq = std::exp(-10.0 * in->q[i]);
        hbc[i] = eq / (eq + 5.0) * scal[i];       // hbpara(10, 5, q) * scalehb (src/ff_hb.f90:256-259)
    }
    std::vector<double> r0(ne * ne), r06(ne * ne), sr42(ne * ne), zab(ne * ne), alpha(ne * ne), rad(ne);
    for (int a = 0; a < ne; ++a) {
        rad[a] = in->rad[zs[a] - 1];
        for (int b = 0; b < ne; ++b) {
            const size_t fz = (size_t)(zs[b] - 1) * 94 + (zs[a] - 1);   // Fortran (z_a, z_b)
            r0[a * ne + b] = in->r094[fz];
            r06[a * ne + b] = std::pow(in->r094[fz], 6);
            sr42[a * ne + b] = in->sr42[fz];
            zab[a * ne + b] = in->zab[fz];
            alpha[a * ne + b] = in->r0ab[fz];
        }
    }
    // 0-based term lists
    auto zero_based = [](const int32_t *p, size_t cnt) {
        std::vector<int> v(cnt);
        for (size_t k = 0; k < cnt; ++k) v[k] = p[k] - 1;
        return v;
    };
    std::vector<int> bond = zero_based(in->bond, 2 * (size_t)in->nbond);
    std::vector<int> angl = zero_based(in->angl, 3 * (size_t)in->nangl);
    std::vector<int> tors(6 * (size_t)in->ntors), nci(3 * (size_t)in->nnci), hb = zero_based(in->hb, 3 * (size_t)in->nhb);
    for (int m = 0; m < in->ntors; ++m)
        for (int c = 0; c < 6; ++c) tors[6 * m + c] = c < 4 ? in->tors[6 * m + c] - 1 : in->tors[6 * m + c];
    for (int m = 0; m < in->nnci; ++m) {
        nci[3 * m] = in->nci[3 * m] - 1;
        nci[3 * m + 1] = in->nci[3 * m + 1] - 1;
        nci[3 * m + 2] = in->nci[3 * m + 2];
    }
    int nm = 0;
    bool multi = false;
    for (int i = 0; i < n; ++i) nm = std::max(nm, mol[i]);
    multi = nm > 1;                                   // nmols = maxval(molnum) (src/rdsolvff.f90:76)
    d.inter = multi;
    // intermolecular hydrogen bonds: donor bonds and acceptor atoms
    auto acceptor_z = [](int z) { return z == 7 || z == 8 || z == 9 || z == 16 || z == 17; };
    std::vector<int> don, acc;
    std::vector<double> don_lim, acc_lim;
    const float k13 = 1.3f, kbohr = 0.52917726f;
    if (multi) {
        for (int m = 0; m < in->nbond; ++m) {
            const int i1 = bond[2 * m], i2 = bond[2 * m + 1];
            int aH = -1, aA = -1;
            if (in->at[i1] == 1 && acceptor_z(in->at[i2])) {
                aH = i1;
                aA = i2;
            }
            if (in->at[i2] == 1 && acceptor_z(in->at[i1])) {
                aH = i2;
                aA = i1;
            }
            if (aH < 0) continue;
            don.push_back(aA);
            don.push_back(aH);
            don_lim.push_back((double)k13 * (in->rad[in->at[aA] - 1] + in->rad[0]) / (double)kbohr);
        }
        for (int j = 0; j < n; ++j)
            if (scal[j] > 0.0) {
                acc.push_back(j);
                acc_lim.push_back((double)k13 * (in->rad[in->at[j] - 1] + in->rad[0]) / (double)kbohr);
            }
    }
    if (don_lim.empty() || acc.empty()) {          // no pair to evaluate
        don.clear();
        don_lim.clear();
        acc.clear();
        acc_lim.clear();
    }
    d.ndon = (int)don_lim.size();
    d.nacc = (int)acc.size();
    // Term slots: one per (term, atom of the term), contiguous per kind;
    // each atom lists its slots (kind << 28 | slot) and its hydrogen-bond
    // parts (kind << 28 | role << 26 | index) in the reference's term order.
    const int64_t nslot64 = 2 * (int64_t)in->nbond + 3 * (int64_t)in->nangl + 4 * (int64_t)in->ntors +
                            2 * (int64_t)in->nnci + 3 * (int64_t)in->nhb;
    if (nslot64 >= (int64_t)1 << 28) return CAM_ERR_ARG;
    d.sbase[0] = 0;
    d.sbase[1] = 2 * in->nbond;
    d.sbase[2] = d.sbase[1] + 3 * in->nangl;
    d.sbase[3] = d.sbase[2] + 4 * in->ntors;
    d.sbase[4] = d.sbase[3] + 2 * in->nnci;
    d.nslot = (int)nslot64;
    std::vector<std::vector<int>> roles(n);
    auto code = [](int kind, int role, int idx) { return kind << 28 | role << 26 | idx; };
    auto slot = [&](int kind, int nroles, int m, int r) { return kind << 28 | (d.sbase[kind] + nroles * m + r); };
    for (int m = 0; m < in->nbond; ++m)
        for (int r = 0; r < 2; ++r) roles[bond[2 * m + r]].push_back(slot(kTBond, 2, m, r));
    for (int m = 0; m < in->nangl; ++m)
        for (int r = 0; r < 3; ++r) roles[angl[3 * m + r]].push_back(slot(kTAngle, 3, m, r));
    for (int m = 0; m < in->ntors; ++m)
        for (int r = 0; r < 4; ++r) roles[tors[6 * m + r]].push_back(slot(kTTors, 4, m, r));
    for (int m = 0; m < in->nnci; ++m)
        for (int r = 0; r < 2; ++r) roles[nci[3 * m + r]].push_back(slot(kTNci, 2, m, r));
    for (int m = 0; m < in->nhb; ++m)
        for (int r = 0; r < 3; ++r) roles[hb[3 * m + r]].push_back(slot(kTHbList, 3, m, r));
    for (int a = 0; a < d.nacc; ++a) roles[acc[a]].push_back(code(kTHbAcc, 0, a));
    for (int dn = 0; dn < d.ndon; ++dn) {
        roles[don[2 * dn]].push_back(code(kTHbDon, 1, dn));
        roles[don[2 * dn + 1]].push_back(code(kTHbDon, 2, dn));
    }
    std::vector<int> rptr(n + 1, 0), rcode;
    for (int i = 0; i < n; ++i) {
        rptr[i + 1] = rptr[i] + (int)roles[i].size();
        rcode.insert(rcode.end(), roles[i].begin(), roles[i].end());
    }
    std::vector<double> c6((size_t)n * n);          // transposed: a wave reads along the row of its atom
    for (int i = 0; i < n; ++i)
        for (int j = 0; j < n; ++j) c6[(size_t)i * n + j] = in->c6xy[(size_t)j * n + i];
    std::vector<double> qv(in->q, in->q + n);
    std::vector<double> vbond(in->vbond, in->vbond + 3 * (size_t)in->nbond);
    std::vector<double> vangl(in->vangl, in->vangl + 2 * (size_t)in->nangl);
    std::vector<double> vtors(in->vtors, in->vtors + 14 * (size_t)in->ntors);
    std::vector<double> vhb(in->vhb, in->vhb + 2 * (size_t)in->nhb);
    QmdffDev *qq = q.get();
    int rc = CAM_OK;
#define CAM_UP(vec, field)                                   \
    if (rc == CAM_OK) rc = upload(qq, vec, &d.field);
    CAM_UP(elem, elem) CAM_UP(mol, mol) CAM_UP(qv, q) CAM_UP(c6, c6) CAM_UP(r0, r0) CAM_UP(r06, r06)
    CAM_UP(sr42, sr42) CAM_UP(zab, zab) CAM_UP(alpha, alpha) CAM_UP(rad, rad) CAM_UP(bond, bond)
    CAM_UP(angl, angl) CAM_UP(tors, tors) CAM_UP(nci, nci) CAM_UP(hb, hb) CAM_UP(vbond, vbond)
    CAM_UP(vangl, vangl) CAM_UP(vtors, vtors) CAM_UP(vhb, vhb) CAM_UP(rptr, rptr) CAM_UP(rcode, rcode)
    CAM_UP(don, don) CAM_UP(acc, acc) CAM_UP(don_lim, don_lim) CAM_UP(acc_lim, acc_lim) CAM_UP(hbc, hbc)
    CAM_UP(scal, scal)
#undef CAM_UP
    if (rc != CAM_OK) return rc;
    *out = q.release();
    return CAM_OK;
}

namespace {
int qmdff_ensure(QmdffDev *q, int nbeads)
{
    if (nbeads <= q->cap_beads) return CAM_OK;
    double **bufs[] = { &q->gpart, &q->epart, &q->gacc, &q->eacc, &q->gdon, &q->gslot, &q->eslot };
    for (double **p : bufs)
        if (*p) {
            CAM_HIP(hipFree(*p));
            *p = nullptr;
        }
    const QDev &d = q->d;
    const int nbx = (d.n + kQWaves - 1) / kQWaves;
    const int ngx = (d.n + 63) / 64;
    CAM_HIP(hipMalloc(&q->gpart, (size_t)kQSplit * nbeads * d.n * 3 * sizeof(double)));
    CAM_HIP(hipMalloc(&q->epart, (size_t)nbeads * (nbx + ngx) * sizeof(double)));
    CAM_HIP(hipMalloc(&q->gacc, ((size_t)std::max(1, d.nacc) * nbeads * 4) * sizeof(double)));
    CAM_HIP(hipMalloc(&q->eacc, ((size_t)std::max(1, d.nacc) * nbeads) * sizeof(double)));
    CAM_HIP(hipMalloc(&q->gdon, ((size_t)std::max(1, d.ndon) * nbeads * 6) * sizeof(double)));
    CAM_HIP(hipMalloc(&q->gslot, ((size_t)std::max(1, d.nslot) * nbeads * 3) * sizeof(double)));
    CAM_HIP(hipMalloc(&q->eslot, ((size_t)std::max(1, (d.nslot + 255) / 256) * nbeads) * sizeof(double)));
    q->cap_beads = nbeads;
    return CAM_OK;
}
}  // namespace

template <typename T>
int qmdff_launch(QmdffDev *q, const double *x, int nbeads, double *e, double *g, hipStream_t s)
{
    int rc = qmdff_ensure(q, nbeads);
    if (rc != CAM_OK) return rc;
    const QDev &d = q->d;
    const int nbx = (d.n + kQWaves - 1) / kQWaves, nsx = (d.nslot + kQTile - 1) / kQTile;
    const int ngx = (d.n + 63) / 64;
    double *egather = q->epart + (size_t)nbeads * nbx;
    const bool hb = d.nacc > 0 && d.ndon > 0;
    const QBlocks nb{ d.inter ? nbx : 0, hb ? (d.nacc + kQWaves - 1) / kQWaves : 0,
                      hb ? (d.ndon + kQWaves - 1) / kQWaves : 0, nsx };
    const int nblk = nb.ninter + nb.nacc + nb.ndon + nb.nslot;
    if (nblk > 0) {
        hipLaunchKernelGGL(qm_terms_kernel<T>, dim3(nblk, nbeads), dim3(kQTile), 0, s, d, nb, x, q->gpart, q->epart,
                           q->gacc, q->eacc, q->gdon, q->gslot, q->eslot);
        CAM_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(qm_gather_kernel, dim3(ngx, nbeads), dim3(256), 0, s, d, q->gslot, q->gpart,
                       q->gacc, q->eacc, q->gdon, g, egather);
    CAM_LAUNCH_CHECK();
    hipLaunchKernelGGL(qm_reduce_kernel, dim3(nbeads), dim3(64), 0, s, q->eslot, nsx, q->epart,
                       nb.ninter, egather, ngx, e);
    CAM_LAUNCH_CHECK();
    return CAM_OK;
}

template int qmdff_launch<double>(QmdffDev *, const double *, int, double *, double *, hipStream_t);
template int qmdff_launch<float>(QmdffDev *, const double *, int, double *, double *, hipStream_t);

bool qmdff_box(const QmdffDev *q, double box[3])
{
    for (int c = 0; c < 3; ++c) box[c] = q->d.box[c];
    return q->d.periodic != 0;
}

}  // namespace cam
