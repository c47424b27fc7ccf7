// Per-pair and per-bond force terms shared by the brute-force and cell-list force kernels,
// so both evaluate every pair with the same instructions.
//
//   Debye-Hueckel  F = (gamma/eps_r) Q_i Q_j (1 + kappa r) e^{-kappa r} / r^2   r <= cutoff_c
//                  (electro.c:36-78)
//   Lennard-Jones  F = alpha eps_ij 6 (s6 (2 s6 - lj6)) / r, s6 = (sigma_ij/r)^6,
//                  sigma_ij = R_i + R_j, eps_ij = sqrt(eps_i eps_j),
//                  r <= cutoff_lj (or 1.122462 sigma_ij when cutoff_lj <= 0)   (LJ.c:37-99)
//   overlap flag   sigma_ij > r (LJ_force / LJ_force_check, LJ.c:58, :101-107)
//   bonds          F = H (r0 - r) / (1 - r^2/rmax^2)                           (bond.c:43-85)
// The branch structure is force_single's (calc_func.c:370-409).
#pragma once

#include "bdh_common.hpp"
#include "bdh_kernels.hpp"

namespace bdh {

struct PairAcc {
    double fx, fy, fz;  // force on the row bead
    double e_lj, e_c;   // energies seen from the row bead (each pair is seen twice)
    int rep;            // bit 0: overlap, bit 1: overstretched bond
};

// 1 / r and, in FP64, 1 / r again: equal for T = double; from T = float one Newton step, so
// that the force's direction keeps the FP64 separation's precision.
__device__ __forceinline__ double wide_inverse(double, double inv) { return inv; }
__device__ __forceinline__ double wide_inverse(float r, float inv)
{
    const double y = (double)inv;
    return fma(y, fma(-(double)r, y, 1.0), y);
}

// a / r with inv = 1 / r at hand to an ulp or two: the product and one step with its residual, as
// good as a division to a few hundredths of an ulp at a fraction of its instructions.  A result that
// is not finite is the product's.
template <typename T>
__device__ __forceinline__ T quotient(T a, T r, T inv)
{
    const T q = a * inv, c = fma(fma(-q, r, a), inv, q);
    return isfinite(c) ? c : q;
}

// Pair (i, j) seen from i: d = r_j - r_i (minimum image applied), r2d = |d|^2 from pair_r2.
// One root and one division a pair, and quotients by its result (five divisions in the formulas
// as written); the cutoffs and the overlap compare with the root itself.  Energies only where asked
// for.  rms error of isolated charged pairs' forces in FP64 1.9e-16 and in FP32 8.4e-8, as with the
// divisions; with products by the reciprocal instead 2.8e-16 and 1.2e-7.
template <typename T>
__device__ __forceinline__ void pair_term(double dx, double dy, double dz, double r2d, double qi,
                                          double qj, double2 lji, double2 ljj, bool conn,
                                          const ForceParams& fp, PairAcc& a, bool energy = true)
{
    const T gam = (T)fp.gam, kap = (T)fp.kappa_c, alj = (T)fp.alpha_lj, lj6 = (T)fp.lj_6_term;
    const T r2 = (T)r2d;
    const T r = sqrt(r2);
    const T inv = (T)1 / r;
    const T sig = (T)(lji.x + ljj.x);
    T F = 0;
    int ov = 0;
    if (fp.elec && r <= (T)fp.cutoff_c && (!conn || fp.bond_c_scale != 0.0)) {
        const T ex = exp(-kap * r);
        T f = quotient(gam * (T)qi * (T)qj * ((T)1 + kap * r) * ex, r2, inv * inv);
        if (conn) f *= (T)fp.bond_c_scale;
        F += f;
        if (energy) {
            T en = quotient(gam * (T)qi * (T)qj * ex, r, inv);
            if (conn) en *= (T)fp.bond_c_scale;
            a.e_c += (double)en;
        }
    }
    const T lj_cut = fp.cutoff_lj > 0.0 ? (T)fp.cutoff_lj : (T)1.122462f * sig;
    if (fp.alpha_lj != 0.0 && r <= lj_cut) {
        if (!conn || fp.bond_lj_scale != 0.0) {
            // equal depths: the root of a square is exact
            const T eps = (T)(lji.y == ljj.y ? fabs(lji.y) : sqrt(lji.y * ljj.y));
            T s6 = quotient(sig, r, inv);
            s6 *= s6;
            s6 *= s6 * s6;
            T f = quotient(alj * eps * (T)6 * (s6 * ((T)2 * s6 - lj6)), r, inv);
            if (conn) f *= (T)fp.bond_lj_scale;
            F += f;
            if (energy) {
                T en = alj * eps * (s6 * (s6 - lj6));
                if (conn) en *= (T)fp.bond_lj_scale;
                a.e_lj += (double)en;
            }
            ov = (sig > r) || !isfinite(f);
        } else {
            ov = sig * sig > r2;
        }
    } else {
        ov = sig * sig > r2;
    }
    a.rep |= ov;
    // force on i: -e_ij F with e_ij = (r_j - r_i)/r
    const double s = quotient((double)F, (double)r, wide_inverse(r, inv));
    a.fx -= dx * s;
    a.fy -= dy * s;
    a.fz -= dz * s;
}

__device__ __forceinline__ bool bonded(const Topology& topo, int nb0, int nb1, int j)
{
    bool conn = false;
    for (int b = nb0; b < nb1; ++b) conn |= (topo.conn[b] == j);
    return conn;
}

// Every stride-th bond of bead i from the first-th (both ends carry each bond); returns, when
// energies are asked for, the bond energy seen from i.
__device__ __forceinline__ double bond_terms(const double4* __restrict__ pos, int i, double4 pi,
                                             const Topology& topo, const ForceParams& fp,
                                             PairAcc& a, bool energy, int first = 0, int stride = 1)
{
    double e_b = 0.0;
    const int end = topo.bond_off[i + 1];
    for (int b = topo.bond_off[i] + first; b < end; b += stride) {
        const int p = topo.bond_p[b];
        const double r0 = topo.bond_parm[3 * b], rmax = topo.bond_parm[3 * b + 1];
        const double H = topo.bond_parm[3 * b + 2];
        double dx = pos[p].x - pi.x, dy = pos[p].y - pi.y, dz = pos[p].z - pi.z;
        const double r2 = pair_r2(dx, dy, dz, fp.pbc, fp.box);
        const double r = sqrt(r2);
        if (!(r < rmax)) a.rep |= 2;  // overstretched bond: fatal in the reference
        const double Ff = H * (r0 - r) / (1.0 - r2 / (rmax * rmax));
        const double s = Ff / r;
        a.fx -= s * dx;
        a.fy -= s * dy;
        a.fz -= s * dz;
        if (energy)
            e_b += -0.5 * H * (rmax * rmax * log((rmax * rmax - r2) / (rmax * rmax - r0 * r0)) +
                               r0 * rmax * log((rmax + r) * (rmax - r0) / ((rmax - r) * (rmax + r0))));
    }
    return e_b;
}

}  // namespace bdh
