// Ewald-summed RPY blocks on the device: Beenakker (src/diff_alg/diff_tensor.c:265-422)
// and Smith (:102-263).
//
// alpha = sqrt(pi)/L (forced by init_tensor, diff_tensor.c:551-554); real and reciprocal
// lattices share the sphere h^2 + f^2 + g^2 <= R^2 (ewald_real == ewald_recip,
// src/input.c:402-409), around the pair's separation as the wrapped positions give it (no
// minimum image).  An extension beyond the reference (bdh_set_ewald_split) scales alpha,
// gives the real and reciprocal sums spheres of their own radii (and the real-space images
// a distance cutoff, bdh_set_ewald_cutoff) and centres the image sum on the minimum-image
// separation, so the omitted images of every pair lie at least (sqrt(R_real^2 + 1) -
// sqrt(3)/2) L away, and forms the wave vectors k = 2 pi (h, f, g) / L of the box (the
// reference's k = 2 pi (h, f, g) is in box units against alpha and sigma in A, so its
// reciprocal terms underflow to zero).  The infinite sums do not depend on alpha or on the
// image chosen as the centre (the reciprocal phases are periodic in the separation); the
// truncated ones do.  The lattice vectors and every pair-independent factor of the
// reciprocal term are tabulated once on the host in FP64 (with the reference's float pi;
// the extension's with the double pi):
//   G_k = 6 pi (1 + (k^2/4a^2)(1 + k^2/2a^2)) exp(-k^2/4a^2) / k^2,  Rk = k^2 / 3,
//   k = 2 pi (h, f, g)  (reference),  k = 2 pi (h, f, g) / L  (extension)
// so a pair's reciprocal sum is sum_k (1 - sigma^2 Rk) G_k cos(2 pi v.hfg) (I - e_k e_k^T),
// with v = r / L.  The vectors that differ only in the signs of h, f and g carry the same factors,
// and their cosines add up to products of per-axis cosines and sines, so the sum runs over the
// octant h, f, g >= 0 (recip_sum: 28 classes where the half sphere of radius 3 has 61 vectors).
// The reciprocal and self sums run in FP64 in both precisions; the real-space image sum runs
// in T.
#pragma once

#include <hip/hip_runtime.h>

#include "bdh_common.hpp"

namespace bdh {

constexpr int EW_MAXV = 98;   // classes h, f, g >= 0 with |hfg| <= 5 (but 0)

enum EwaldMethod { EW_SMITH = 0, EW_BEENAKKER = 1 };

struct EwaldTables {
    int RR_real;             // real-space images with h^2 + f^2 + g^2 <= RR_real
    int min_image;           // image sum around the minimum-image separation (extension)
    double rc2;              // extension: real-space images within this squared distance only
    int RR_recip;            // reciprocal vectors with |(h, f, g)|^2 <= RR_recip
    int nrecip;              // classes in c_recip (0: the sum vanishes)
    int method;              // EwaldMethod
    double box, inv_L, alpha, alpha2, alpha3, inv_alpha2;
    double phase;            // 2 pi_f / (pi L): the phase of wave number 1 in half turns per A
    double self_a, self_b;   // Beenakker self term: -6 alpha/sqrt(pi), 40 alpha^3/(3 sqrt(pi))
    double preO;             // Smith: 0.75 / L
};

extern __constant__ EwaldTables c_ew;

// One class of reciprocal vectors (+-h, +-f, +-g), h then f then g ascending over the octant: the
// sum over its members of cos(2 pi v.hfg) (u I + w e e^T) with u = u0 + sigma^2 u1, w = w0 +
// sigma^2 w1, all factors but the phases tabulated: m = the number of members (1, 2, 4 or 8)
//   u, w        m u, m w
//   e[0..2]     e_x^2, e_y^2, e_z^2
//   e[3..5]     e_x e_y, e_x e_z, e_y e_z
struct RecipClass {
    double u0, u1, w0, w1;
    double e[6];
};
extern __constant__ RecipClass c_recip[EW_MAXV];

// Upload the tables of one method for box edge L, lattice radius R and (Smith) the
// splitting parameter alpha in units of 1/L; returns the count of reciprocal classes.  Beenakker with
// alpha_scale > 0 (the extension): alpha = alpha_scale sqrt(pi) / L, spheres of radius
// R_real (images) and R_recip (reciprocal vectors) instead of R, minimum-image centres, and
// with r_cut > 0 only the images within r_cut (A) of the pair.
int ewald_upload(double box, int R, int method, double alpha, double alpha_scale = 0.0, int R_real = -1,
                 int R_recip = -1, double r_cut = 0.0);

struct Blk6 {
    double xx, yy, zz, xy, xz, yz;
};

// (re, im) *= (c + i s)
__device__ __forceinline__ void cmul_step(double& re, double& im, double c, double s)
{
    const double r = re * c - im * s;
    im = re * s + im * c;
    re = r;
}

// Coefficients of the FP64 image functions below, read through the scalar cache: as literals they
// are kept in vector registers across the image loop and cost a wavefront per SIMD.
struct ImageCoef {
    double erfcx[23];   // erfcx_image
    double expo[14];    // exp_image: 1 / k!
};
extern __constant__ ImageCoef c_img;
constexpr ImageCoef IMAGE_COEF = {
    {
        1.2375126308378275, -0.14024059858554525, 0.0035854154854790257,
        0.08227673848999506, -0.10880393014244462, 0.09230432116428125,
        -0.05869339857664934, 0.02836227737211114, -0.009746579683265262,
        0.0017556261651970652, 0.000293714378044958, -0.00029015535246077655,
        5.164652974177416e-05, 2.2387565714911816e-05, -1.1438048033346894e-05,
        -9.792625707303523e-07, 1.7419821586224816e-06, -5.084465378687302e-08,
        -2.4857126248016745e-07, 1.879082322370048e-08, 3.197926671666804e-08,
        -1.9551358868985616e-09, -2.623107347133476e-09},
    {1.0, 1.0, 1.0 / 2, 1.0 / 6, 1.0 / 24, 1.0 / 120, 1.0 / 720, 1.0 / 5040, 1.0 / 40320, 1.0 / 362880,
     1.0 / 3628800, 1.0 / 39916800, 1.0 / 479001600, 1.0 / 6227020800.0}};

// exp(-u) for the squared distance r2 with u = alpha^2 r2.  FP32: the hardware's base-2 exponential
// of the product with -alpha^2 log2(e) in two parts (nl, nl_lo), so the argument is rounded once.
// FP64 (nl = -alpha^2): 2^n exp(r) with |r| <= ln(2)/2, n ln(2) taken off in two parts (Cody and
// Waite, Software Manual for the Elementary Functions, 1980), and the Taylor polynomial of degree
// 13, even and odd powers in chains of their own; arguments of any size (the result goes to zero).
__device__ __forceinline__ double exp_image(double r2, double nl, double)
{
    const double x = nl * r2;
    const double n = __builtin_rint(x * 1.4426950408889634074);
    const double r = __builtin_fma(n, -1.90821492927058770002e-10, __builtin_fma(n, -6.93147180369123816490e-01, x));
    const double q = r * r;
    const double* c = c_img.expo;
    double e = c[12], o = c[13];
#pragma unroll
    for (int k = 10; k >= 0; k -= 2) {
        e = __builtin_fma(e, q, c[k]);
        o = __builtin_fma(o, q, c[k + 1]);
    }
    return __builtin_amdgcn_ldexp(__builtin_fma(o, r, e), (int)__builtin_fmax(n, -4000.0));
}
__device__ __forceinline__ float exp_image(float r2, float nl, float nl_lo)
{
    return __builtin_amdgcn_exp2f(__builtin_fmaf(r2, nl, r2 * nl_lo));
}

// exp(x^2) erfc(x) for x >= 0.  FP32 (the mixed step's real-space images): the form of Abramowitz &
// Stegun 7.1.26, t (a1 + t (a2 + ...)), t = 1 / (1 + p x), with one term more and p and the
// coefficients fitted to the smallest largest error of erfc, which with the coefficients as rounded
// here is 4.5e-8, at x = 0 (7.1.26: 1.4e-7); with the sum in FP32 too it is 3.8e-7 (7.1.26: 5.6e-7).
// The reciprocal is the hardware's with one Newton step.  FP64: the expansion of Shepherd and
// Laframboise (Math. Comp. 36 (1981) 249), (1 + 2 x) exp(x^2) erfc(x) as a polynomial in t = (x -
// 3.75) / (x + 3.75), degree 22, coefficients fitted in 60-digit arithmetic: relative error <=
// 3.2e-16 over 0 <= x <= 30; even and odd powers in chains of their own.  The exponential is the
// one the image term needs anyway.
__device__ __forceinline__ float erfcx_image(float x)
{
    const float d = __builtin_fmaf(0.39f, x, 1.0f);
    float t = __builtin_amdgcn_rcpf(d);
    t = __builtin_fmaf(__builtin_fmaf(-d, t, 1.0f), t, t);
    return t * (0.23532544076442719f + t * (0.09138698875904083f + t * (0.6495629549026489f +
           t * (-0.6354047656059265f + t * (0.8866671323776245f + t * -0.22753779590129852f)))));
}
__device__ __forceinline__ double erfcx_image(double x)
{
    const double a = x + 3.75, b = __builtin_fma(2.0, x, 1.0), d = a * b;
    double q = __builtin_amdgcn_rcp(d);
    q = __builtin_fma(__builtin_fma(-d, q, 1.0), q, q);
    q = __builtin_fma(__builtin_fma(-d, q, 1.0), q, q);
    const double t = (x - 3.75) * (b * q), u = t * t;
    const double* c = c_img.erfcx;
    double e = c[22], o = c[21];
#pragma unroll
    for (int k = 20; k >= 0; k -= 2) {
        e = __builtin_fma(e, u, c[k]);
        if (k > 0) o = __builtin_fma(o, u, c[k - 1]);
    }
    return __builtin_fma(o, t, e) * (a * q);
}

// 1/r of an image at squared distance r2: FP32 the hardware's reciprocal square root (about 1
// ulp); FP64 its estimate refined by one third-order step (below an ulp).
__device__ __forceinline__ float inv_dist(float r2) { return __builtin_amdgcn_rsqf(r2); }
__device__ __forceinline__ double inv_dist(double r2)
{
    const double y = __builtin_amdgcn_rsq(r2);
    const double e = __builtin_fma(-(r2 * y), y, 1.0);
    return __builtin_fma(__builtin_fma(e, 0.375, 0.5), y * e, y);
}

// floor(sqrt(m)) for 0 <= m <= 25 (lattice radius <= 5)
__device__ __forceinline__ int isqrt_small(int m)
{
    int r = 0;
    while ((r + 1) * (r + 1) <= m) ++r;
    return r;
}

// Overlapping beads: + overlapping RPY - non-overlapping RPY, which the lattice sums count
// (diff_tensor.c:115-148 Smith, :279-313 Beenakker; the same terms).
__device__ __forceinline__ void overlap_correction(double rx, double ry, double rz, double r2,
                                                   double ai, double aj, double preDii,
                                                   double preDij, Blk6& out)
{
    const double rn = sqrt(r2), inv = 1.0 / rn;
    const double ex = rx * inv, ey = ry * inv, ez = rz * inv;
    const double sig = 0.5 * (ai + aj);
    const double pre1 = preDii / sig;
    const double part1 = 1.0 - 9.0 * rn / (32.0 * sig);
    const double c1 = 3.0 * rn / (32.0 * sig);
    const double pre2 = preDij / rn;
    const double sr = (ai * ai + aj * aj) / r2;
    const double d2 = 1.0 + sr / 3.0, o2 = 1.0 - sr;
    out.xx += pre1 * (part1 + c1 * ex * ex) - pre2 * (d2 + ex * ex * o2);
    out.yy += pre1 * (part1 + c1 * ey * ey) - pre2 * (d2 + ey * ey * o2);
    out.zz += pre1 * (part1 + c1 * ez * ez) - pre2 * (d2 + ez * ez * o2);
    out.xy += pre1 * c1 * ex * ey - pre2 * ex * ey * o2;
    out.xz += pre1 * c1 * ex * ez - pre2 * ex * ez * o2;
    out.yz += pre1 * c1 * ey * ez - pre2 * ey * ez * o2;
}

// The reciprocal sum of a pair at separation (rx, ry, rz) into Q (xx yy zz xy xz yz), FP64.  With
// C_h = cos(h a), S_h = sin(h a) of the axis phase a, the members of a class (+-h, +-f, +-g) add up to
//   sum cos = C_h C_f C_g,  sum (sign h)(sign f) cos = -S_h S_f C_g  (and alike for the other pairs)
// per member, so the diagonal of e e^T takes C C C and its off-diagonals -S S C, -S C S, -C S S.
__device__ __forceinline__ void recip_sum(const EwaldTables& E, double rx, double ry, double rz, double sigma_sq,
                                          double (&Q)[6])
{
    constexpr int RMAX = 5;
    double sx, cx, sy, cy, cz[RMAX + 1], sz[RMAX + 1];
    sincospi(E.phase * rx, &sx, &cx);
    sincospi(E.phase * ry, &sy, &cy);
    cz[0] = 1.0;
    sz[0] = 0.0;
    sincospi(E.phase * rz, &sz[1], &cz[1]);
    const int RR = E.RR_recip, R = isqrt_small(RR);
#pragma unroll
    for (int g = 2; g <= RMAX; ++g) {
        cz[g] = cz[g - 1];
        sz[g] = sz[g - 1];
        if (g <= R) cmul_step(cz[g], sz[g], cz[1], sz[1]);
    }
    double tr = 0.0, d0 = 0.0, d1 = 0.0, d2 = 0.0, o0 = 0.0, o1 = 0.0, o2 = 0.0;
    double hc = 1.0, hs = 0.0;
    int q = 0;
    for (int h = 0; h <= R; ++h) {
        const int nf = isqrt_small(RR - h * h);
        double fc = 1.0, fs = 0.0;
        for (int f = 0; f <= nf; ++f) {
            const int ng = isqrt_small(RR - h * h - f * f);
            const double cc = hc * fc, ss = hs * fs, sc = hs * fc, cs = hc * fs;
#pragma unroll
            for (int g = 0; g <= RMAX; ++g) {
                if (g > ng || (g == 0 && h == 0 && f == 0)) continue;
                const RecipClass& k = c_recip[q++];
                const double u = __builtin_fma(sigma_sq, k.u1, k.u0), w = __builtin_fma(sigma_sq, k.w1, k.w0);
                const double ccc = cc * cz[g], wc = w * cz[g], ws = w * sz[g], t = w * ccc;
                tr = __builtin_fma(u, ccc, tr);
                d0 = __builtin_fma(t, k.e[0], d0);
                d1 = __builtin_fma(t, k.e[1], d1);
                d2 = __builtin_fma(t, k.e[2], d2);
                o0 = __builtin_fma(wc * k.e[3], ss, o0);
                o1 = __builtin_fma(ws * k.e[4], sc, o1);
                o2 = __builtin_fma(ws * k.e[5], cs, o2);
            }
            cmul_step(fc, fs, cy, sy);
        }
        cmul_step(hc, hs, cx, sx);
    }
    Q[0] = tr + d0;
    Q[1] = tr + d1;
    Q[2] = tr + d2;
    Q[3] = -o0;
    Q[4] = -o1;
    Q[5] = -o2;
}

// Real-space images r + L (h, f, g) with h^2 + f^2 + g^2 <= RR, h, then f, then g ascending, with CUT
// within sqrt(rc2) of the pair: image(x, y, z, r2) for each.  A column (h, f) that lies beyond the
// cutoff for every pair of the wavefront is skipped whole.  Without CUT a coordinate that is not a
// number reaches the image term and the tensor.
// Every coordinate is formed from its index with one rounding.  A coordinate stepped by L from r - R L
// carries the rounding at R L: the pair (i, i) then misses its central image's zero for most boxes
// that are not exact in a few bits, and near images lose bits in all of them.
template <typename T, bool CUT, typename F>
__device__ __forceinline__ void each_image(const double box, const int RR, const T rc2, double rx, double ry,
                                           double rz, F&& image)
{
    const int R = isqrt_small(RR);
    for (int h = -R; h <= R; ++h) {
        const T x = (T)__builtin_fma(box, (double)h, rx);
        const int nf = isqrt_small(RR - h * h);
        for (int f = -nf; f <= nf; ++f) {
            const T y = (T)__builtin_fma(box, (double)f, ry), rho = x * x + y * y;
            if (CUT && !__any(rho <= rc2)) continue;
            const int ng = isqrt_small(RR - h * h - f * f);
            double gd = -ng;
            for (int g = -ng; g <= ng; ++g, gd += 1.0) {
                const T z = (T)__builtin_fma(box, gd, rz), r2 = rho + z * z;
                if (r2 != (T)0 && (!CUT || r2 <= rc2)) image(x, y, z, r2);
            }
        }
    }
}

// Beenakker block for the pair (i, j): r = r_j - r_i (no minimum image, dist_vec), radii
// ai, aj; self = (i == j) adds the self term and clears the off-diagonal entries.
// What bounds it: VALU issue (93 % of the cycles of the N = 8192 TEA sums), per image about 40
// instructions in FP32 and 100 in FP64 after the pair's constants are taken out of the loop, where
// the term as written in the reference took 78 in FP32 with its divisions and exponentials
// (converged split at N = 8192, mixed: 6.2 -> 4.0 ms for all pairs).
template <typename T>
__device__ __forceinline__ Blk6 beenakker_block(double rx, double ry, double rz, double ai,
                                                double aj, bool self, double preDii,
                                                double preDij)
{
    const EwaldTables& E = c_ew;
    if (E.min_image) {
        rx -= E.box * rint(rx * E.inv_L);
        ry -= E.box * rint(ry * E.inv_L);
        rz -= E.box * rint(rz * E.inv_L);
    }
    const double sigma_sq = 0.5 * (ai * ai + aj * aj);
    double Qr[6] = {0, 0, 0, 0, 0, 0};  // xx yy zz xy xz yz
    Blk6 out{0, 0, 0, 0, 0, 0};
    const double r2 = rx * rx + ry * ry + rz * rz;
    const double s2 = (ai + aj) * (ai + aj);
    if (!self && r2 < s2) overlap_correction(rx, ry, rz, r2, ai, aj, preDii, preDij, out);
    // An image's term is c1 I + c2 e e^T (diff_tensor.c:328-369) with E = exp(-alpha^2 r^2), X =
    // exp(alpha^2 r^2) erfc(alpha r), s = sigma^2:
    //   c1 = E (P1 / sqrt(pi) + X (0.75 + 0.5 s / r^2) / r),  P1 = (14 alpha^3 s - 4.5 alpha) +
    //        alpha s / r^2 + r^2 (3 alpha^3 - 20 alpha^5 s + 4 alpha^7 s r^2)
    //   c2 = E (P2 / sqrt(pi) + X (0.75 - 1.5 s / r^2) / r),  P2 = (1.5 alpha - 2 alpha^3 s) -
    //        3 alpha s / r^2 + r^2 (16 alpha^5 s - 3 alpha^3 - 4 alpha^7 s r^2)
    // (factors formed in FP64 and rounded to T once: their error is the same for every image)
    const double ap = E.alpha * (1.0 / SQRTPI), a3p = E.alpha3 * (1.0 / SQRTPI), a3s = a3p * sigma_sq, a5s = a3s * E.alpha2;
    const T al = (T)E.alpha, sg1 = (T)(0.5 * sigma_sq), sg2 = (T)(-1.5 * sigma_sq);
    const T as = (T)(ap * sigma_sq), as3 = (T)(-3.0 * ap * sigma_sq), p0 = (T)(14.0 * a3s - 4.5 * ap);
    const T p1 = (T)(3.0 * a3p - 20.0 * a5s), p2 = (T)(4.0 * a5s * E.alpha2);
    const T q0 = (T)(1.5 * ap - 2.0 * a3s), q1 = (T)(16.0 * a5s - 3.0 * a3p);
    // exponent factor: FP64 -alpha^2; FP32 -alpha^2 log2(e), high and low part
    const double nlg = sizeof(T) == 8 ? -E.alpha2 : -E.alpha2 * 1.4426950408889634074;
    const T nl = (T)nlg, nl_lo = (T)(nlg - (double)nl);
    T Ot[7] = {0, 0, 0, 0, 0, 0, 0};   // xx yy zz xy xz yz of c2 e e^T, and c1 (FP32)
    each_image<T, true>(E.box, E.RR_real, (T)E.rc2, rx, ry, rz, [&](T x, T y, T z, T rr) {
        const T inv_r = inv_dist(rr), ir2 = inv_r * inv_r;
        const T X = erfcx_image(rr * inv_r * al) * inv_r;
        const T ex = exp_image(rr, nl, nl_lo);
        const T c1 = ex * (X * ((T)0.75 + sg1 * ir2) + (p0 + as * ir2 + rr * (p1 + p2 * rr)));
        const T w = ex * ir2 * (X * ((T)0.75 + sg2 * ir2) + (q0 + as3 * ir2 + rr * (q1 - p2 * rr)));
        const T wx = w * x, wy = w * y, wz = w * z;
        // FP64: c1 and c2 e e^T, of opposite signs, meet before the sum over the images rounds them;
        // FP32's error is the terms' own
        if constexpr (sizeof(T) == 8) {
            Ot[0] += wx * x + c1;
            Ot[1] += wy * y + c1;
            Ot[2] += wz * z + c1;
        } else {
            Ot[0] += wx * x;
            Ot[1] += wy * y;
            Ot[2] += wz * z;
            Ot[6] += c1;
        }
        Ot[3] += wx * y;
        Ot[4] += wx * z;
        Ot[5] += wy * z;
    });
    // reciprocal space (FP64); none when every factor is zero (the reference's split, whose
    // factors underflow)
    if (E.nrecip > 0) recip_sum(E, rx, ry, rz, sigma_sq, Qr);
    out.xx += preDii * ((double)Ot[0] + (double)Ot[6] + Qr[0]);
    out.yy += preDii * ((double)Ot[1] + (double)Ot[6] + Qr[1]);
    out.zz += preDii * ((double)Ot[2] + (double)Ot[6] + Qr[2]);
    out.xy += preDii * ((double)Ot[3] + Qr[3]);
    out.xz += preDii * ((double)Ot[4] + Qr[4]);
    out.yz += preDii * ((double)Ot[5] + Qr[5]);
    if (self) {
        // diff_tensor.c:403-422
        const double sc3 = preDii * (E.self_a + E.self_b * ai * ai);
        out.xx = preDii / ai + sc3 + out.xx;
        out.yy = preDii / ai + sc3 + out.yy;
        out.zz = preDii / ai + sc3 + out.zz;
        out.xy = out.xz = out.yz = 0.0;
    }
    return out;
}

// Smith-Ewald block (src/diff_alg/diff_tensor.c:102-263) in reduced units v = r / L with
// the .prm alpha (EwaldTables.alpha): per lattice vector (h, f, g) of the sphere,
//   real space, x = v + (h, f, g), |x| = r, e = x / r (in T):
//     Op += (erfc(a r)/r) I + (erfc(a r)/r + 2 a exp(-a^2 r^2)/sqrt(pi)) e e^T
//     Qp += s I + (-3 s - 4 a^3 exp(-a^2 r^2)/sqrt(pi)) e e^T,
//           s = (erfc(a r) + 2 a r exp(-a^2 r^2)/sqrt(pi)) / r^3
//   reciprocal, (h, f, g) != 0, k^2 = h^2 + f^2 + g^2 (FP64, tabulated factors):
//     Op += G1 cos I + (-1 + m k^2) G1 cos e e^T,  Qp += G2 cos e e^T,
//     cos = cos 2 pi v.(h, f, g)
//   D_ij += preDii (0.75/L Op + sigma^2/(2 L^3) Qp); self: + preDii/a - self term.
// Both parts of an image's term are added with their factors before the sum over images (FP64).
// 1/sqrt(pi) is the reference's M1_SQRTPI = 0.5641895835 (src/data.h:228).
template <typename T>
__device__ __forceinline__ Blk6 smith_block(double rx, double ry, double rz, double ai,
                                            double aj, bool self, double preDii, double preDij)
{
    const EwaldTables& E = c_ew;
    const double sigma_sq = 0.5 * (ai * ai + aj * aj);
    double O[7] = {0, 0, 0, 0, 0, 0, 0};  // xx yy zz xy xz yz of c2 e e^T, and c1
    double Qr[6] = {0, 0, 0, 0, 0, 0};
    Blk6 out{0, 0, 0, 0, 0, 0};
    const double r2 = rx * rx + ry * ry + rz * rz;
    const double s2 = (ai + aj) * (ai + aj);
    if (!self && r2 < s2) overlap_correction(rx, ry, rz, r2, ai, aj, preDii, preDij, out);
    const double preQ = 0.5 * sigma_sq * E.inv_L * E.inv_L * E.inv_L;
    const T al = (T)E.alpha, m1sp = (T)0.5641895835, am2 = (T)2 * al * m1sp, am4 = (T)4 * (T)E.alpha3 * m1sp;
    const T fo = (T)E.preO, fq = (T)preQ;
    const double nlg = sizeof(T) == 8 ? -E.alpha2 : -E.alpha2 * 1.4426950408889634074;
    const T nl = (T)nlg, nl_lo = (T)(nlg - (double)nl);
    each_image<T, false>(1.0, E.RR_real, (T)0, rx * E.inv_L, ry * E.inv_L, rz * E.inv_L, [&](T x, T y, T z, T rr) {
        const T inv_r = inv_dist(rr), ir2 = inv_r * inv_r, rn = rr * inv_r;
        const T eg = exp_image(rr, nl, nl_lo);
        const T ec = erfcx_image(rn * al) * eg;
        const T so = ec * inv_r, e2 = am2 * eg;
        const T sq = ir2 * (so + e2);
        const T c1 = fo * so + fq * sq;
        const T w = ir2 * (fo * (so + e2) - fq * ((T)3 * sq + am4 * eg));
        const T wx = w * x, wy = w * y, wz = w * z;
        O[0] += (double)(wx * x);
        O[1] += (double)(wy * y);
        O[2] += (double)(wz * z);
        O[3] += (double)(wx * y);
        O[4] += (double)(wx * z);
        O[5] += (double)(wy * z);
        O[6] += (double)c1;
    });
    if (E.nrecip > 0) recip_sum(E, rx, ry, rz, sigma_sq, Qr);
    out.xx += preDii * (O[0] + O[6] + Qr[0]);
    out.yy += preDii * (O[1] + O[6] + Qr[1]);
    out.zz += preDii * (O[2] + O[6] + Qr[2]);
    out.xy += preDii * (O[3] + Qr[3]);
    out.xz += preDii * (O[4] + Qr[4]);
    out.yz += preDii * (O[5] + Qr[5]);
    if (self) {
        // diff_tensor.c:241-263
        const double m1 = 0.5641895835;
        double sc3 = E.alpha * ai * E.inv_L;
        sc3 = sc3 * sc3 * sc3 * m1 / 3;
        sc3 = 0.75 * E.inv_L * 1.5 * E.alpha * ai * m1 * E.inv_L +
              0.5 * ai * ai * E.inv_L * E.inv_L * E.inv_L * sc3;
        sc3 *= preDii;
        out.xx = preDii / ai - sc3 + out.xx;
        out.yy = preDii / ai - sc3 + out.yy;
        out.zz = preDii / ai - sc3 + out.zz;
        out.xy = out.xz = out.yz = 0.0;
    }
    return out;
}

}  // namespace bdh
