// Reverse-mode derivative (vector-Jacobian product) of one FP64 Ermak-McCammon step with
// Cholesky noise refactored at the step's positions (the step of comp_step_ermak /
// compute_hydro_ermak, src/diff_alg/diff_comp.c:152-179, diff_equation.c:216-286,
// diff_rand.c:64-85):
//
//   r' = r + c D(r) F(r) + s L(r) xi,        c = dt / kT,  s = sqrt(2 dt),  D = L L^T
//
// For a cotangent g of r' the cotangent of r is
//
//   rbar = g + grad_r <U, D(r)> - c H(r) (D g)
//   U    = c sym(g F^T) + sym(S),  S = L^-T Phi(L^T Lbar) L^-1,  Lbar = s tril(g xi^T)
//
// H is the Hessian of the potential energy (dF/dr = -H), Phi the lower triangle with the
// diagonal halved (derivative of the Cholesky factor, Murray 2016).  With a = L^T g,
// Phi(L^T Lbar) = s Phi(a xi^T), and the contraction needs only
//
//   Z = S + S^T = L^-T B L^-1,   B = s (Phi(a xi^T) + Phi(a xi^T)^T):  B_ij = s a_max(i,j) xi_min(i,j)
//
// B is a rank-one matrix on either side of its diagonal, so with M = L^-1 the product G^T =
// L^-T B costs two running sums along each column of M:
//   G(j, r) = s (xi_j sum_{i >= j} M_ir a_i + a_j sum_{r <= i < j} M_ir xi_i),   j >= r
// and Z(r, c) = sum_{j >= c} G(j, r) M(j, c) for r <= c, the only half a symmetric Z needs.  The
// inverse and that product are n^3 / 3 operations each; the two triangular solves with n
// right-hand sides that give S as written are n^3 each.
//
// Kernels (FP64; the inverse and the product are the O(n^3) part):
//   adj_lt_g_kernel         a = L^T g
//   adj_diag_inv_kernel     64 x 64 diagonal blocks of M
//   adj_mul_kernel          M from its diagonal blocks, doubling their size: [A 0; C D]^-1 has
//                           -D^-1 (C A^-1) below the diagonal; and Z's upper triangle
//   adj_semi_kernel         G
//   adj_mirror_kernel       Z from its upper triangle
//   adj_contract_kernel     grad_r <U, D(r)> over the RPY blocks (diff_tensor.c:45-92), column splits
//   adj_hvp_pairs_kernel,   g + contraction - c H y  (pair and bond Hessians, the forward
//   adj_hvp_finish_kernel   pass's cutoffs and bonded-partner scaling; bond.c:43-85)
#include <algorithm>

#include "bdh_common.hpp"
#include "bdh_kernels.hpp"
#include "bdh_mfma.hpp"
#include "bdh_pairterm.hpp"

namespace bdh {

__global__ void __launch_bounds__(256)
adj_lt_g_kernel(const double* __restrict__ L, long long ld, int n, const double* __restrict__ g,
                double* __restrict__ a)
{
    __shared__ double s_red[256];
    const int i = blockIdx.x;
    const double* col = L + (long long)i * ld;
    double acc = 0.0;
    for (int k = i + threadIdx.x; k < n; k += 256) acc += col[k] * g[k];
    s_red[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s_red[threadIdx.x] += s_red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) a[i] = s_red[0];
}

constexpr int ADJ_NB = 64;

// Column c of the inverse of the 64 x 64 diagonal block J of L by forward substitution
// (workgroup J, thread c), zeros above the diagonal included, into the diagonal block of M.
__global__ void __launch_bounds__(64)
adj_diag_inv_kernel(const double* __restrict__ L, long long ld, int np, double* __restrict__ M)
{
    __shared__ double sL[ADJ_NB][ADJ_NB + 1];   // sL[i][k] = L(64 J + i, 64 J + k)
    __shared__ double s_inv[ADJ_NB];
    const int j0 = blockIdx.x * ADJ_NB, c = threadIdx.x;
    double m[ADJ_NB];
#pragma unroll
    for (int k = 0; k < ADJ_NB; ++k) m[k] = L[(long long)(j0 + k) * ld + j0 + c];
#pragma unroll
    for (int k = 0; k < ADJ_NB; ++k) sL[c][k] = m[k];
    s_inv[c] = 1.0 / sL[c][c];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ADJ_NB; ++i) {
        double b[2] = {(i == c) ? 1.0 : 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < i; ++k) b[k & 1] -= sL[i][k] * m[k];
        m[i] = (i >= c) ? (b[0] + b[1]) * s_inv[i] : 0.0;
    }
    double* out = M + (long long)(j0 + c) * np + j0;
#pragma unroll
    for (int i = 0; i < ADJ_NB; ++i) out[i] = m[i];
}

// One 64 x 64 tile of a product per workgroup, over the 64-blocks k0 .. k1 - 1 of its inner
// index, in stages of 32: FP64 MFMA, wavefront w the 32 x 16 part at rows 32 (w % 2), columns
// 16 (w / 2), the next two stages in registers while the current one is multiplied from LDS.
// Eight wavefronts, so that one alone on a SIMD does not wait for the LDS between its MFMAs where
// tiles are fewer than CUs.
// All matrices are column-major.  An operand whose tile index runs along memory lies in LDS as
// [k][tile index], one whose k does as [tile index][k], both with pitches that leave the operand
// reads without bank conflicts.
//   MUL_T  T(i, q) = sum_k L(i, k) M(k, q), k in the first of two blocks of sb 64-blocks, q there,
//          i in the second
//   MUL_M  M(i, q) = -sum_k M(i, k) T(k, q), k in the second block
//   MUL_Z  Z(r, c) = sum_j G(j, r) M(j, c), r <= c
// Every stage's partial sum starts from zero and is added as a whole: Z's terms cancel, and with sums
// over all of n the reverse step of 300 beads was 2.4e-15 off (of its norm, extended precision),
// where the two triangular solves these products replace had 8.8e-16; so 8.4e-16, for 2 % of the time.
// Tiles with the longest sums come first.  Bound by MFMA issue in the large levels and MUL_Z and
// by one tile's length in the small ones: n = 3072 the inverse 0.38 ms in 12 launches, Z 0.20 ms,
// against 2.25 ms for the triangular solves; with four wavefronts 0.44 and 0.20 ms.
enum { MUL_T, MUL_M, MUL_Z };
constexpr int ADJ_KC = 32, ADJ_PN = ADJ_NB + 16, ADJ_PT = ADJ_KC + 2;

template <int MODE>
__global__ void __launch_bounds__(512, 4)
adj_mul_kernel(const double* A, long long lda, const double* B, int np, int sb, int last, double* C)
{
    constexpr bool AN = MODE != MUL_Z;   // A's tile index runs along memory
    constexpr int ASZ = AN ? ADJ_KC * ADJ_PN : ADJ_NB * ADJ_PT, BSZ = ADJ_NB * ADJ_PT;
    __shared__ __align__(16) double smem[2 * (ASZ + BSZ)];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nb = np / ADJ_NB;
    int i, q, k0, k1;   // 64-blocks
    if constexpr (MODE == MUL_Z) {
        int c = (int)((sqrt(8.0 * blockIdx.x + 1.0) - 1.0) * 0.5);
        while (c * (c + 1) / 2 > (int)blockIdx.x) --c;
        while ((c + 1) * (c + 2) / 2 <= (int)blockIdx.x) ++c;
        q = c;
        i = blockIdx.x - c * (c + 1) / 2;
        k0 = c;
        k1 = nb;
    } else {
        // `last` is the number of block rows of the last pair's second block
        const int pair = min((int)blockIdx.x / (sb * sb), ((int)gridDim.x - sb * last) / (sb * sb));
        const int e = blockIdx.x - pair * sb * sb, base = 2 * sb * pair;
        const int rows = base + 2 * sb <= nb ? sb : last;
        if (MODE == MUL_T) {
            i = base + sb + e % rows;
            q = base + e / rows;
            k0 = q;
            k1 = base + sb;
        } else {
            i = base + sb + rows - 1 - e / sb;
            q = base + e % sb;
            k0 = base + sb;
            k1 = i + 1;
        }
    }
    const double* a0 = AN ? A + (long long)i * ADJ_NB : A + (long long)i * ADJ_NB * lda;
    const double* b0 = B + (long long)q * ADJ_NB * np;
    doublex2 va[2][2], vb[2][2];
    const int nr = (tid & 31) * 2, nk = tid >> 5;    // [k][tile index]: two rows of columns nk + 16 u
    const int tk = (tid & 15) * 2, tc = tid >> 4;    // [tile index][k]: two k of tile columns tc + 32 u
    auto load = [&](int k, int h) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            va[h][u] = *reinterpret_cast<const doublex2*>(AN ? a0 + (long long)(k + nk + 16 * u) * lda + nr
                                                          : a0 + (long long)(tc + 32 * u) * lda + k + tk);
            vb[h][u] = *reinterpret_cast<const doublex2*>(b0 + (long long)(tc + 32 * u) * np + k + tk);
        }
    };
    auto store = [&](int buf, int h) {
        double* sa = smem + buf * (ASZ + BSZ);
        double* sb_ = sa + ASZ;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            *reinterpret_cast<doublex2*>(AN ? sa + (nk + 16 * u) * ADJ_PN + nr : sa + (tc + 32 * u) * ADJ_PT + tk) = va[h][u];
            *reinterpret_cast<doublex2*>(sb_ + (tc + 32 * u) * ADJ_PT + tk) = vb[h][u];
        }
    };
    const int r0 = 32 * (wave & 1), c0 = 16 * (wave >> 1), lr = lane & 15, lk = lane >> 4;
    doublex4 sum[2] = {doublex4{0.0, 0.0, 0.0, 0.0}, doublex4{0.0, 0.0, 0.0, 0.0}};
    // transposed: accumulator r of lane l is column 4 r + l / 16, row l % 16
    const int kb = k0 * ADJ_NB, ke = k1 * ADJ_NB;
    auto stage = [&](int k, int buf) {   // stage k is in LDS half buf, the next in registers buf ^ 1, two on to buf
        __syncthreads();
        if (k + 2 * ADJ_KC < ke) load(k + 2 * ADJ_KC, buf);
        const double* sa = smem + buf * (ASZ + BSZ);
        const double* sb_ = sa + ASZ;
        double av[2][2], bv[2];
        auto fetch = [&](int s) {
            const int kk = 4 * s + lk;
            bv[s & 1] = sb_[(c0 + lr) * ADJ_PT + kk];
#pragma unroll
            for (int x = 0; x < 2; ++x)
                av[s & 1][x] = AN ? sa[kk * ADJ_PN + r0 + 16 * x + lr] : sa[(r0 + 16 * x + lr) * ADJ_PT + kk];
        };
        doublex4 acc[2] = {doublex4{0.0, 0.0, 0.0, 0.0}, doublex4{0.0, 0.0, 0.0, 0.0}};
        fetch(0);
#pragma unroll
        for (int s = 0; s < ADJ_KC / 4; ++s) {
            if (s + 1 < ADJ_KC / 4) fetch(s + 1);
#pragma unroll
            for (int x = 0; x < 2; ++x) acc[x] = mfma_f64_16x16x4(bv[s & 1], av[s & 1][x], acc[x]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int x = 0; x < 2; ++x) sum[x] += acc[x];
        if (k + ADJ_KC < ke) store(buf ^ 1, buf ^ 1);
    };
    static_assert(ADJ_NB % (2 * ADJ_KC) == 0, "whole pairs of stages");
    load(kb, 0);
    load(kb + ADJ_KC, 1);
    store(0, 0);
    for (int k = kb; k < ke; k += 2 * ADJ_KC) {
        stage(k, 0);
        stage(k + ADJ_KC, 1);
    }
    double* out = C + ((long long)q * ADJ_NB + c0 + lk) * np + i * ADJ_NB + r0 + lr;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int x = 0; x < 2; ++x) out[(long long)4 * r * np + 16 * x] = MODE == MUL_M ? -sum[x][r] : sum[x][r];
}

// Column r of G (workgroup r) from the start of r's 64-block, zero above the diagonal.  Thread t
// takes rows 4 t .. 4 t + 3 of each 1024 of a span of 4096; sums of a wavefront by lane shifts, of
// the workgroup through LDS.  Bound by reading M's and writing G's lower triangle: n = 3072 39 us.
constexpr int SEMI_SPAN = 4096, SEMI_SPANS = 64;

__global__ void __launch_bounds__(256)
adj_semi_kernel(int np, int n, const double* __restrict__ M, const double* __restrict__ a,
                const double* __restrict__ xi, double s, double* __restrict__ G)
{
    __shared__ double s_w[2][16];      // wavefront w's part u of the span at 4 u + w
    __shared__ double s_off[2][16];    // sums of M_ir a_i after, of M_ir xi_i before each part
    __shared__ double s_span[SEMI_SPANS];   // sums of M_ir a_i over the spans
    const int r = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int jb = r & ~(ADJ_NB - 1);
    const double* m = M + (long long)r * np;
    double* g = G + (long long)r * np;
    const int spans = (np - jb + SEMI_SPAN - 1) / SEMI_SPAN;
    if (spans > 1) {
        for (int p = 0; p < spans; ++p) {
            double v = 0.0;
            for (int j = jb + p * SEMI_SPAN + t, e = min(n, jb + (p + 1) * SEMI_SPAN); j < e; j += 256)
                if (j >= r) v += m[j] * a[j];
#pragma unroll
            for (int w = 32; w > 0; w >>= 1) v += __shfl_xor(v, w);
            if (lane == 0) s_w[0][wave] = v;
            __syncthreads();
            if (t == 0) s_span[p] = (s_w[0][0] + s_w[0][1]) + (s_w[0][2] + s_w[0][3]);
            __syncthreads();
        }
    }
    double before = 0.0;   // sum of M_ir xi_i over the spans before
    for (int p = 0; p < spans; ++p) {
        double after = 0.0;
        for (int x = spans - 1; x > p; --x) after += s_span[x];
        double va[4][4], vx[4][4], sa[4], sx[4], ca[4], cx[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = jb + p * SEMI_SPAN + 1024 * u + 4 * t;
            doublex2 v[2] = {{0.0, 0.0}, {0.0, 0.0}};
            if (j < np) {
                v[0] = *reinterpret_cast<const doublex2*>(m + j);
                v[1] = *reinterpret_cast<const doublex2*>(m + j + 2);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool in = j + e >= r && j + e < n;
                va[u][e] = in ? v[e >> 1][e & 1] * a[j + e] : 0.0;
                vx[u][e] = in ? v[e >> 1][e & 1] * xi[j + e] : 0.0;
            }
            sa[u] = ca[u] = (va[u][0] + va[u][1]) + (va[u][2] + va[u][3]);
            sx[u] = cx[u] = (vx[u][0] + vx[u][1]) + (vx[u][2] + vx[u][3]);
        }
#pragma unroll
        for (int w = 1; w < 64; w <<= 1)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const double da = __shfl_down(ca[u], w), dx = __shfl_up(cx[u], w);
                if (lane + w < 64) ca[u] += da;
                if (lane >= w) cx[u] += dx;
            }
        __syncthreads();   // s_w is free
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (lane == 0) s_w[0][4 * u + wave] = ca[u];
            if (lane == 63) s_w[1][4 * u + wave] = cx[u];
        }
        __syncthreads();
        if (t < 16) {
            double v = after;
            for (int x = 15; x > t; --x) v += s_w[0][x];
            s_off[0][t] = v;
        } else if (t >= 64 && t < 80) {
            double v = before;
            for (int x = 0; x < t - 64; ++x) v += s_w[1][x];
            s_off[1][t - 64] = v;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            double oa = s_off[0][4 * u + wave] + (ca[u] - sa[u]);
            double ox = s_off[1][4 * u + wave] + (cx[u] - sx[u]);
            const int j = jb + p * SEMI_SPAN + 1024 * u + 4 * t;
            double o[4];
#pragma unroll
            for (int e = 3; e >= 0; --e) {
                oa += va[u][e];
                o[e] = oa;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool in = j + e >= r && j + e < n;
                o[e] = in ? s * (xi[j + e] * o[e] + a[j + e] * ox) : 0.0;
                ox += vx[u][e];
            }
            if (j < np) {
                *reinterpret_cast<doublex2*>(g + j) = doublex2{o[0], o[1]};
                *reinterpret_cast<doublex2*>(g + j + 2) = doublex2{o[2], o[3]};
            }
        }
        before = s_off[1][15] + s_w[1][15];
    }
}

// Z (np x np) from its upper triangle in Y; 64 x 64 tiles through LDS, so that the contraction
// reads one coalesced matrix.
__global__ void __launch_bounds__(256)
adj_mirror_kernel(int np, const double* __restrict__ Y, double* __restrict__ Z)
{
    __shared__ double t[ADJ_NB][ADJ_NB + 1];
    const int i0 = blockIdx.x * ADJ_NB, q0 = blockIdx.y * ADJ_NB;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const bool upper = i0 < q0;
    // t[c][x]: the tile itself (upper) or its mirror image (rows q0 .., columns i0 ..)
    const double* src = upper ? Y + (long long)q0 * np + i0 : Y + (long long)i0 * np + q0;
#pragma unroll
    for (int u = 0; u < ADJ_NB / 4; ++u) t[ty + 4 * u][tx] = src[(long long)(ty + 4 * u) * np + tx];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < ADJ_NB / 4; ++u) {
        const int qq = ty + 4 * u;
        const bool direct = upper || (i0 == q0 && tx <= qq);   // on the diagonal tile both are the same tile
        Z[(long long)(q0 + qq) * np + i0 + tx] = direct ? t[qq][tx] : t[tx][qq];
    }
}

// f, f', g, g' of the RPY block B = f I + g e e^T at separation r (radii ai, aj).
__device__ __forceinline__ void rpy_fg(double r, double ai, double aj, double preDii, double preDij,
                                       double& fp, double& gv, double& gp)
{
    if (r < ai + aj) {
        const double abar = 0.5 * (ai + aj);
        fp = -9.0 * preDii / (32.0 * abar * abar);
        gv = preDii / abar * (3.0 * r / (32.0 * abar));
        gp = 3.0 * preDii / (32.0 * abar * abar);
    } else {
        const double sig2 = ai * ai + aj * aj, r2 = r * r;
        fp = preDij * (-1.0 / r2 - sig2 / (r2 * r2));
        gv = preDij * (1.0 / r - sig2 / (r2 * r));
        gp = preDij * (-1.0 / r2 + 3.0 * sig2 / (r2 * r2));
    }
}

// Term of pair (k, j) of out_k = sum_{j != k} grad_d <W_kj, B(d)> at d = r_k - r_j, with
// W_kj = c (g_k F_j^T + F_k g_j^T) + Z(3k.., 3j..)  (W = 2 U_kj).
__device__ __forceinline__ void contract_pair(const double4& pk, const double4& pj, int k, int j,
                                              double preDii, double preDij, const double* __restrict__ Z,
                                              long long ldz, const double* gk, const double* Fk,
                                              const double* __restrict__ g, const double* __restrict__ F,
                                              double c, double* acc)
{
    const double d[3] = {pk.x - pj.x, pk.y - pj.y, pk.z - pj.z};
    const double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    const double e[3] = {d[0] / r, d[1] / r, d[2] / r};
    double fp, gv, gp;
    rpy_fg(r, pk.w, pj.w, preDii, preDij, fp, gv, gp);
    double W[3][3];
#pragma unroll
    for (int u = 0; u < 3; ++u)
#pragma unroll
        for (int v = 0; v < 3; ++v) {
            const long long row = 3LL * k + u, col = 3LL * j + v;
            W[u][v] = c * (gk[u] * F[3 * j + v] + Fk[u] * g[3 * j + v]) + Z[col * ldz + row];
        }
    const double trW = W[0][0] + W[1][1] + W[2][2];
    double We[3], WTe[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        We[u] = W[u][0] * e[0] + W[u][1] * e[1] + W[u][2] * e[2];
        WTe[u] = W[0][u] * e[0] + W[1][u] * e[1] + W[2][u] * e[2];
    }
    const double eWe = e[0] * We[0] + e[1] * We[1] + e[2] * We[2];
    double v[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) v[u] = We[u] + WTe[u];
    const double ev = e[0] * v[0] + e[1] * v[1] + e[2] * v[2];
#pragma unroll
    for (int u = 0; u < 3; ++u)
        acc[u] += (fp * trW + gp * eWe) * e[u] + (gv / r) * (v[u] - ev * e[u]);
}

// Workgroup (x, s): row beads k = 64 x + lane, column beads j of split s
// (js beads from s js); wave w takes j = s js + w, + 4, ...  The four waves' sums meet in
// LDS in wave order and land in P[s][3k + u]; the splits are summed afterwards in split
// order, so the result does not depend on scheduling.
__global__ void __launch_bounds__(256)
adj_contract_kernel(const double4* __restrict__ pos, int N, double preDii, double preDij,
                    const double* __restrict__ Z, long long ldz, const double* __restrict__ g,
                    const double* __restrict__ F, double c, int js, double* __restrict__ P)
{
    __shared__ double red[3][3][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k = blockIdx.x * 64 + lane;
    const int j0 = blockIdx.y * js, j1 = min(N, j0 + js);
    double acc[3] = {0.0, 0.0, 0.0};
    if (k < N) {
        const double4 pk = pos[k];
        const double gk[3] = {g[3 * k], g[3 * k + 1], g[3 * k + 2]};
        const double Fk[3] = {F[3 * k], F[3 * k + 1], F[3 * k + 2]};
        for (int j = j0 + wave; j < j1; j += 4) {
            if (j == k) continue;
            contract_pair(pk, pos[j], k, j, preDii, preDij, Z, ldz, gk, Fk, g, F, c, acc);
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int u = 0; u < 3; ++u) red[wave - 1][u][lane] = acc[u];
    }
    __syncthreads();
    if (wave == 0 && k < N) {
        double* out = P + (long long)blockIdx.y * 3 * N;
#pragma unroll
        for (int u = 0; u < 3; ++u)
            out[3 * k + u] = ((acc[u] + red[0][u][lane]) + red[1][u][lane]) + red[2][u][lane];
    }
}

// Pair part of (H y)_k over the column beads of split s (the forward pass's cutoffs and
// bonded-partner scaling); workgroups, waves and the wave-order LDS sum as in
// adj_contract_kernel, partials in P[s][3k + u].
__global__ void __launch_bounds__(256)
adj_hvp_pairs_kernel(const double4* __restrict__ pos, const double* __restrict__ Q,
                     const double2* __restrict__ LJ, int N, Topology topo, ForceParams fp,
                     const double* __restrict__ y, int js, double* __restrict__ P)
{
    __shared__ double red[3][3][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k = blockIdx.x * 64 + lane;
    const int j0 = blockIdx.y * js, j1 = min(N, j0 + js);
    double acc[3] = {0.0, 0.0, 0.0};
    if (k < N) {
        const double4 pk = pos[k];
        const double2 ljk = LJ[k];
        const double qk = Q[k];
        const double yk[3] = {y[3 * k], y[3 * k + 1], y[3 * k + 2]};
        const int nb0 = fp.use_conn ? topo.conn_off[k] : 0;
        const int nb1 = fp.use_conn ? topo.conn_off[k + 1] : 0;
        const double lj6 = fp.lj_6_term;
        for (int j = j0 + wave; j < j1; j += 4) {
            if (j == k) continue;
            const double4 pj = pos[j];
            const double d[3] = {pk.x - pj.x, pk.y - pj.y, pk.z - pj.z};
            const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
            if (r2 > fp.far_r2) continue;
            const double r = sqrt(r2);
            const bool conn = bonded(topo, nb0, nb1, j);
            double d1 = 0.0, d2 = 0.0;
            if (fp.alpha_lj != 0.0) {
                const double2 ljj = LJ[j];
                const double sig = ljk.x + ljj.x;
                const double cut = fp.cutoff_lj > 0.0 ? fp.cutoff_lj : (double)1.122462f * sig;
                const double scale = conn ? fp.bond_lj_scale : 1.0;
                if (r <= cut && scale != 0.0) {
                    const double eps = sqrt(ljk.y * ljj.y);
                    double s6 = sig / r;
                    s6 *= s6;
                    s6 *= s6 * s6;
                    d1 += scale * fp.alpha_lj * eps * (-12.0 * s6 * s6 + 6.0 * lj6 * s6) / r;
                    d2 += scale * fp.alpha_lj * eps * (156.0 * s6 * s6 - 42.0 * lj6 * s6) / r2;
                }
            }
            if (fp.elec) {
                const double scale = conn ? fp.bond_c_scale : 1.0;
                if (r <= fp.cutoff_c && scale != 0.0) {
                    const double qq = fp.gam * qk * Q[j];
                    const double ex = exp(-fp.kappa_c * r);
                    const double kap = fp.kappa_c;
                    d1 += -scale * qq * ex * (1.0 / r2 + kap / r);
                    d2 += scale * qq * ex * (2.0 / (r2 * r) + 2.0 * kap / r2 + kap * kap / r);
                }
            }
            if (d1 == 0.0 && d2 == 0.0) continue;
            const double e[3] = {d[0] / r, d[1] / r, d[2] / r};
            const double dy[3] = {yk[0] - y[3 * j], yk[1] - y[3 * j + 1], yk[2] - y[3 * j + 2]};
            const double ed = e[0] * dy[0] + e[1] * dy[1] + e[2] * dy[2];
    #pragma unroll
            for (int u = 0; u < 3; ++u) acc[u] += d2 * ed * e[u] + (d1 / r) * (dy[u] - ed * e[u]);
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int u = 0; u < 3; ++u) red[wave - 1][u][lane] = acc[u];
    }
    __syncthreads();
    if (wave == 0 && k < N) {
        double* out = P + (long long)blockIdx.y * 3 * N;
#pragma unroll
        for (int u = 0; u < 3; ++u)
            out[3 * k + u] = ((acc[u] + red[0][u][lane]) + red[1][u][lane]) + red[2][u][lane];
    }
}

// out_k = g_k + contraction_k - c (H y)_k: the pair partials summed in split order, then the
// bond Hessians (bond.c:43-85).
__global__ void __launch_bounds__(256)
adj_hvp_finish_kernel(const double4* __restrict__ pos, int N, Topology topo, const double* __restrict__ y,
                      const double* __restrict__ P, int S, const double* __restrict__ contract,
                      const double* __restrict__ g, double c, double* __restrict__ out)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= N) return;
    const double4 pk = pos[k];
    const double yk[3] = {y[3 * k], y[3 * k + 1], y[3 * k + 2]};
    double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll 8
    for (int sp = 0; sp < S; ++sp) {
#pragma unroll
        for (int u = 0; u < 3; ++u) acc[u] += P[(long long)sp * 3 * N + 3 * k + u];
    }
    for (int b = topo.bond_off[k]; b < topo.bond_off[k + 1]; ++b) {
        const int p = topo.bond_p[b];
        const double r0 = topo.bond_parm[3 * b], rmax = topo.bond_parm[3 * b + 1];
        const double H = topo.bond_parm[3 * b + 2];
        const double4 pp = pos[p];
        const double d[3] = {pk.x - pp.x, pk.y - pp.y, pk.z - pp.z};
        const double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
        const double e[3] = {d[0] / r, d[1] / r, d[2] / r};
        const double den = 1.0 - r * r / (rmax * rmax);
        const double b1 = H * (r - r0) / den;
        const double b2 = H * (den + (r - r0) * 2.0 * r / (rmax * rmax)) / (den * den);
        const double dy[3] = {yk[0] - y[3 * p], yk[1] - y[3 * p + 1], yk[2] - y[3 * p + 2]};
        const double ed = e[0] * dy[0] + e[1] * dy[1] + e[2] * dy[2];
#pragma unroll
        for (int u = 0; u < 3; ++u) acc[u] += b2 * ed * e[u] + (b1 / r) * (dy[u] - ed * e[u]);
    }
#pragma unroll
    for (int u = 0; u < 3; ++u) out[3 * k + u] = g[3 * k + u] + contract[3 * k + u] - c * acc[u];
}

__global__ void __launch_bounds__(256)
adj_promote_kernel(const float* __restrict__ A, long long count, double* __restrict__ Ld)
{
    const long long e = (long long)blockIdx.x * 1024 + 4 * threadIdx.x;
    if (e + 3 < count) {
        const float4 v = *reinterpret_cast<const float4*>(A + e);
        Ld[e] = v.x;
        Ld[e + 1] = v.y;
        Ld[e + 2] = v.z;
        Ld[e + 3] = v.w;
    } else {
        for (long long q = e; q < count; ++q) Ld[q] = A[q];
    }
}

int launch_adj_promote(const float* d_A, long long count, double* d_Ld, hipStream_t st)
{
    BDH_CHECK(count > 0 && count % 4 == 0, "adjoint: promote count");
    hipLaunchKernelGGL(adj_promote_kernel, dim3((unsigned)ceil_div_ll(count, 1024)), dim3(256), 0, st, d_A, count,
                       d_Ld);
    BDH_LAUNCH_CHECK();
    return 0;
}

int launch_adj_lt_g(const double* d_L, long long ld, int n, const double* d_g, double* d_a, hipStream_t st)
{
    hipLaunchKernelGGL(adj_lt_g_kernel, dim3(n), dim3(256), 0, st, d_L, ld, n, d_g, d_a);
    BDH_LAUNCH_CHECK();
    return 0;
}

int launch_adj_inverse(const double* d_L, long long ld, int np, double* d_M, double* d_T, hipStream_t st)
{
    BDH_CHECK(np % ADJ_NB == 0 && ld >= np && ld % 2 == 0, "adjoint inverse: padded order");
    const int nb = np / ADJ_NB;
    hipLaunchKernelGGL(adj_diag_inv_kernel, dim3(nb), dim3(ADJ_NB), 0, st, d_L, ld, np, d_M);
    BDH_LAUNCH_CHECK();
    for (int sb = 1; sb < nb; sb *= 2) {
        const int pairs = (nb + sb - 1) / (2 * sb);   // those with a second block, perhaps a short one
        const int last = std::min(sb, nb - (2 * pairs - 1) * sb);
        const dim3 grid((unsigned)((pairs - 1) * sb * sb + sb * last));
        hipLaunchKernelGGL(adj_mul_kernel<MUL_T>, grid, dim3(512), 0, st, d_L, ld, (const double*)d_M, np, sb, last,
                           d_T);
        BDH_LAUNCH_CHECK();
        hipLaunchKernelGGL(adj_mul_kernel<MUL_M>, grid, dim3(512), 0, st, (const double*)d_M, (long long)np,
                           (const double*)d_T, np, sb, last, d_M);
        BDH_LAUNCH_CHECK();
    }
    return 0;
}

int launch_adj_noise_part(int np, int n, const double* d_M, const double* d_a, const double* d_xi, double s,
                          double* d_G, hipStream_t st)
{
    BDH_CHECK(np % ADJ_NB == 0 && np <= SEMI_SPAN * SEMI_SPANS, "adjoint: padded order");
    const int nb = np / ADJ_NB;
    hipLaunchKernelGGL(adj_semi_kernel, dim3(np), dim3(256), 0, st, np, n, d_M, d_a, d_xi, s, d_G);
    BDH_LAUNCH_CHECK();
    // Z's upper triangle into G's storage: its diagonal tiles are G's own, read by no other
    hipLaunchKernelGGL(adj_mul_kernel<MUL_Z>, dim3(nb * (nb + 1) / 2), dim3(512), 0, st, (const double*)d_G,
                       (long long)np, d_M, np, 0, 0, d_G);
    BDH_LAUNCH_CHECK();
    return 0;
}

int launch_adj_mirror(int np, const double* d_Y, double* d_Z, hipStream_t st)
{
    BDH_CHECK(np % ADJ_NB == 0, "adjoint: padded order");
    hipLaunchKernelGGL(adj_mirror_kernel, dim3(np / ADJ_NB, np / ADJ_NB), dim3(256), 0, st, np, d_Y, d_Z);
    BDH_LAUNCH_CHECK();
    return 0;
}

int adj_contract_splits(int N)
{
    const int rows = ceil_div(N, 64);
    return std::max(1, std::min({ADJ_CONTRACT_MAX_SPLITS, ceil_div(1024, rows), ceil_div(N, 4)}));
}

int launch_adj_contract(const double4* d_pos, int N, double preDii, double preDij, const double* d_Y2,
                        long long ldy, const double* d_g, const double* d_F, double c, double* d_part,
                        double* d_out, hipStream_t st)
{
    const int S = adj_contract_splits(N);
    const int js = ceil_div(N, S);
    hipLaunchKernelGGL(adj_contract_kernel, dim3(ceil_div(N, 64), S), dim3(256), 0, st, d_pos, N, preDii,
                       preDij, d_Y2, ldy, d_g, d_F, c, js, d_part);
    BDH_LAUNCH_CHECK();
    ReduceJobs jobs{};
    jobs.job[0] = ReduceJob{d_part, d_out, 3 * N, S, 0, 1.0};
    return launch_reduce_partials(jobs, 1, 3 * N, st);
}

int launch_adj_hvp(const double4* d_pos, const double* d_Q, const double2* d_LJ, int N,
                   const Topology& topo, const ForceParams& fp, const double* d_y,
                   const double* d_contract, const double* d_g, double c, double* d_part, double* d_out,
                   hipStream_t st)
{
    const int S = adj_contract_splits(N);
    const int js = ceil_div(N, S);
    hipLaunchKernelGGL(adj_hvp_pairs_kernel, dim3(ceil_div(N, 64), S), dim3(256), 0, st, d_pos, d_Q, d_LJ,
                       N, topo, fp, d_y, js, d_part);
    BDH_LAUNCH_CHECK();
    hipLaunchKernelGGL(adj_hvp_finish_kernel, dim3(ceil_div(N, 64)), dim3(64), 0, st, d_pos, N, topo, d_y,
                       (const double*)d_part, S, d_contract, d_g, c, d_out);
    BDH_LAUNCH_CHECK();
    return 0;
}


// ---- parameter cotangents of one step: theta_bar = (c D g)^T dF/dtheta for the per-bead LJ
// epsilon_k and radius R_k, the charges Q_k and the per-bond constants H_b.  With
// F_k = -sum_j phi'(r_kj) e_kj, pair (k, j) contributes -(y_k - y_j).e_kj dphi'/dtheta:
//   LJ  (LJ.c:37-64, sigma_kj = R_k + R_j, eps_kj = sqrt(eps_k eps_j), data.c:97-102)
//        phi' = a eps_kj (-12 s6^2 + 6 lj6 s6) / r                 -> d/deps_k = phi' / (2 eps_k)
//        d phi' / d sigma = a eps_kj (-144 s6^2 + 36 lj6 s6) / (sigma r)  (= d / dR_k)
//   DH  (electro.c:36-56)  phi' = -(gamma/eps_r) Q_k Q_j e^{-kappa r} (1/r^2 + kappa/r)
//        d phi' / dQ_k = -(gamma/eps_r) Q_j e^{-kappa r} (1/r^2 + kappa/r)
//   bond (bond.c:43-85)   phi' = H (r - r0) / (1 - r^2/rmax^2)     -> d/dH = (r - r0) / den
// Row k sums its pairs over one column split (four wavefronts interleave the columns and
// meet in LDS in wave order); P[split][3][N] holds (eps, R, Q) sums, combined in split order.
__global__ void __launch_bounds__(256)
adj_param_pairs_kernel(const double4* __restrict__ pos, const double* __restrict__ Q,
                       const double2* __restrict__ LJ, int N, Topology topo, ForceParams fp,
                       const double* __restrict__ y, int js, double* __restrict__ P)
{
    __shared__ double red[3][3][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k = blockIdx.x * 64 + lane;
    const int j0 = blockIdx.y * js, j1 = min(N, j0 + js);
    double acc[3] = {0.0, 0.0, 0.0};
    if (k < N) {
        const double4 pk = pos[k];
        const double2 ljk = LJ[k];
        const double yk[3] = {y[3 * k], y[3 * k + 1], y[3 * k + 2]};
        const int nb0 = fp.use_conn ? topo.conn_off[k] : 0;
        const int nb1 = fp.use_conn ? topo.conn_off[k + 1] : 0;
        const double lj6 = fp.lj_6_term;
        for (int j = j0 + wave; j < j1; j += 4) {
            if (j == k) continue;
            const double4 pj = pos[j];
            const double d[3] = {pk.x - pj.x, pk.y - pj.y, pk.z - pj.z};
            const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
            if (r2 > fp.far_r2) continue;
            const double r = sqrt(r2);
            const bool conn = bonded(topo, nb0, nb1, j);
            const double ed = (d[0] * (yk[0] - y[3 * j]) + d[1] * (yk[1] - y[3 * j + 1]) +
                               d[2] * (yk[2] - y[3 * j + 2])) / r;
            if (fp.alpha_lj != 0.0) {
                const double2 ljj = LJ[j];
                const double sig = ljk.x + ljj.x;
                const double cut = fp.cutoff_lj > 0.0 ? fp.cutoff_lj : (double)1.122462f * sig;
                const double scale = conn ? fp.bond_lj_scale : 1.0;
                if (r <= cut && scale != 0.0) {
                    const double eps = sqrt(ljk.y * ljj.y);
                    double s6 = sig / r;
                    s6 *= s6;
                    s6 *= s6 * s6;
                    const double a = scale * fp.alpha_lj * eps;
                    acc[0] += ed * (a * (-12.0 * s6 * s6 + 6.0 * lj6 * s6) / r);
                    acc[1] += ed * (a * (-144.0 * s6 * s6 + 36.0 * lj6 * s6) / (sig * r));
                }
            }
            if (fp.elec) {
                const double scale = conn ? fp.bond_c_scale : 1.0;
                if (r <= fp.cutoff_c && scale != 0.0) {
                    const double ex = exp(-fp.kappa_c * r);
                    acc[2] += ed * (-scale * fp.gam * Q[j] * ex * (1.0 / r2 + fp.kappa_c / r));
                }
            }
        }
    }
    if (wave > 0) {
#pragma unroll
        for (int u = 0; u < 3; ++u) red[wave - 1][u][lane] = acc[u];
    }
    __syncthreads();
    if (wave == 0 && k < N) {
        double* out = P + (long long)blockIdx.y * 3 * N;
#pragma unroll
        for (int u = 0; u < 3; ++u)
            out[u * N + k] = ((acc[u] + red[0][u][lane]) + red[1][u][lane]) + red[2][u][lane];
    }
}

// Per bead: the split partials summed in split order, scaled by -c (and 1 / (2 eps_k) for
// epsilon); per bond, at its lower-index end, -c (y_k - y_p).e (r - r0) / den into
// H_bar[bond_id] (each bond written once).
__global__ void __launch_bounds__(256)
adj_param_finish_kernel(const double4* __restrict__ pos, const double2* __restrict__ LJ, int N,
                        Topology topo, const int* __restrict__ bond_id, const double* __restrict__ y,
                        const double* __restrict__ P, int S, double c, double* __restrict__ eps_bar,
                        double* __restrict__ R_bar, double* __restrict__ Q_bar, double* __restrict__ H_bar)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= N) return;
    double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll 8
    for (int sp = 0; sp < S; ++sp) {
#pragma unroll
        for (int u = 0; u < 3; ++u) acc[u] += P[(long long)sp * 3 * N + u * N + k];
    }
    eps_bar[k] = -c * acc[0] / (2.0 * LJ[k].y);
    R_bar[k] = -c * acc[1];
    Q_bar[k] = -c * acc[2];
    const double4 pk = pos[k];
    for (int b = topo.bond_off[k]; b < topo.bond_off[k + 1]; ++b) {
        const int p = topo.bond_p[b];
        if (p < k) continue;
        const double r0 = topo.bond_parm[3 * b], rmax = topo.bond_parm[3 * b + 1];
        const double4 pp = pos[p];
        const double d[3] = {pk.x - pp.x, pk.y - pp.y, pk.z - pp.z};
        const double r = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
        const double den = 1.0 - r * r / (rmax * rmax);
        const double ed = (d[0] * (y[3 * k] - y[3 * p]) + d[1] * (y[3 * k + 1] - y[3 * p + 1]) +
                           d[2] * (y[3 * k + 2] - y[3 * p + 2])) / r;
        H_bar[bond_id[b]] = -c * ed * (r - r0) / den;
    }
}

int launch_adj_params(const double4* d_pos, const double* d_Q, const double2* d_LJ, int N,
                      const Topology& topo, const int* d_bond_id, const ForceParams& fp,
                      const double* d_y, double c, double* d_part, double* d_eps_bar,
                      double* d_R_bar, double* d_Q_bar, double* d_H_bar, hipStream_t st)
{
    const int S = adj_contract_splits(N);
    const int js = ceil_div(N, S);
    hipLaunchKernelGGL(adj_param_pairs_kernel, dim3(ceil_div(N, 64), S), dim3(256), 0, st, d_pos, d_Q, d_LJ,
                       N, topo, fp, d_y, js, d_part);
    BDH_LAUNCH_CHECK();
    hipLaunchKernelGGL(adj_param_finish_kernel, dim3(ceil_div(N, 64)), dim3(64), 0, st, d_pos, d_LJ, N, topo,
                       d_bond_id, d_y, (const double*)d_part, S, c, d_eps_bar, d_R_bar, d_Q_bar, d_H_bar);
    BDH_LAUNCH_CHECK();
    return 0;
}

}  // namespace bdh
