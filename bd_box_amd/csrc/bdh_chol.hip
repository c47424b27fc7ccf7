// Blocked Cholesky D = L L^T and the triangular product L.x on gfx950.
//
// Replaces the reference's my_dpotrf / my_dtrmv (src/myblas.c:45-118: LAPACK
// dpotrf("U") + dtrmv("U","T"), or MAGMA spotrf_gpu('L') + cublasStrmv in the CUDA
// build).  The factor is stored lower, column-major, in place of D; n is padded to a
// multiple of PAD_TO with an identity block so every tile is whole.
//
// One launch factors a matrix, or all matrices of a batch: one workgroup per 128x128 tile,
// left-looking (chol_flow_kernel).  The sums over earlier columns run on MFMA:
//   T = float : v_mfma_f32_32x32x2_f32 (or split-bf16 v_mfma_f32_32x32x16_bf16), FP32 accumulation
//   T = double: v_mfma_f64_16x16x4_f64
// The 64x64 diagonal blocks are factored (factor_diag64) and the blocks below them solved
// (flow_solve64) in FP64 in both precisions; in the FP32 variant the factor is rounded to FP32
// when stored.
#include <algorithm>

#include "bdh_common.hpp"
#include "bdh_kernels.hpp"
#include "bdh_mfma.hpp"

namespace bdh {

constexpr int DG_LD = CHOL_NB + 1;   // row pitch (doubles) of the diagonal block in LDS

// Value of v held by lane `src` (uniform), through two v_readlane_b32.
__device__ __forceinline__ double readlane_f64(double v, int src)
{
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, src);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), src);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Per diagonal block, the workspace Lb holds (FP64):
//   Lb[0 .. 4095]      L_kk column-major, zeros above the diagonal
//   Lb[4096 + SINV J]  inverse of its J-th 16x16 diagonal sub-block, column-major with pitch
//                      SINV_P (odd, so the factor's rows and the solve's columns of it both
//                      spread over the LDS banks), J = 0..3
// What lies above the diagonal of either is not part of the factor and is not read.
constexpr int SINV_P = 17;
constexpr int SINV = 16 * SINV_P;
constexpr int LB_STRIDE = CHOL_NB * CHOL_NB + 4 * SINV;

// threadIdx.x; OPAQUE: as if unknown to the compiler, so that what depends on it is computed where it
// is used.  Otherwise the FP64 tile functions keep addresses in registers that they then spill in
// the chain (n = 768 205 us, 189 so; FP32 has the registers and is 1 % faster without), and in the
// loop over tasks every address is taken out of the loop and spilled.
template <bool OPAQUE>
__device__ __forceinline__ int flow_tid()
{
    int t = threadIdx.x;
    if constexpr (OPAQUE) asm volatile("" : "+v"(t));
    return t;
}

// One wavefront: columns cw .. cw + 15 of the 64x64 block, lane = row, p[u] = column cw + u with
// every earlier group's update made; finished columns go to L (LDS, column-major; what a lane
// above the diagonal holds is not part of the factor).
// Per column t the pivot chain is: reciprocal square root, l_{t+1,t}, the next pivot
// a_{t+1,t+1} - l_{t+1,t}^2.  The root is the hardware's estimate (relative error about 2^-23) refined
// by one third-order step, y (1 + e/2 + 3 e^2/8) with e = 1 - x y^2, whose truncation (5/16 e^3) is
// below 2^-68: four dependent operations where two Newton steps take eight.  Column t + 1 takes
// column t's update from a broadcast (v_readlane) of its entry before it is scaled, so it does not
// wait for the LDS; the later ones take it one
// column late from LDS broadcasts of the stored column, two at a time between the dependent
// operations of the next pivot (fill), which are 12 cycles apart where an FP64 FMA issues in 4.
// step(t): work of the caller's for the same gaps.
// The inverse of the 16x16 diagonal sub-block is the solution of X L^T = I, i.e. what the column
// steps make of 16 more rows that hold the identity: FIRST (cw = 0, every lane a row of the
// block) carries them in y; the other groups hold them in lanes 0 .. 15 of p, whose rows lie
// above the group's diagonal.
template <bool FIRST, typename Step>
__device__ __forceinline__ void factor_group16(double (&p)[16], double (&y)[16], double* __restrict__ L, int cw,
                                               int lane, Step&& step)
{
    double piv = readlane_f64(p[0], cw);
    double lprev = 0.0, yprev = 0.0, far[2][16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const int c = cw + t;
        double (&fp)[16] = far[(t + 1) & 1], (&fn)[16] = far[t & 1];
        auto fill = [&](int u0, int u1) {
#pragma unroll
            for (int u = u0; u < u1; ++u)
                if (t > 0 && u < 16) {
                    p[u] = __builtin_fma(-lprev, fp[u], p[u]);
                    if (FIRST) {
                        y[u] = __builtin_fma(-yprev, fp[u], y[u]);
                        // keeps the step here: left alone, all of y sinks behind the pivots
                        asm volatile("" : "+v"(y[u]));
                    }
                }
            __builtin_amdgcn_sched_barrier(0);
        };
        const double q = __builtin_amdgcn_rsq(piv);
        double a1 = 0.0, a2 = 0.0;
        if (t < 15) a1 = readlane_f64(p[t], c + 1);
        __builtin_amdgcn_sched_barrier(0);
        const double m = piv * q;
        step(t);
        __builtin_amdgcn_sched_barrier(0);
        const double e = __builtin_fma(-m, q, 1.0);
        fill(t + 1, t + 3);
        const double k = __builtin_fma(e, 0.375, 0.5), qe = q * e;
        if (t < 15) a2 = readlane_f64(p[t + 1], c + 1);
        fill(t + 3, t + 5);
        const double rs = __builtin_fma(k, qe, q);
        fill(t + 5, t + 7);
        const double s1 = a1 * rs;   // l_{c+1, c}
        const double l = p[t] * rs;
        fill(t + 7, t + 9);
        piv = __builtin_fma(-s1, s1, a2);
        L[c * CHOL_NB + lane] = l;
        // l_{cw+u, c}: LDS broadcasts of the column this wavefront has just stored (its own
        // store, in order before these loads)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = t + 2; u < 16; ++u) fn[u] = L[c * CHOL_NB + cw + u];
        p[t] = l;
        if (FIRST) y[t] *= rs;
        if (t < 15) {
            p[t + 1] = __builtin_fma(-l, s1, p[t + 1]);
            if (FIRST) y[t + 1] = __builtin_fma(-y[t], s1, y[t + 1]);
        }
        fill(t + 9, 16);
        lprev = l;
        if (FIRST) yprev = y[t];
    }
}

// In-place FP64 Cholesky of the 64x64 block held in LDS, called by all 256 threads.
//   in : sD[r * DG_LD + c], lower part (r >= c) read
//   out: the same memory in the layout of Lb (L[c * 64 + r], then the inverses of its four
//        16x16 diagonal sub-blocks: sD is then sLT / sInv of the solve), and the same in Lb.
//        sD must hold LB_STRIDE doubles.
// Wavefront 0 factors the block alone, so no step of the chain waits for another wavefront; the
// other three are free for work of the caller's (others(), called by each of them) until the
// barrier at the end.  The block is taken in four groups of 16 columns: the group's columns on
// the VALU (factor_group16), its update of the columns beyond on v_mfma_f64_16x16x4_f64.  The
// trailing 16x16 tiles stay in MFMA accumulators from the start, transposed (accumulator r of
// lane l: column 4 r + l/16 of the tile, row l%16), so the next group's tiles reach the
// lane = row form with one conflict-free pass through the LDS columns they will be factored in.
// What bounds it: one wavefront's serial work.  Of 19000 cycles (7.9 us) on an idle GPU the 64
// pivots take 62 %, 160 to 215 cycles each: about 80 of dependent operations, then the issue of the
// column's updates and the LDS reads of its broadcasts.  The inverses' stores, the updates between
// the groups and the tiles' way through the LDS take 36 %.
// 64x64 block on an idle GPU: 11.2 us as a pipeline of the four wavefronts over the column
// groups, 8.2 us as here.
// A non-positive (or NaN) pivot records row c0 + j + 1 in *status (the first one wins) and the
// factorization continues with NaN, as the reference's dpotrf reports INFO.
template <typename Others>
__device__ __forceinline__ void factor_diag64(double* __restrict__ sD, int c0, int* __restrict__ status,
                                              Others&& others)
{
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __syncthreads();   // the block in sD may have been written by another wavefront
    if (w == 0) {
        const int lr = lane & 15, lq = lane >> 4;
        double p[16], y[16];
        doublex4 T[3][3];   // tile (i + 1, j + 1), j <= i, transposed
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            p[u] = sD[lane * DG_LD + u];
            y[u] = (u == lane) ? 1.0 : 0.0;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j <= i; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) T[i][j][r] = sD[(16 * i + 16 + lr) * DG_LD + 16 * j + 16 + 4 * r + lq];
        __builtin_amdgcn_wave_barrier();   // the block is in registers: its memory is reused for L
        double* L = sD;
        double* sInv = sD + CHOL_NB * CHOL_NB;
        double x[3][4];   // the last group's rows below, as MFMA operands
        // the group's update of tile (i + 1, j + 1), its k-step s4
        auto update = [&](int i, int j, int s4) { T[i][j] = mfma_f64_16x16x4(-x[j][s4], x[i][s4], T[i][j]); };
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int cw = 16 * g;
            if (g == 0) {
                factor_group16<true>(p, y, L, 0, lane, [](int) {});
            } else {
                // the previous group's update of the tiles beyond this one, a step per column
                factor_group16<false>(p, y, L, cw, lane, [&](int t) {
                    const int s4 = t & 3, q = t >> 2;
                    if (g == 1 && q < 3) update(q == 0 ? 1 : 2, q == 2 ? 2 : 1, s4);
                    if (g == 2 && q < 1) update(2, 2, s4);
                });
            }
            if (lane < 16) {
#pragma unroll
                for (int u = 0; u < 16; ++u) sInv[SINV * g + lane * SINV_P + u] = g == 0 ? y[u] : p[u];
            }
            if (g < 3) {
                // this group's update of the next group's tiles
                const int cn = cw + 16;
#pragma unroll
                for (int i = g; i < 3; ++i)
#pragma unroll
                    for (int s4 = 0; s4 < 4; ++s4) x[i][s4] = L[(cw + 4 * s4 + lq) * CHOL_NB + 16 * i + 16 + lr];
#pragma unroll
                for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
                    for (int i = g; i < 3; ++i) update(i, g, s4);
                // into the lane = row form through the LDS columns they will be factored in
#pragma unroll
                for (int i = g; i < 3; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) L[(cn + 4 * r + lq) * CHOL_NB + 16 * i + 16 + lr] = T[i][g][r];
                __builtin_amdgcn_wave_barrier();
                // rows from the group's diagonal down; the identity in lanes 0 .. 15
#pragma unroll
                for (int u = 0; u < 16; ++u) {
                    double v = L[(cn + u) * CHOL_NB + lane];
                    asm volatile("" : "+v"(v));   // a select, not a branch around the load
                    p[u] = (lane >= cn) ? v : (lane == u ? 1.0 : 0.0);
                }
            }
        }
        // a pivot that is not positive leaves NaN on the diagonal from its column on
        const unsigned long long bad = __ballot(!(L[lane * CHOL_NB + lane] > 0.0));
        if (bad && lane == 0) atomicCAS(status, 0, c0 + __builtin_ctzll(bad) + 1);
    } else {
        others();
    }
    __syncthreads();   // L and the inverses complete in LDS
}

// Agent-scope store: written through to memory, so it is visible to every workgroup once it has
// completed.
__device__ __forceinline__ void st_agent(double* p, double v)
{
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), __builtin_bit_cast(unsigned long long, v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(float* p, float v)
{
    __hip_atomic_store(reinterpret_cast<unsigned*>(p), __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// The factored block and its inverses from the LDS into Lb (the same layout), at agent scope.
__device__ __forceinline__ void store_lkk(const double* __restrict__ sD, double* __restrict__ Lb)
{
    constexpr int NL = LB_STRIDE / 256;
    double v[NL + 1];
#pragma unroll
    for (int i = 0; i < NL; ++i) v[i] = sD[threadIdx.x + 256 * i];
    if (threadIdx.x < LB_STRIDE % 256) v[NL] = sD[threadIdx.x + 256 * NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) st_agent(Lb + threadIdx.x + 256 * i, v[i]);
    if (threadIdx.x < LB_STRIDE % 256) st_agent(Lb + threadIdx.x + 256 * NL, v[NL]);
}

// L (lower part) of the factored block, L[c * 64 + r] in LDS, into A, in T.
template <typename T>
__device__ __forceinline__ void store_diag64(const double* __restrict__ L, T* __restrict__ A,
                                             long long ld, int c0)
{
    for (int e = threadIdx.x; e < CHOL_NB * CHOL_NB; e += 256) {
        const int r = e % CHOL_NB, c = e / CHOL_NB;
        if (r >= c) A[(long long)(c0 + c) * ld + c0 + r] = (T)L[c * CHOL_NB + r];
    }
}

// L_kk and its diagonal sub-block inverses (Lb, FP64) into LDS at sLT, in Lb's own layout.
__device__ __forceinline__ void load_lkk(const double* __restrict__ Lb, double* __restrict__ sLT)
{
    // all loads are issued before the LDS stores (which the compiler would otherwise order
    // between them)
    constexpr int NL = LB_STRIDE / 256;
    double v[NL + 1];
#pragma unroll
    for (int i = 0; i < NL; ++i) v[i] = Lb[threadIdx.x + 256 * i];
    if (threadIdx.x < LB_STRIDE % 256) v[NL] = Lb[threadIdx.x + 256 * NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) sLT[threadIdx.x + 256 * i] = v[i];
    if (threadIdx.x < LB_STRIDE % 256) sLT[threadIdx.x + 256 * NL] = v[NL];
    __syncthreads();
}

// ------------------------------------------------------------------ MFMA pieces
constexpr int SY_KCH = 32;                 // k per stage of the split products
constexpr int SY_HP = SY_KCH / 2 + 4;      // row pitch of a split stage, in 32-bit words

// bf16 bits of x, round to nearest even (finite inputs)
__device__ __forceinline__ unsigned bf16_bits(float x)
{
    const unsigned u = __builtin_bit_cast(unsigned, x);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ void split_bf16(float x, unsigned& hi, unsigned& lo)
{
    hi = bf16_bits(x);
    lo = bf16_bits(x - __builtin_bit_cast(float, hi << 16));
}

// acc = sum_k A[ra + i][k] A[ca + j][k], k < K (a multiple of 32), of a 32 x 32 block on one
// wavefront's MFMA with operands loaded straight from A (no LDS), 32 k at a time with the next 32 in
// flight.  v_mfma_f32_32x32x2_f32: lane l feeds row l % 32, k = l / 32; acc[r] holds row
// 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
__device__ __forceinline__ void quad_acc(const float* __restrict__ A, long long ld, int ra, int ca, int K,
                                         floatx16& acc)
{
    constexpr int KC = 32, NJ = KC / 2;
    const int lane = flow_tid<true>() & 63, l32 = lane & 31, lh = lane >> 5;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    float av[NJ], bv[NJ];
    auto load = [&](int k0, float (&a)[NJ], float (&b)[NJ]) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const float* col = A + (long long)(k0 + 2 * j + lh) * ld;
            a[j] = col[ra + l32];
            b[j] = col[ca + l32];
        }
    };
    load(0, av, bv);
    for (int k0 = 0; k0 < K; k0 += KC) {
        float an[NJ], bn[NJ];
        if (k0 + KC < K) load(k0 + KC, an, bn);
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc = mfma_f32_32x32x2(av[j], bv[j], acc);
        if (k0 + KC < K) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                av[j] = an[j];
                bv[j] = bn[j];
            }
        }
    }
}

// The same in FP64, K a multiple of 16: v_mfma_f64_16x16x4_f64 on the 2 x 2 tiles of the block,
// lane l feeds row l % 16, k = l / 16; acc[i][j][r] holds row 16 i + 4 r + l / 16, column
// 16 j + l % 16.  16 k at a time with the next 16 in flight.
__device__ __forceinline__ void quad_acc(const double* __restrict__ A, long long ld, int ra, int ca, int K,
                                         doublex4 (&acc)[2][2])
{
    const int lane = flow_tid<true>() & 63, l16 = lane & 15, lq = lane >> 4;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = doublex4{0.0, 0.0, 0.0, 0.0};
    double av[4][2], bv[4][2];
    auto load = [&](int k0, double (&a)[4][2], double (&b)[4][2]) {
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
            const double* col = A + (long long)(k0 + 4 * s4 + lq) * ld;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                a[s4][i] = col[ra + 16 * i + l16];
                b[s4][i] = col[ca + 16 * i + l16];
            }
        }
    };
    load(0, av, bv);
    for (int k0 = 0; k0 < K; k0 += 16) {
        double an[4][2], bn[4][2];
        if (k0 + 16 < K) load(k0 + 16, an, bn);
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = mfma_f64_16x16x4(av[s4][i], bv[s4][j], acc[i][j]);
        if (k0 + 16 < K) {
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    av[s4][i] = an[s4][i];
                    bv[s4][i] = bn[s4][i];
                }
        }
    }
}

// ------------------------------------------------------------------ factorization as one launch
// The whole factorization of one matrix, or of every matrix of a batch, is one launch of one
// workgroup per 128x128 tile of the lower triangle, left-looking: the workgroup of tile (i, j)
// accumulates sum_k L_ik L_jk^T over the tile columns k < j as they are published, then finishes
// its tile and publishes it.
//   i > j  (flow_tile)  z = A_ij - sum, solved with L_jj and stored: the rows 128 i .. of panel j.
//   i = j  (flow_diag)  z factored: the two 64x64 diagonal blocks and the block below the first.
// A workgroup takes its tile from a counter when it starts (flow_task), column by column, so every
// tile it waits for was taken before by a workgroup that is finished or running, and the waits end
// whatever the number of resident workgroups, the order in which they start, and what else runs.
// With the workgroup's index in place of the counter they would not have to: workgroups go to the
// XCDs by index and wait there for room, and two factorizations on two streams could each hold all
// places of the XCD on which the other's lowest unfinished tile waits for one.
// The waits are bounded anyway (flow_wait).
// What bounds it: for small matrices the chain diagonal block -> solve of the next block row ->
// its update -> next diagonal block; for large ones MFMA issue of the accumulation, whose operands
// are shared in L2 (C is read and written once in FP32, once per 256 columns in FP64).  The chain
// overlaps with everything else, since the workgroups of the following tile columns are
// resident and accumulate what is already published.
// Measured against one launch per 256-column outer panel (n_pad >= 1024) or per 64-column panel
// (below), right-looking: n = 768 FP64 640 -> 202 us, n = 1353 FP32 720 -> 331 us, n = 3072 FP64
// 1900 -> 840 us, n = 9000 FP32 5.95 -> 2.82 ms, FP64 11.3 -> 5.7 ms; the batch of 256 chains of
// 64 .. 1024 beads FP32 6.9 -> 4.0 ms.  Beside another tile on its CU a tile takes 13.4 us for 128
// columns in FP32 and 28.7 in FP64 (without the passes over C), MFMA issue at its peak; the rest at
// n = 9000 is the chain (31 us per tile column FP32, 33 FP64) and tiles that become resident too
// late to have caught up.
//
// Visibility across XCDs, whose L2 caches are not coherent within a launch: what other
// workgroups read is stored at agent scope (write-through), the flag that announces it is set
// after those stores have completed, and it lies in memory that no workgroup reads before that
// flag -- the operand copy of tile (i, k) is the mirrored tile (k, i) of the upper triangle, which
// holds no part of the factor; the diagonal blocks are in the workspace.  So no cache holds an
// older copy of such a line, plain loads after the flag see the stored values, and no L2
// invalidation is needed (an acquire per tile was measured to halve the rate of the tiles).
// A tile's own entries (D before, L after) are read and written by its workgroup alone.
//   operand copy: L(128 i + r, 128 k + c) at A[(128 i + c) ld + 128 k + r], r, c < 128, k < i.

// Workspace per tile column j (doubles): diagonal block 2 j (LB_STRIDE), L21 (64 x 64, column c
// at 64 c), diagonal block 2 j + 1; after all of them the flags, one per 128-byte line:
//   dprog[j]  1: diagonal block 2 j and L21 are published, 2: diagonal block 2 j + 1 also
//   rdy[i]    64-column panels of tile row i published so far
constexpr int FLOW_T = 128;
constexpr int FLOW_COL = 2 * LB_STRIDE + CHOL_NB * CHOL_NB;
constexpr int FLAG_STRIDE = 32;

// LOOP: the kernel runs a loop over tasks.
template <typename T, bool LOOP = false>
struct FlowMat {
    __device__ static int tid() { return flow_tid<LOOP || sizeof(T) == 8>(); }
    T* A;
    long long ld;
    int n, nt;   // order (without the identity padding), tile rows
    double* ws;
    int* status;
    int* quiet;  // FLOW_CUS counters (FlowQuiet), or null
    __device__ int* dprog(int j) const { return flags() + j * FLAG_STRIDE; }
    __device__ int* rdy(int i) const { return flags() + (nt + i) * FLAG_STRIDE; }
    __device__ int* flags() const { return reinterpret_cast<int*>(ws + (long long)nt * FLOW_COL); }
    // first element of column k (k < 128 x) of the operand copy of tile row x: rows r = 0 .. 127
    __device__ const T* opnd(int x, int k) const
    {
        return A + (long long)(FLOW_T * x + (k & (FLOW_T - 1))) * ld + (k & ~(FLOW_T - 1));
    }
    __device__ T* tile(int i, int j) const { return A + (long long)FLOW_T * j * ld + FLOW_T * i; }
};

// All threads: this workgroup's agent-scope stores have completed, then *flag = v.
__device__ __forceinline__ void flow_publish(int* flag, int v)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(flag, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Each wavefront: wait until *flag >= need, return the value seen.  After FLOW_TIMEOUT (100 MHz
// ticks: 10 s), or once another wait has timed out, it reports -1 through status and returns
// need: the factorization then ends with wrong values and that status instead of hanging.
constexpr long long FLOW_TIMEOUT = 1000000000ll;
__device__ __forceinline__ int flow_wait(int* flag, int need, int* status)
{
    int v = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (v < need) {
        const long long t0 = wall_clock64();
        for (int it = 1;; ++it) {
            __builtin_amdgcn_s_sleep(1);
            v = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (v >= need) break;
            if ((it & 255) == 0 && (wall_clock64() - t0 > FLOW_TIMEOUT ||
                                    __hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < 0)) {
                if ((threadIdx.x & 63) == 0) atomicCAS(status, 0, -1);
                v = need;
                break;
            }
        }
    }
    // the loads that follow stay behind the flag
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    return __builtin_amdgcn_readfirstlane(v);
}

// The chain's steps are a serial FP64 chain on one wavefront and short MFMA solves.  Beside the
// MFMAs of another workgroup on the same CU, none of which can be interrupted, a diagonal block
// takes 20 .. 27 us instead of 10 and a solve 9 instead of 6, and the whole factorization waits.  So
// the workgroups of tiles (j, j) and (j + 1, j) count themselves on their CU's counter while they
// take those steps, and a workgroup further below the diagonal pauses its accumulation, between
// two stages, while its CU's counter is not zero.  A workgroup counts itself only once what it
// still waits for comes from workgroups that are past their accumulation (or none is left to wait
// for), so a paused one is never waited for.
// Only where workgroups share CUs, that is with more tiles than the chip's 256 CUs (us without /
// with, FP32 and FP64): n = 3072 737 / 735, 861 / 856; 4500 1175 / 1103, 1413 / 1318; 6000 1606 /
// 1467, 2111 / 1917; 9000 3087 / 2808, 5092 / 5009.
constexpr int FLOW_CUS = 2048;
constexpr int QUIET_TILES = 256;
struct FlowQuiet {
    int* q;
    __device__ explicit FlowQuiet(int* quiet)
    {
        // HW_ID bits 8 .. 15: CU and shader array of the XCD; XCC_ID: the XCD
        q = quiet ? quiet + ((__builtin_amdgcn_s_getreg(20 | (2 << 11)) << 8) | __builtin_amdgcn_s_getreg(4 | (8 << 6) | (7 << 11)))
                  : nullptr;
    }
    __device__ void add(int v)
    {
        if (q && flow_tid<true>() == 0) __hip_atomic_fetch_add(q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ int busy() const { return q ? __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0; }
    __device__ void pause() const
    {
        const long long t0 = wall_clock64();
        while (busy() && wall_clock64() - t0 < FLOW_TIMEOUT) __builtin_amdgcn_s_sleep(8);
    }
};

// Panels known to be published in two tile rows (the same row twice for a diagonal tile).
struct FlowReady {
    int *fi, *fj, *status;
    int ri = 0, rj = 0;
    __device__ bool poll(int need)
    {
        if (ri < need) ri = __builtin_amdgcn_readfirstlane(__hip_atomic_load(fi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (rj < need) rj = fj == fi ? ri : __builtin_amdgcn_readfirstlane(__hip_atomic_load(fj, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        const bool ok = ri >= need && rj >= need;
        if (ok) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        return ok;
    }
    __device__ void wait(int need)
    {
        if (ri < need) ri = flow_wait(fi, need, status);
        if (rj < need) rj = fj == fi ? ri : flow_wait(fj, need, status);
    }
};

constexpr int FLOW_KC32 = 32, FLOW_KC64 = 16;        // columns per LDS stage
constexpr int FLOW_P32 = FLOW_T + 4, FLOW_P64 = FLOW_T + 2;   // row pitch of a stage
constexpr int FLOW_SMEM = (LB_STRIDE + CHOL_NB * CHOL_NB) * 8;
static_assert(2 * 2 * FLOW_KC32 * FLOW_P32 * 4 <= FLOW_SMEM && 2 * 2 * FLOW_KC64 * FLOW_P64 * 8 <= FLOW_SMEM &&
              4 * FLOW_T * SY_HP * 4 <= FLOW_SMEM && CHOL_NB * DG_LD <= LB_STRIDE, "LDS of the factorization");

// The accumulated sums of a tile, per wavefront w rows 32 w .. 32 w + 31 of tile row i and all
// 128 columns, transposed (the MFMA row index runs over the tile's columns): FP32 four 32x32 blocks,
// FP64 8 x 2 16x16 blocks.  A partial sum of at most FLOW_FLUSH columns starts from zero and is
// then taken from C as a whole, so that its rounding is relative to that part alone: FP32 keeps
// C - sum in m; FP64 has registers for one set, and C - sum stays in the tile's own entries of A.
// Errors ||(A - L L^T) x|| / ||A x|| in extended precision, tensors of chains and of periodic
// suspensions, N = 60 .. 3000: 1.9e-16 .. 2.9e-16 and 2.2e-16 .. 4.3e-16; with C updated by a launch
// per 256 columns 2.0e-16 .. 3.2e-16 and 2.4e-16 .. 4.4e-16.  Accumulating on -C, without a pass over
// C in memory: 7.2e-16 at n = 768, 2.9e-15 at n = 9000.  From zero, but with no pass in between: 4.6e-16
// at n = 9000; with one every 512 columns 4.2e-16 at n = 2100, periodic (3.0e-16 as here).
// FP64 us on -C / as here: n = 768 196 / 202, 1353 361 / 371, 3072 812 / 840, 4500 1270 / 1350, 9000
// 5050 / 5680; the batch of 256 chains 6.4 / 6.9 ms.  A pass moves 256 kB a tile every 57 us; one
// block at a time beside the stages' products it spills (n = 9000 7.1 ms), as FP64 atomics 5.8 ms.
constexpr int FLOW_FLUSH = 256;
template <typename T>
struct FlowAcc;
template <>
struct FlowAcc<float> {
    floatx16 m[4], a[4];
};
template <>
struct FlowAcc<double> {
    doublex4 a[8][2];
};

// Lane l's entries of FP64 tiles: (column c, row r) of a tile at t is entry (c + l / 16, r + l % 16).
// One 32-bit offset a lane beside addresses that are the same for all lanes, all of them formed where
// they are used: taken out of the loop they would spill.
struct FlowLane {
    unsigned off;
    long long ld;
    __device__ explicit FlowLane(long long ld_) : ld(ld_)
    {
        asm volatile("" : "+s"(ld));
        const int l = flow_tid<true>() & 63;
        off = ((unsigned)(l >> 4) * (unsigned)ld + (l & 15)) * (unsigned)sizeof(double);
    }
    __device__ double* operator()(double* t, int c, int r) const
    {
        return reinterpret_cast<double*>(reinterpret_cast<char*>(t + c * ld) + off) + r;
    }
};

// Sums over the K columns 0 .. K - 1 (K a multiple of 128) of tile (i, j) into acc.  The next
// stage's columns are in registers while this one's are multiplied (ext_vector_type elements: an
// array of HIP's own vector class, loaded under a condition, went through scratch memory and each
// load was waited for at once), and the LDS reads of a product are issued before the MFMAs of the
// one before: 22.6 -> 13.4 us per 128 columns FP32, 46.5 -> 28.7 FP64.
template <bool SPLIT, bool LOOP>
__device__ __forceinline__ void flow_accumulate(const FlowMat<float, LOOP>& M, int i, int j, int K, FlowReady& rd,
                                                const FlowQuiet& quiet, unsigned char* smem, FlowAcc<float>& acc)
{
    const int tid = M.tid(), lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const float* C = M.tile(i, j) + 32 * w + l32;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc.m[q][r] = C[(long long)(32 * q + 8 * (r >> 2) + 4 * lh + (r & 3)) * M.ld];
            acc.a[q][r] = 0.f;
        }
    const int nc = K / FLOW_KC32;
    if (nc == 0) return;
    auto flush = [&] {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc.m[q][r] -= acc.a[q][r];
                acc.a[q][r] = 0.f;
            }
    };
    auto need = [](int c) { return c * FLOW_KC32 / CHOL_NB + 1; };
    if constexpr (SPLIT) {
        // [0] hi, [1] lo of tile row j; [2] hi, [3] lo of tile row i; row-major (row, k pairs)
        unsigned (*sH)[FLOW_T][SY_HP] = reinterpret_cast<unsigned (*)[FLOW_T][SY_HP]>(smem);
        const bool isI = tid >= FLOW_T;
        const int lrow = tid & (FLOW_T - 1);
        float v[FLOW_KC32];
        auto load = [&](int c) {
            const float* src = M.opnd(isI ? i : j, c * FLOW_KC32) + lrow;
#pragma unroll
            for (int k = 0; k < FLOW_KC32; ++k) v[k] = src[(long long)k * M.ld];
        };
        rd.wait(need(0));
        load(0);
        for (int c = 0; c < nc; ++c) {
            __syncthreads();
#pragma unroll
            for (int k = 0; k < FLOW_KC32; k += 8) {
                unsigned h[8], l[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) split_bf16(v[k + u], h[u], l[u]);
                *reinterpret_cast<uint4*>(&sH[isI ? 2 : 0][lrow][k / 2]) =
                    make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
                *reinterpret_cast<uint4*>(&sH[isI ? 3 : 1][lrow][k / 2]) =
                    make_uint4(l[0] | (l[1] << 16), l[2] | (l[3] << 16), l[4] | (l[5] << 16), l[6] | (l[7] << 16));
            }
            __syncthreads();
            const bool more = c + 1 < nc;
            const bool pre = more && rd.poll(need(c + 1));
            const int busy = quiet.busy();
            if (pre) load(c + 1);
#pragma unroll
            for (int t = 0; t < FLOW_KC32 / 16; ++t) {
                const int x = 8 * t + 4 * lh;   // lane holds k = 16 t + 8 lh + 0..7
                const bf16x8 bh = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&sH[2][32 * w + l32][x]));
                const bf16x8 bl = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&sH[3][32 * w + l32][x]));
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const bf16x8 ah = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&sH[0][32 * q + l32][x]));
                    const bf16x8 al = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&sH[1][32 * q + l32][x]));
                    acc.a[q] = mfma_bf16_32x32x16(al, bh, acc.a[q]);
                    acc.a[q] = mfma_bf16_32x32x16(ah, bl, acc.a[q]);
                    acc.a[q] = mfma_bf16_32x32x16(ah, bh, acc.a[q]);
                }
            }
            if (busy) quiet.pause();
            if (more && !pre) {
                rd.wait(need(c + 1));
                load(c + 1);
            }
            if ((c + 1) % (FLOW_FLUSH / FLOW_KC32) == 0 || !more) flush();
        }
        __syncthreads();
    } else {
        float (*st)[2][FLOW_KC32][FLOW_P32] = reinterpret_cast<float (*)[2][FLOW_KC32][FLOW_P32]>(smem);
        constexpr int NV = FLOW_KC32 * FLOW_T / 4 / 256;
        floatx4 vj[NV], vi[NV];
        auto load = [&](int c) {
            const float *pj = M.opnd(j, c * FLOW_KC32), *pi = M.opnd(i, c * FLOW_KC32);
#pragma unroll
            for (int u = 0; u < NV; ++u) {
                const int idx = tid + 256 * u, k = idx / (FLOW_T / 4), r = (idx % (FLOW_T / 4)) * 4;
                vj[u] = *reinterpret_cast<const floatx4*>(pj + (long long)k * M.ld + r);
                vi[u] = *reinterpret_cast<const floatx4*>(pi + (long long)k * M.ld + r);
            }
        };
        auto store = [&](int b) {
#pragma unroll
            for (int u = 0; u < NV; ++u) {
                const int idx = tid + 256 * u, k = idx / (FLOW_T / 4), r = (idx % (FLOW_T / 4)) * 4;
                *reinterpret_cast<floatx4*>(&st[b][0][k][r]) = vj[u];
                *reinterpret_cast<floatx4*>(&st[b][1][k][r]) = vi[u];
            }
        };
        rd.wait(need(0));
        load(0);
        store(0);
        __syncthreads();
        for (int c = 0; c < nc; ++c) {
            const bool more = c + 1 < nc;
            const bool pre = more && rd.poll(need(c + 1));
            const int busy = quiet.busy();
            if (pre) load(c + 1);
            float (*sj)[FLOW_P32] = st[c & 1][0], (*si)[FLOW_P32] = st[c & 1][1];
            float a[2][4], b[2];
            auto fetch = [&](int s) {
                b[s & 1] = si[2 * s + lh][32 * w + l32];
#pragma unroll
                for (int q = 0; q < 4; ++q) a[s & 1][q] = sj[2 * s + lh][32 * q + l32];
            };
            fetch(0);
#pragma unroll
            for (int s = 0; s < FLOW_KC32 / 2; ++s) {
                if (s + 1 < FLOW_KC32 / 2) fetch(s + 1);
#pragma unroll
                for (int q = 0; q < 4; ++q) acc.a[q] = mfma_f32_32x32x2(a[s & 1][q], b[s & 1], acc.a[q]);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (busy) quiet.pause();
            if (more) {
                if (!pre) {
                    rd.wait(need(c + 1));
                    load(c + 1);
                }
                store((c + 1) & 1);
            }
            if ((c + 1) % (FLOW_FLUSH / FLOW_KC32) == 0 || !more) flush();
            __syncthreads();
        }
    }
}

template <bool SPLIT, bool LOOP>
__device__ __forceinline__ void flow_accumulate(const FlowMat<double, LOOP>& M, int i, int j, int K, FlowReady& rd,
                                                const FlowQuiet& quiet, unsigned char* smem, FlowAcc<double>& acc)
{
    const int tid = M.tid(), lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lq = lane >> 4;
    double* C = M.tile(i, j) + 32 * w;
    const int nc = K / FLOW_KC64;
#pragma unroll
    for (int J = 0; J < 8; ++J)
#pragma unroll
        for (int g = 0; g < 2; ++g) acc.a[J][g] = doublex4{0.0, 0.0, 0.0, 0.0};
    // acc -= C, the loads of four blocks in flight together
    auto less_c = [&] {
        const FlowLane at(M.ld);
#pragma unroll
        for (int J0 = 0; J0 < 8; J0 += 4) {
            double v[4][4][2];
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int g = 0; g < 2; ++g) v[x][r][g] = *at(C, 16 * (J0 + x) + 4 * r, 16 * g);
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int g = 0; g < 2; ++g) acc.a[J0 + x][g][r] -= v[x][r][g];
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // C -= acc, two blocks at a time (more of them spill); acc starts anew
    auto fold = [&] {
        const FlowLane at(M.ld);
#pragma unroll
        for (int J = 0; J < 8; ++J) {
            double v[4][2];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int g = 0; g < 2; ++g) v[r][g] = *at(C, 16 * J + 4 * r, 16 * g);
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    *at(C, 16 * J + 4 * r, 16 * g) = v[r][g] - acc.a[J][g][r];
                    acc.a[J][g][r] = 0.0;
                }
            if (J & 1) __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (nc == 0) {
        less_c();
        return;
    }
    auto need = [](int c) { return c * FLOW_KC64 / CHOL_NB + 1; };
    double (*st)[2][FLOW_KC64][FLOW_P64] = reinterpret_cast<double (*)[2][FLOW_KC64][FLOW_P64]>(smem);
    constexpr int NV = FLOW_KC64 * FLOW_T / 2 / 256;
    doublex2 vj[NV], vi[NV];
    auto load = [&](int c) {
        const double *pj = M.opnd(j, c * FLOW_KC64), *pi = M.opnd(i, c * FLOW_KC64);
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int idx = tid + 256 * u, k = idx / (FLOW_T / 2), r = (idx % (FLOW_T / 2)) * 2;
            vj[u] = *reinterpret_cast<const doublex2*>(pj + (long long)k * M.ld + r);
            vi[u] = *reinterpret_cast<const doublex2*>(pi + (long long)k * M.ld + r);
        }
    };
    auto store = [&](int b) {
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int idx = tid + 256 * u, k = idx / (FLOW_T / 2), r = (idx % (FLOW_T / 2)) * 2;
            *reinterpret_cast<doublex2*>(&st[b][0][k][r]) = vj[u];
            *reinterpret_cast<doublex2*>(&st[b][1][k][r]) = vi[u];
        }
    };
    rd.wait(need(0));
    load(0);
    store(0);
    __syncthreads();
    for (int c = 0; c < nc; ++c) {
        const bool more = c + 1 < nc;
        const bool pre = more && rd.poll(need(c + 1));
        const int busy = quiet.busy();
        if (pre) load(c + 1);
        double (*sj)[FLOW_P64] = st[c & 1][0], (*si)[FLOW_P64] = st[c & 1][1];
        double a[2][8], b[2][2];
        auto fetch = [&](int s) {
            const int k = 4 * s + lq;
#pragma unroll
            for (int g = 0; g < 2; ++g) b[s & 1][g] = si[k][32 * w + 16 * g + lr];
#pragma unroll
            for (int J = 0; J < 8; ++J) a[s & 1][J] = sj[k][16 * J + lr];
        };
        fetch(0);
#pragma unroll
        for (int s = 0; s < FLOW_KC64 / 4; ++s) {
            if (s + 1 < FLOW_KC64 / 4) fetch(s + 1);
#pragma unroll
            for (int J = 0; J < 8; ++J)
#pragma unroll
                for (int g = 0; g < 2; ++g) acc.a[J][g] = mfma_f64_16x16x4(a[s & 1][J], b[s & 1][g], acc.a[J][g]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (more && (c + 1) % (FLOW_FLUSH / FLOW_KC64) == 0) fold();
        if (busy) quiet.pause();
        if (more) {
            if (!pre) {
                rd.wait(need(c + 1));
                load(c + 1);
            }
            store((c + 1) & 1);
        }
        __syncthreads();
    }
    less_c();
}

// z = sum - C in FP64, z[J][g][r] = column 16 J + 4 r + l/16, row 16 g + l%16 of the wavefront's 32
// rows.  FP32: through the wavefront's own part of the LDS at sc (2048 floats).
__device__ __forceinline__ void flow_negated(const FlowAcc<double>& acc, float*, doublex4 (&z)[8][2])
{
#pragma unroll
    for (int J = 0; J < 8; ++J)
#pragma unroll
        for (int g = 0; g < 2; ++g) z[J][g] = acc.a[J][g];
}
__device__ __forceinline__ void flow_negated(const FlowAcc<float>& acc, float* __restrict__ sc, doublex4 (&z)[8][2])
{
    const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4, l32 = lane & 31, lh = lane >> 5;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                sc[(32 * q + 8 * (r >> 2) + 4 * lh + (r & 3)) * 32 + l32] = acc.m[2 * h + q][r];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int J = 0; J < 4; ++J)
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int r = 0; r < 4; ++r) z[4 * h + J][g][r] = -(double)sc[(16 * J + 4 * r + lq) * 32 + 16 * g + lr];
        __builtin_amdgcn_wave_barrier();
    }
}

// X L_kk^T = -z for G groups of 16 rows on one wavefront, X over z: transposed, X_J^T = -Linv_J
// (z_J^T + sum_K L_JK X_K^T), so a finished block's accumulators (column 4 r + l/16, row l%16) are
// the next product's operands as they are (k = 4 s + l/16 of row l%16), and only L comes from the
// LDS.  sLT[k * 64 + c] = L_kk[c][k]; sInv[SINV J + c' * SINV_P + c] = Linv_JJ[c][c'].
template <int G, int Z>
__device__ __forceinline__ void flow_solve64(doublex4 (&z)[Z][G], int J0, const double* __restrict__ sLT,
                                             const double* __restrict__ sInv)
{
    const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4;
#pragma unroll
    for (int J = 0; J < 4; ++J) {
#pragma unroll
        for (int K = 0; K < J; ++K)
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) {
                const double a = sLT[(16 * K + 4 * s4 + lq) * CHOL_NB + 16 * J + lr];
#pragma unroll
                for (int g = 0; g < G; ++g) z[J0 + J][g] = mfma_f64_16x16x4(a, z[J0 + K][g][s4], z[J0 + J][g]);
            }
        doublex4 x[G];
#pragma unroll
        for (int g = 0; g < G; ++g) x[g] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
            const double a = sInv[SINV * J + (4 * s4 + lq) * SINV_P + lr];
#pragma unroll
            for (int g = 0; g < G; ++g) x[g] = mfma_f64_16x16x4(a, z[J0 + J][g][s4], x[g]);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) z[J0 + J][g] = -x[g];
    }
}

// Blocks J0 .. J0 + 3 of z (X): their operand copy, published as panel 2 j + J0 / 4 of tile row i,
// then the tile (i, j) itself, which nobody waits for (stored before the flag it cost the chain
// 0.4 us a panel in FP64).
template <typename T, bool LOOP>
__device__ __forceinline__ void flow_store(const FlowMat<T, LOOP>& M, int i, int j, int J0, const doublex4 (&z)[8][2])
{
    const int lane = M.tid() & 63, lr = lane & 15, lq = lane >> 4;
    const int row = 32 * (M.tid() >> 6) + lr;
    T* o = const_cast<T*>(M.opnd(i, FLOW_T * j)) + row;   // columns of tile column j: ld apart, as in the tile
    T* t = M.tile(i, j) + row;
#pragma unroll
    for (int J = 0; J < 4; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const long long col = (long long)(16 * (J0 + J) + 4 * r + lq) * M.ld;
#pragma unroll
            for (int g = 0; g < 2; ++g) st_agent(o + col + 16 * g, (T)z[J0 + J][g][r]);
        }
    flow_publish(M.rdy(i), 2 * j + J0 / 4 + 1);
#pragma unroll
    for (int J = 0; J < 4; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const long long col = (long long)(16 * (J0 + J) + 4 * r + lq) * M.ld;
#pragma unroll
            for (int g = 0; g < 2; ++g) t[col + 16 * g] = (T)z[J0 + J][g][r];
        }
}

template <typename T, bool SPLIT, bool LOOP>
__device__ __forceinline__ void flow_tile(const FlowMat<T, LOOP>& M, int i, int j, unsigned char* smem)
{
    double* s0 = reinterpret_cast<double*>(smem);   // diagonal block
    double* s1 = s0 + LB_STRIDE;                    // L21
    const int tid = M.tid(), lane = tid & 63, lr = lane & 15, lq = lane >> 4;
    doublex4 z[8][2];
    FlowQuiet quiet(i == j + 1 ? M.quiet : nullptr);
    {
        FlowAcc<T> acc;
        FlowReady rd{M.rdy(i), M.rdy(j), M.status};
        flow_accumulate<SPLIT>(M, i, j, FLOW_T * j, rd, FlowQuiet(i == j + 1 ? nullptr : M.quiet), smem, acc);   // ends with a barrier
        quiet.add(1);   // all of row j is published: tile (j, j) is past its accumulation or about to be
        flow_negated(acc, reinterpret_cast<float*>(s1) + 2048 * (tid >> 6), z);
    }
    const double* ws = M.ws + (long long)j * FLOW_COL;
    int have = flow_wait(M.dprog(j), 1, M.status);
    __syncthreads();   // s1 is free
    {
        constexpr int N1 = CHOL_NB * CHOL_NB / 256;
        double v[N1];
#pragma unroll
        for (int u = 0; u < N1; ++u) v[u] = ws[LB_STRIDE + tid + 256 * u];
        load_lkk(ws, s0);   // ends with a barrier
#pragma unroll
        for (int u = 0; u < N1; ++u) s1[tid + 256 * u] = v[u];
    }
    flow_solve64<2>(z, 0, s0, s0 + CHOL_NB * CHOL_NB);
    flow_store(M, i, j, 0, z);   // with a barrier: s1 is complete, s0 free
    // z_2 += L21 X_1^T; FP64 as a sum of its own, like the partial sums before
    constexpr int NJ = sizeof(T) == 8 ? 2 : 4;
#pragma unroll
    for (int J0 = 4; J0 < 8; J0 += NJ) {
        doublex4 y[NJ][2];
#pragma unroll
        for (int J = 0; J < NJ; ++J)
#pragma unroll
            for (int g = 0; g < 2; ++g) y[J][g] = sizeof(T) == 8 ? doublex4{0.0, 0.0, 0.0, 0.0} : z[J0 + J][g];
#pragma unroll
        for (int K = 0; K < 4; ++K)
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
                for (int J = 0; J < NJ; ++J) {
                    const double a = s1[(16 * K + 4 * s4 + lq) * CHOL_NB + 16 * (J0 - 4 + J) + lr];
#pragma unroll
                    for (int g = 0; g < 2; ++g) y[J][g] = mfma_f64_16x16x4(a, z[K][g][s4], y[J][g]);
                }
#pragma unroll
        for (int J = 0; J < NJ; ++J)
#pragma unroll
            for (int g = 0; g < 2; ++g) z[J0 + J][g] = sizeof(T) == 8 ? z[J0 + J][g] + y[J][g] : y[J][g];
    }
    if (have < 2) flow_wait(M.dprog(j), 2, M.status);
    load_lkk(ws + LB_STRIDE + CHOL_NB * CHOL_NB, s0);
    flow_solve64<2>(z, 4, s0, s0 + CHOL_NB * CHOL_NB);
    flow_store(M, i, j, 4, z);
    quiet.add(-1);
}

// One 32x32 block of a diagonal tile on one wavefront, transposed as in FlowAcc: columns 32 mb ..,
// rows 32 nb .. of the tile at t.  a is the partial sum; C - sum is in m, in FP64 from hold() on and
// in the tile's entries before (three blocks a wavefront have no registers for both).
template <typename T>
struct FlowQuad;
template <>
struct FlowQuad<float> {
    floatx16 m, a;
    __device__ void init(const float* t, long long ld, int mb, int nb, int lane)
    {
        const float* C = t + 32 * nb + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            m[r] = C[(long long)(32 * mb + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * ld];
            a[r] = 0.f;
        }
    }
    __device__ void hold(const float*, long long, int, int) {}
    __device__ void flush(float*, long long, int, int)
    {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            m[r] -= a[r];
            a[r] = 0.f;
        }
    }
    // rows k0 .. of s (pitch P): the k-th holds column k of the 128 (or 64) rows
    template <int KC, typename S>
    __device__ void mac(const S* s, int P, int mb, int nb, int lane)
    {
        const int l32 = lane & 31, lh = lane >> 5;
#pragma unroll 8
        for (int k = 0; k < KC; k += 2)
            a = mfma_f32_32x32x2((float)s[(k + lh) * P + 32 * mb + l32], (float)s[(k + lh) * P + 32 * nb + l32], a);
    }
    // K = 64 columns straight from memory
    __device__ void mac_global(const float* p, long long ld, int mb, int nb)
    {
        floatx16 t;
        quad_acc(p, ld, 32 * mb, 32 * nb, CHOL_NB, t);
        a += t;
    }
    template <typename F>
    __device__ void each(int lane, F&& f)
    {
#pragma unroll
        for (int r = 0; r < 16; ++r) f(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), lane & 31, (double)(m[r] - a[r]));
    }
};
template <>
struct FlowQuad<double> {
    doublex4 a[2][2], m[2][2];
    __device__ void init(const double*, long long, int, int, int)
    {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) a[x][y] = doublex4{0.0, 0.0, 0.0, 0.0};
    }
    __device__ void hold(double* t, long long ld, int mb, int nb)
    {
        const FlowLane at(ld);
        t += 32 * mb * ld + 32 * nb;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int r = 0; r < 4; ++r) m[x][y][r] = *at(t, 16 * x + 4 * r, 16 * y);
    }
    __device__ void flush(double* t, long long ld, int mb, int nb)
    {
        hold(t, ld, mb, nb);
        const FlowLane at(ld);
        t += 32 * mb * ld + 32 * nb;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
#pragma unroll
                for (int r = 0; r < 4; ++r) *at(t, 16 * x + 4 * r, 16 * y) = m[x][y][r] - a[x][y][r];
                a[x][y] = doublex4{0.0, 0.0, 0.0, 0.0};
            }
        __builtin_amdgcn_sched_barrier(0);
    }
    template <int KC, typename S>
    __device__ void mac(const S* s, int P, int mb, int nb, int lane)
    {
        const int lr = lane & 15, lq = lane >> 4;
#pragma unroll 4
        for (int k = 0; k < KC; k += 4) {
            double u[2], v[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                u[x] = s[(k + lq) * P + 32 * mb + 16 * x + lr];
                v[x] = s[(k + lq) * P + 32 * nb + 16 * x + lr];
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) a[x][y] = mfma_f64_16x16x4(u[x], v[y], a[x][y]);
        }
    }
    __device__ void mac_global(const double* p, long long ld, int mb, int nb)
    {
        doublex4 t[2][2];
        quad_acc(p, ld, 32 * mb, 32 * nb, CHOL_NB, t);
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) a[x][y] += t[x][y];
    }
    template <typename F>
    __device__ void each(int lane, F&& f)
    {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int r = 0; r < 4; ++r) f(16 * x + 4 * r + (lane >> 4), 16 * y + (lane & 15), m[x][y][r] - a[x][y][r]);
    }
};

// Diagonal tile j.  Its ten 32x32 blocks of the lower triangle lie on the wavefronts as (column
// block, row block)
//   wavefront 0: (0,0)           1: (0,1) (0,2) (2,2)    2: (1,1) (0,3) (2,3)    3: (1,2) (1,3) (3,3)
// so that the update that precedes each diagonal block's factor, the last step of the chain, is
// one block per wavefront: the last 64 columns are applied to the first diagonal block from the
// LDS, to the others by wavefronts 1 .. 3 while wavefront 0 factors it.
template <typename T, bool LOOP>
__device__ __forceinline__ void flow_diag(const FlowMat<T, LOOP>& M, int j, unsigned char* smem)
{
    constexpr int KC = sizeof(T) == 4 ? FLOW_KC32 : FLOW_KC64;
    constexpr int P = sizeof(T) == 4 ? FLOW_P32 : FLOW_P64;
    constexpr int V = 16 / sizeof(T);   // entries of one 16-byte access
    const int tid = M.tid(), lane = tid & 63, lr = lane & 15, lq = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    double* s0 = reinterpret_cast<double*>(smem);
    double* s1 = s0 + LB_STRIDE;
    double* ws = M.ws + (long long)j * FLOW_COL;
    T* tl = M.tile(j, j);
    const int c0 = FLOW_T * j;
    const bool second = c0 + CHOL_NB < M.n;   // else the second block is identity padding
    const int m0 = w == 2 || w == 3 ? 1 : 0, n0 = w == 0 ? 0 : (w == 3 ? 2 : 1);
    const int m1 = w == 3 ? 1 : 0, n1 = w == 1 ? 2 : 3;
    const int m2 = w == 3 ? 3 : 2, n2 = w == 1 ? 2 : 3;
    FlowQuiet quiet(M.quiet);
    FlowQuad<T> q0, q1, q2;
    q0.init(tl, M.ld, m0, n0, lane);
    if (w) {
        q1.init(tl, M.ld, m1, n1, lane);
        q2.init(tl, M.ld, m2, n2, lane);
    }
    if (j > 0) {
        FlowReady rd{M.rdy(j), M.rdy(j), M.status};
        const int nc = (FLOW_T * j - CHOL_NB) / KC;
        auto need = [](int c) { return c * KC / CHOL_NB + 1; };
        T (*st)[KC][P] = reinterpret_cast<T (*)[KC][P]>(smem);
        constexpr int NV = KC * FLOW_T / V / 256;
        typedef T vec __attribute__((ext_vector_type(V)));
        vec v[NV];
        auto load = [&](int c) {
            const T* p = M.opnd(j, c * KC);
#pragma unroll
            for (int u = 0; u < NV; ++u) {
                const int idx = tid + 256 * u, k = idx / (FLOW_T / V), r = (idx % (FLOW_T / V)) * V;
                v[u] = *reinterpret_cast<const vec*>(p + (long long)k * M.ld + r);
            }
        };
        auto store = [&](int b) {
#pragma unroll
            for (int u = 0; u < NV; ++u) {
                const int idx = tid + 256 * u, k = idx / (FLOW_T / V), r = (idx % (FLOW_T / V)) * V;
                *reinterpret_cast<vec*>(&st[b][k][r]) = v[u];
            }
        };
        rd.wait(need(0));
        load(0);
        store(0);
        __syncthreads();
        for (int c = 0; c < nc; ++c) {
            const bool more = c + 1 < nc;
            const bool pre = more && rd.poll(need(c + 1));
            if (pre) load(c + 1);
            const T* s = &st[c & 1][0][0];
            q0.template mac<KC>(s, P, m0, n0, lane);
            if (w) {
                q1.template mac<KC>(s, P, m1, n1, lane);
                q2.template mac<KC>(s, P, m2, n2, lane);
            }
            if (more) {
                if (!pre) {
                    rd.wait(need(c + 1));
                    load(c + 1);
                }
                store((c + 1) & 1);
            }
            // (the last part stays apart in FP64, where it costs a pass over memory)
            if ((c + 1) % (FLOW_FLUSH / KC) == 0 ? more || sizeof(T) == 4 : !more && sizeof(T) == 4) {
                q0.flush(tl, M.ld, m0, n0);
                if (w) {
                    q1.flush(tl, M.ld, m1, n1);
                    q2.flush(tl, M.ld, m2, n2);
                }
            }
            __syncthreads();
        }
        // the last 64 columns of rows 0 .. 63 through s1
        quiet.add(1);   // tile (j, j - 1) has published its first panel
        q0.hold(tl, M.ld, m0, n0);
        rd.wait(2 * j);
        constexpr int NL = CHOL_NB * CHOL_NB / V / 256;
        vec x[NL];
        const T* p = M.opnd(j, FLOW_T * j - CHOL_NB);
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            const int idx = tid + 256 * u, k = idx / (CHOL_NB / V), r = (idx % (CHOL_NB / V)) * V;
            x[u] = *reinterpret_cast<const vec*>(p + (long long)k * M.ld + r);
        }
        T* sl = reinterpret_cast<T*>(s1);
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            const int idx = tid + 256 * u, k = idx / (CHOL_NB / V), r = (idx % (CHOL_NB / V)) * V;
            *reinterpret_cast<vec*>(sl + k * CHOL_NB + r) = x[u];
        }
        __syncthreads();
        if (w < 3) q0.template mac<CHOL_NB>(sl, CHOL_NB, m0, n0, lane);
    } else {
        q0.hold(tl, M.ld, m0, n0);
    }
    auto to_block = [&](FlowQuad<T>& q, int mb, int nb) {
        q.each(lane, [&](int c, int r, double v) { s0[(32 * nb + r) * DG_LD + 32 * mb + c] = v; });
    };
    auto to_lower = [&](FlowQuad<T>& q, int mb, int nb) {
        q.each(lane, [&](int c, int r, double v) { s1[(32 * mb + c) * CHOL_NB + 32 * (nb - 2) + r] = v; });
    };
    if (w < 3) to_block(q0, m0, n0);
    factor_diag64(s0, c0, M.status, [&] {   // begins with a barrier
        if (!second) return;
        const T* p = j > 0 ? M.opnd(j, FLOW_T * j - CHOL_NB) : nullptr;
        if constexpr (sizeof(T) == 8) {
            // one block at a time: together their operands spill
            if (w == 3) {
                if (p) q0.mac_global(p, M.ld, m0, n0);
                to_lower(q0, m0, n0);
            }
            if (p) q1.mac_global(p, M.ld, m1, n1);
            q1.hold(tl, M.ld, m1, n1);
            if (p) q2.mac_global(p, M.ld, m2, n2);
            to_lower(q1, m1, n1);
        } else {
            // all of the loads ahead of the sums: one block at a time n = 768 takes 197 us instead of 187
            if (p) {
                if (w == 3) q0.mac_global(p, M.ld, m0, n0);
                q1.mac_global(p, M.ld, m1, n1);
                q2.mac_global(p, M.ld, m2, n2);
            }
            if (w == 3) to_lower(q0, m0, n0);
            to_lower(q1, m1, n1);
        }
    });
    store_lkk(s0, ws);
    if (!second) {
        store_diag64<T>(s0, tl, M.ld, 0);
        if (j > 0) quiet.add(-1);
        return;
    }
    // L21: 16 rows per wavefront
    doublex4 z[4][1];
#pragma unroll
    for (int J = 0; J < 4; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) z[J][0][r] = -s1[(16 * J + 4 * r + lq) * CHOL_NB + 16 * w + lr];
    flow_solve64<1>(z, 0, s0, s0 + CHOL_NB * CHOL_NB);
#pragma unroll
    for (int J = 0; J < 4; ++J)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = 16 * J + 4 * r + lq, row = 16 * w + lr;
            s1[c * CHOL_NB + row] = z[J][0][r];
            st_agent(ws + LB_STRIDE + c * CHOL_NB + row, z[J][0][r]);
            tl[(long long)c * M.ld + CHOL_NB + row] = (T)z[J][0][r];
        }
    __syncthreads();   // L21 in s1; s0 is free
    if (w) {
        if constexpr (sizeof(T) == 4) q2.flush(tl, M.ld, m2, n2);
        q2.hold(tl, M.ld, m2, n2);
        q2.template mac<CHOL_NB>(s1, CHOL_NB, m2 - 2, n2 - 2, lane);
        to_block(q2, m2 - 2, n2 - 2);
    }
    flow_publish(M.dprog(j), 1);
    factor_diag64(s0, c0 + CHOL_NB, M.status, [&] {
        // L11 into the tile
        for (int e = tid - 64; e < CHOL_NB * CHOL_NB; e += 192) {
            const int r = e % CHOL_NB, c = e / CHOL_NB;
            if (r >= c) tl[(long long)c * M.ld + r] = (T)ws[e];
        }
    });
    store_lkk(s0, ws + LB_STRIDE + CHOL_NB * CHOL_NB);
    flow_publish(M.dprog(j), 2);
    if (j > 0) quiet.add(-1);
    store_diag64<T>(s0, tl, M.ld, CHOL_NB);
}

// The next index of the counter, for the workgroup.
__device__ __forceinline__ int flow_task(int* __restrict__ next)
{
    __shared__ int s_task;
    if (threadIdx.x == 0) s_task = __hip_atomic_fetch_add(next, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();   // and the LDS of the task before is free
    return __builtin_amdgcn_readfirstlane(s_task);
}

// The tasks of a batch in the order of the counter.  With more of them than workgroups fit on the
// chip, workgroups stay and take another: left to the dispatcher, which places workgroups in order
// and waits for room in the shader engine whose turn it is, a sixth of the places stood empty (256
// chains of 64 .. 1024 beads FP32: 3.64 -> 3.39 ms).  One matrix keeps a workgroup per tile: its
// columns end together, and the loop's extra instructions lie on its chain (n = 9000 FP32 2.79 ms,
// 2.98 with the loop, FP64 4.94 and 5.27, both before FP64 took its sums in parts).
constexpr int FLOW_PLACES = 512;   // two workgroups on each of 256 CUs
constexpr int FLOW_STEP = 10;      // 100 ns (in 100 MHz ticks), in which the counter serves eight workgroups
// A null counter: one task, no loop (with a loop in every case the compiler spills 30 to 50 registers).
template <typename Body>
__device__ __forceinline__ void flow_tasks(int* __restrict__ next, int count, Body&& body)
{
    for (;;) {
        const int x = next ? flow_task(next) : 0;
        if (x >= count) break;
        body(x);
        if (!next) break;
    }
}

template <typename T, bool SPLIT, bool LOOP>
__device__ __forceinline__ void flow_body(const FlowMat<T, LOOP>& M, int i, int j)
{
    __shared__ __align__(16) unsigned char smem[FLOW_SMEM];
    if (i == j) flow_diag(M, j, smem);
    else flow_tile<T, SPLIT>(M, i, j, smem);
}

template <typename T, bool SPLIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
chol_flow_kernel(FlowMat<T> M, int* __restrict__ next)
{
    // The first workgroups ask in the order of their index, one of each XCD at a time: all at once, the
    // counter serves one XCD after the other, and neighbouring tiles share an XCD and its CUs (FP64
    // n = 4500 1350 -> 1650 us).
    if (threadIdx.x == 0 && blockIdx.x < FLOW_PLACES) {
        const long long t0 = wall_clock64(), wait = (long long)(blockIdx.x / 8) * FLOW_STEP;
        while (wall_clock64() - t0 < wait) __builtin_amdgcn_s_sleep(1);
    }
    // tile column by column
    int x = flow_task(next), j = 0;
    while (x >= M.nt - j) {
        x -= M.nt - j;
        ++j;
    }
    flow_body<T, SPLIT>(M, j + x, j);
}

__global__ void chol_flow_clear_kernel(int* __restrict__ flags, int count)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) flags[i] = 0;
}

// d_status: 0, or the 1-based row of the first non-positive pivot; -1 after a timed-out wait.
template <typename T>
int chol_factor(T* d_A, long long ld, int n, int n_pad, double* d_Lbuf, int* d_status, int syrk_mode,
                hipStream_t st, PhaseRecorder* rec)
{
    BDH_CHECK(n_pad % PAD_TO == 0 && n <= n_pad && n > n_pad - PAD_TO, "chol_factor: n_pad must be n rounded up to 128");
    BDH_CHECK(ld >= n_pad && ld % 4 == 0, "chol_factor: bad leading dimension");
    BDH_CHECK(syrk_mode != SYRK_BF16X3 || sizeof(T) == 4, "chol_factor: split SYRK needs FP32 storage");
    const int nt = n_pad / FLOW_T;
    int* d_flags = reinterpret_cast<int*>(d_Lbuf + (long long)nt * FLOW_COL);
    int nflags = 2 * nt * FLAG_STRIDE;
    const int tiles = nt * (nt + 1) / 2;
    const bool shared = tiles > QUIET_TILES;
    FlowMat<T> M{d_A, ld, n, nt, d_Lbuf, d_status, shared ? d_flags + nflags : nullptr};
    if (shared) nflags += FLOW_CUS;
    int* next = d_flags + nflags;
    nflags += 1;
    if (rec) rec->begin(PH_PANEL, st);
    hipLaunchKernelGGL(chol_flow_clear_kernel, dim3(ceil_div(nflags, 256)), dim3(256), 0, st, d_flags, nflags);
    BDH_LAUNCH_CHECK();
    if (rec) rec->end(PH_PANEL, st);
    if (rec) rec->begin(PH_SYRK, st);
    const dim3 grid(tiles);
    if constexpr (sizeof(T) == 4) {
        if (syrk_mode == SYRK_BF16X3)
            hipLaunchKernelGGL((chol_flow_kernel<T, true>), grid, dim3(256), 0, st, M, next);
        else
            hipLaunchKernelGGL((chol_flow_kernel<T, false>), grid, dim3(256), 0, st, M, next);
    } else {
        hipLaunchKernelGGL((chol_flow_kernel<T, false>), grid, dim3(256), 0, st, M, next);
    }
    BDH_LAUNCH_CHECK();
    if (rec) rec->end(PH_SYRK, st);
    return 0;
}

size_t chol_lbuf_doubles(int n_pad)
{
    const size_t nt = n_pad / FLOW_T;
    return nt * FLOW_COL + (2 * nt * FLAG_STRIDE + FLOW_CUS + FLAG_STRIDE) / 2;   // flags, quiet counters, task counter
}

// ------------------------------------------------------------------ Y = L X (partials)
// X holds m right-hand sides (m <= M, X[k * ldx + c]): with L fixed between refactorizations,
// the noise of a whole refactor cycle is one pass over L instead of one per step.
// Tile: (64 lanes x V rows) x TRMV_COLS columns, V = 16 / sizeof(T) so each lane issues one
// 16-byte load per column; the 4 waves split the tile's columns and meet in LDS.  Entries above
// the diagonal are masked with a select after the load (the storage there is finite but
// meaningless), so diagonal tiles take the same vector path.  P[cb][k][r] receives row r's
// partial of right-hand side k over column block cb (FP64 products and accumulation).
//
// Bound: reading the lower triangle of L once.  The X values come four columns per scalar load
// (an index clamped to m - 1 instead of a condition: the sums beyond m are not stored), and the
// next columns of L are in flight during the sums.  With a condition around each X value, one
// load and one branch per value, and without loads ahead, ten right-hand sides took at n = 9000
// 70 us in FP32 and 89 in FP64; now 41 and 68 (162 and 324 MB: 3.9 and 4.7 TB/s).  One
// right-hand side at n = 768 in FP64: 8.0 -> 5.9 us.
constexpr int TRMV_COLS = 256;

template <typename T>
using trmv_vec = T __attribute__((ext_vector_type(16 / sizeof(T))));

// Column c's entries of a lane's V rows.  In a tile on the diagonal the lanes whose rows all
// lie above it read the diagonal's own entry again instead of memory that the sum masks out.
template <typename T, bool MASK>
__device__ __forceinline__ trmv_vec<T> trmv_load(const T* __restrict__ col, int rbase, int c)
{
    constexpr int V = 16 / sizeof(T);
    return *reinterpret_cast<const trmv_vec<T>*>(col + (MASK ? max(rbase, c & -V) : rbase));
}

template <typename T, int M, bool MASK>
__device__ __forceinline__ void trmv_accum(trmv_vec<T> w, int rbase, int c,
                                           const double* __restrict__ xc, double (*acc)[M])
{
    constexpr int V = 16 / sizeof(T);
#pragma unroll
    for (int q = 0; q < V; ++q) {
        const double v = (!MASK || rbase + q >= c) ? (double)w[q] : 0.0;
#pragma unroll
        for (int k = 0; k < M; ++k) acc[q][k] += v * xc[k];
    }
}

// One wavefront's columns c .. c_hi - 1 of a tile, UNR at a time; the next UNR columns' loads
// are in flight while these are summed.
template <typename T, int M, bool MASK>
__device__ __forceinline__ void trmv_columns(const T* __restrict__ L, long long ld, int rbase, int c,
                                             int c_hi, const double* __restrict__ X, long long ldx,
                                             int m, double (*acc)[M])
{
    constexpr int UNR = M >= 4 ? 4 : 8;
    trmv_vec<T> w[UNR];
    if (c + UNR <= c_hi) {
#pragma unroll
        for (int u = 0; u < UNR; ++u)
            w[u] = trmv_load<T, MASK>(L + (long long)(c + u) * ld, rbase, c + u);
    }
    for (; c + UNR <= c_hi; c += UNR) {
        trmv_vec<T> wn[UNR];
        // past the last whole group: this group's columns again, so the loads need no branch
        const int cn = c + 2 * UNR <= c_hi ? c + UNR : c;
#pragma unroll
        for (int u = 0; u < UNR; ++u)
            wn[u] = trmv_load<T, MASK>(L + (long long)(cn + u) * ld, rbase, cn + u);
        double xc[UNR][M];
#pragma unroll
        for (int u = 0; u < UNR; ++u)
#pragma unroll
            for (int k = 0; k < M; ++k) xc[u][k] = X[min(k, m - 1) * ldx + c + u];
#pragma unroll
        for (int u = 0; u < UNR; ++u) trmv_accum<T, M, MASK>(w[u], rbase, c + u, xc[u], acc);
        // without it the next group's loads are waited for before this group's sums
        if constexpr (M >= 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < UNR; ++u) w[u] = wn[u];
    }
    for (; c < c_hi; ++c) {
        double xc[M];
#pragma unroll
        for (int k = 0; k < M; ++k) xc[k] = X[min(k, m - 1) * ldx + c];
        trmv_accum<T, M, MASK>(trmv_load<T, MASK>(L + (long long)c * ld, rbase, c), rbase, c, xc, acc);
    }
}

// Right-hand sides K .. m - 1 of a tile: the four wavefronts' sums meet in alternate halves of
// s_red, one barrier each (every thread that passes it has read the half written next).  A
// recursion, since with k a variable the sums would have to be indexed at run time.
template <int K, int V, int M>
__device__ __forceinline__ void trmv_store(double (*acc)[M], int m, double (*s_red)[4][64 * V], int wave,
                                           int lane, double* __restrict__ P, int n, int r0)
{
    if constexpr (K < M) {
        if (K >= m) return;
        double(*red)[64 * V] = s_red[K & 1];
#pragma unroll
        for (int q = 0; q < V; ++q) red[wave][lane * V + q] = acc[q][K];
        __syncthreads();
        for (int rr = threadIdx.x; rr < 64 * V && r0 + rr < n; rr += 256)
            P[(long long)K * n + r0 + rr] = (red[0][rr] + red[1][rr]) + (red[2][rr] + red[3][rr]);
        trmv_store<K + 1, V, M>(acc, m, s_red, wave, lane, P, n, r0);
    }
}

template <typename T, int M>
__device__ __forceinline__ void trmv_partial_body(const T* __restrict__ L, long long ld, int n,
                                                  const double* __restrict__ X, long long ldx, int m,
                                                  double* __restrict__ P, int rb, int cb)
{
    constexpr int V = 16 / sizeof(T);
    constexpr int ROWS = 64 * V;
    const int r0 = rb * ROWS, cbeg = cb * TRMV_COLS;
    if (cbeg > r0 + ROWS - 1 || cbeg >= n) return;  // tile entirely above the diagonal
    __shared__ double s_red[2][4][ROWS];
    // the wavefront index is uniform: its columns, and so the X values, come through the
    // scalar cache into SGPRs instead of one vector load per lane
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rbase = r0 + lane * V;
    double acc[V][M];
#pragma unroll
    for (int q = 0; q < V; ++q)
#pragma unroll
        for (int k = 0; k < M; ++k) acc[q][k] = 0.0;
    const int wcols = TRMV_COLS / 4;
    // columns beyond the tile's last row hold nothing of the lower triangle
    const int cend = min(min(n, cbeg + TRMV_COLS), r0 + ROWS);
    const int c_lo = cbeg + wave * wcols, c_hi = min(cend, c_lo + wcols);
    // the whole tile is below the diagonal when its last column precedes its first row
    if (rbase < n) {
        if (cbeg + TRMV_COLS - 1 > r0)
            trmv_columns<T, M, true>(L, ld, rbase, c_lo, c_hi, X, ldx, m, acc);
        else
            trmv_columns<T, M, false>(L, ld, rbase, c_lo, c_hi, X, ldx, m, acc);
    }
    trmv_store<0, V, M>(acc, m, s_red, wave, lane, P + (long long)cb * m * n, n, r0);
}

template <typename T, int M>
__global__ void __launch_bounds__(256)
trmv_partial_kernel(const T* __restrict__ L, long long ld, int n, const double* __restrict__ X,
                    long long ldx, int m, double* __restrict__ P)
{
    trmv_partial_body<T, M>(L, ld, n, X, ldx, m, P, blockIdx.x, blockIdx.y);
}

int trmv_col_blocks(int n) { return ceil_div(n, TRMV_COLS); }

template <typename T>
int launch_trmv_partials(const T* d_L, long long ld, int n, const double* d_X, long long ldx, int m,
                         double* d_P, hipStream_t st)
{
    constexpr int ROWS = 64 * (16 / sizeof(T));
    BDH_CHECK(ld % (16 / sizeof(T)) == 0, "trmv: leading dimension not 16-byte aligned");
    BDH_CHECK(m >= 1 && m <= TRMV_MAX_RHS, "trmv: 1..16 right-hand sides");
    dim3 grid(ceil_div(n, ROWS), trmv_col_blocks(n));
    if (m == 1)
        hipLaunchKernelGGL((trmv_partial_kernel<T, 1>), grid, dim3(256), 0, st, d_L, ld, n, d_X, ldx, m, d_P);
    else if (m == 2)
        hipLaunchKernelGGL((trmv_partial_kernel<T, 2>), grid, dim3(256), 0, st, d_L, ld, n, d_X, ldx, m, d_P);
    else if (m <= 4)
        hipLaunchKernelGGL((trmv_partial_kernel<T, 4>), grid, dim3(256), 0, st, d_L, ld, n, d_X, ldx, m, d_P);
    else if (m <= 8)
        hipLaunchKernelGGL((trmv_partial_kernel<T, 8>), grid, dim3(256), 0, st, d_L, ld, n, d_X, ldx, m, d_P);
    else if (m <= 10)
        hipLaunchKernelGGL((trmv_partial_kernel<T, 10>), grid, dim3(256), 0, st, d_L, ld, n, d_X, ldx, m, d_P);
    else
        hipLaunchKernelGGL((trmv_partial_kernel<T, 16>), grid, dim3(256), 0, st, d_L, ld, n, d_X, ldx, m, d_P);
    BDH_LAUNCH_CHECK();
    return 0;
}

int trmv_blk_cols() { return TRMV_COLS; }

// ------------------------------------------------------------------ batches of matrices
template <typename T>
int trmv_blocks(int n)
{
    constexpr int ROWS = 64 * (16 / sizeof(T));
    return ceil_div(n, ROWS) * trmv_col_blocks(n);
}

// The tiles of every chain's matrix in one launch.  Key of a tile (i, j) of a matrix of nt tile
// rows: nt - j, the tile columns left on its chain of diagonal blocks; larger keys first, so the
// chains with the most columns left start first and all end together.  Among equal keys the
// diagonal tiles, then the tiles below them (the next on their chains), then the rest.  A tile
// waits for tiles of larger keys and for its own diagonal tile only, all of lower index.
std::vector<FlowTask> chol_batch_tasks(const std::vector<int>& n_pad)
{
    std::vector<FlowTask> t;
    int key = 0;
    for (int np : n_pad) key = std::max(key, np / FLOW_T);
    for (; key > 0; --key)
        for (int d = 0; d < 3; ++d)
            for (size_t c = 0; c < n_pad.size(); ++c) {
                const int nt = n_pad[c] / FLOW_T, j = nt - key;
                if (j < 0) continue;
                const int i0 = j + d, i1 = d < 2 ? std::min(nt, i0 + 1) : nt;
                for (int i = i0; i < i1; ++i) t.push_back(FlowTask{(int)c, (short)i, (short)j});
            }
    return t;
}

template <typename T>
__device__ __forceinline__ FlowMat<T, true> flow_mat(T* A, double* Lbuf, const BatchChain& b, int* status)
{
    return FlowMat<T, true>{A + b.mat, b.n_pad, b.n, b.n_pad / FLOW_T, Lbuf + b.lb, status, nullptr};
}

template <typename T, bool SPLIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
chol_flow_batch_kernel(T* __restrict__ A, double* __restrict__ Lbuf, const BatchChain* __restrict__ ch,
                       const FlowTask* __restrict__ tasks, int ntasks, int* __restrict__ next,
                       int* __restrict__ status)
{
    flow_tasks(next, ntasks, [&](int x) {
        const FlowTask t = tasks[x];
        flow_body<T, SPLIT>(flow_mat(A, Lbuf, ch[t.c], status + t.c), t.i, t.j);
    });
}

template <typename T>
__global__ void chol_flow_clear_batch_kernel(double* __restrict__ Lbuf, const BatchChain* __restrict__ ch,
                                             int* __restrict__ next)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *next = 0;
    const auto M = flow_mat((T*)nullptr, Lbuf, ch[blockIdx.x], nullptr);
    for (int x = threadIdx.x; x < 2 * M.nt * FLAG_STRIDE; x += blockDim.x) M.flags()[x] = 0;
}

template <typename T>
int chol_factor_batch(T* d_A, double* d_Lbuf, const BatchPlan& plan, int* d_status, int syrk_mode,
                      hipStream_t st, PhaseRecorder* rec)
{
    BDH_CHECK(syrk_mode != SYRK_BF16X3 || sizeof(T) == 4, "chol_factor_batch: split SYRK needs FP32 storage");
    BDH_CHECK(sizeof(T) == 8 || syrk_mode != SYRK_F64, "chol_factor_batch: FP32 storage needs an FP32 SYRK");
    if (rec) rec->begin(PH_PANEL, st);
    hipLaunchKernelGGL(chol_flow_clear_batch_kernel<T>, dim3(plan.nch), dim3(256), 0, st, d_Lbuf, plan.ch,
                       plan.next);
    BDH_LAUNCH_CHECK();
    if (rec) rec->end(PH_PANEL, st);
    if (rec) rec->begin(PH_SYRK, st);
    int* next = plan.ntasks > 1 ? plan.next : nullptr;
    const dim3 grid(std::min(plan.ntasks, FLOW_PLACES));
    if (sizeof(T) == 4 && syrk_mode == SYRK_BF16X3)
        hipLaunchKernelGGL((chol_flow_batch_kernel<T, sizeof(T) == 4>), grid, dim3(256), 0, st, d_A, d_Lbuf, plan.ch,
                           plan.tasks, plan.ntasks, next, d_status);
    else
        hipLaunchKernelGGL((chol_flow_batch_kernel<T, false>), grid, dim3(256), 0, st, d_A, d_Lbuf, plan.ch,
                           plan.tasks, plan.ntasks, next, d_status);
    BDH_LAUNCH_CHECK();
    if (rec) rec->end(PH_SYRK, st);
    return 0;
}

// At least four wavefronts a SIMD for up to ten right-hand sides (128 registers, five of them
// spilled in FP32): a batch has tiles for many rounds of workgroups, and their number in flight
// hides the tiles' starts and ends.  256 chains of 64 .. 1024 beads, ten sides, FP32: 278 us
// with the 133 registers the compiler takes by itself, 255 with 128; the launch of one matrix is
// a single round and measured 41 -> 46 us at n = 9000, so it keeps its registers.
template <typename T, int M>
__global__ void __launch_bounds__(256, M <= 10 ? 4 : 2)
trmv_batch_kernel(const T* __restrict__ A, const double* __restrict__ X, long long x_stride, int m,
                  const BatchChain* __restrict__ ch, const int* __restrict__ prefix, int nch,
                  double* __restrict__ Pt)
{
    constexpr int ROWS = 64 * (16 / sizeof(T));
    const int c = batch_find(prefix, nch, blockIdx.x);
    const BatchChain b = ch[c];
    const int x = blockIdx.x - prefix[c];
    const int gx = (b.n + ROWS - 1) / ROWS;
    const double* Xc = x_stride > 0 ? X + 3LL * b.bead0 : X + b.xi_off;
    const long long ldx = x_stride > 0 ? x_stride : b.ldx;
    trmv_partial_body<T, M>(A + b.mat, b.n_pad, b.n, Xc, ldx, m, Pt + b.pt, x % gx, x / gx);
}

template <typename T>
int launch_trmv_batch(const T* d_A, const double* d_X, long long x_stride, int m, const BatchPlan& plan,
                      double* d_Pt, hipStream_t st)
{
    BDH_CHECK(m >= 1 && m <= TRMV_MAX_RHS, "trmv: 1..16 right-hand sides");
    const dim3 grid(plan.trmv_blocks);
#define TB_LAUNCH(MM)                                                                              \
    hipLaunchKernelGGL((trmv_batch_kernel<T, MM>), grid, dim3(256), 0, st, d_A, d_X, x_stride, m, \
                       plan.ch, plan.trmv_pre, plan.nch, d_Pt)
    if (m == 1) TB_LAUNCH(1);
    else if (m == 2) TB_LAUNCH(2);
    else if (m <= 4) TB_LAUNCH(4);
    else if (m <= 8) TB_LAUNCH(8);
    else if (m <= 10) TB_LAUNCH(10);
    else TB_LAUNCH(16);
#undef TB_LAUNCH
    BDH_LAUNCH_CHECK();
    return 0;
}

template int chol_factor_batch<float>(float*, double*, const BatchPlan&, int*, int, hipStream_t, PhaseRecorder*);
template int chol_factor_batch<double>(double*, double*, const BatchPlan&, int*, int, hipStream_t, PhaseRecorder*);
template int launch_trmv_batch<float>(const float*, const double*, long long, int, const BatchPlan&, double*, hipStream_t);
template int launch_trmv_batch<double>(const double*, const double*, long long, int, const BatchPlan&, double*, hipStream_t);
template int trmv_blocks<float>(int);
template int trmv_blocks<double>(int);

template int chol_factor<float>(float*, long long, int, int, double*, int*, int, hipStream_t, PhaseRecorder*);
template int chol_factor<double>(double*, long long, int, int, double*, int*, int, hipStream_t, PhaseRecorder*);
template int launch_trmv_partials<float>(const float*, long long, int, const double*, long long, int, double*, hipStream_t);
template int launch_trmv_partials<double>(const double*, long long, int, const double*, long long, int, double*, hipStream_t);

}  // namespace bdh
