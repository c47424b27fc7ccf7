// Device reproduction of the reference's Gaussian stream.
//
// The reference draws its noise on the host: glibc drand48_r (48-bit LCG, a = 0x5DEECE66D,
// c = 0xB, value X / 2^48) feeding the polar Box-Muller method of gauss_rand
// (src/rand_move.c:132-168): attempt t consumes two uniforms, v = 2u - 1, accepts when
// 0 < v1^2 + v2^2 < 1, and an accepted pair yields (v2*fac, v1*fac) at table positions
// (2p, 2p+1); for an odd table length the last v1*fac is dropped (the pair state is local
// to the call).
//
// gauss_rounds: one workgroup draws from one stream (each of a batch's chains, a short call of a
// single stream, the remainder of a long one).  Each round, thread t jumps the LCG ahead to its
// chunk of K attempts (jump constants A^(2^b), C_b for b < 48 live in constant memory),
// evaluates them, and a workgroup scan of the accept counts gives every accepted attempt
// its pair index p.  The stream state after the call is the state after the attempt that
// produced the last needed pair -- so the integer stream is bit-identical to the host's,
// and repeated calls continue it exactly as repeated gauss_rand calls do.
// v1*v1 + v2*v2 and -2 log(rsq) / rsq are evaluated without FMA contraction, as the
// x86-64 reference does; the device log differs
// from glibc's by an ulp now and then, so Gaussian values agree to ~1e-15 while the
// integer stream (and so which attempts are accepted) is identical.
#include <algorithm>
#include <type_traits>

#include "bdh_common.hpp"
#include "bdh_kernels.hpp"

namespace bdh {

namespace {

constexpr uint64_t LCG_A = 0x5DEECE66DULL;
constexpr uint64_t LCG_C = 0xBULL;
constexpr uint64_t MASK48 = (1ULL << 48) - 1;

__constant__ uint64_t c_jumpA[48];
__constant__ uint64_t c_jumpC[48];

constexpr int RNG_THREADS = 1024;

__device__ __forceinline__ uint64_t lcg_step(uint64_t x) { return (LCG_A * x + LCG_C) & MASK48; }

__device__ __forceinline__ uint64_t lcg_jump(uint64_t x, uint64_t k)
{
    for (int b = 0; k; ++b, k >>= 1)
        if (k & 1) x = (c_jumpA[b] * x + c_jumpC[b]) & MASK48;
    return x;
}

__device__ __forceinline__ double u48(uint64_t x) { return (double)x * 0x1p-48; }

// log(r) for r in (0.5, 1) with small relative error as log(r) -> 0:
// log(1 + d) = 2 atanh(s), s = d / (2 + d), d = r - 1 exact (Sterbenz); |s| < 1/3 so the
// odd series 2 s (1 + s^2/3 + s^4/5 + ...) is summed to 20 terms (s^40/41 < 1e-20).
__device__ __forceinline__ double log_near_one(double r)
{
#pragma clang fp contract(off)
    const double d = r - 1.0;
    const double s = d / (2.0 + d);
    const double s2 = s * s;
    double p = 1.0 / 41.0;
#pragma unroll
    for (int k = 19; k >= 0; --k) p = 1.0 / (2 * k + 1) + s2 * p;
    return (2.0 * s) * p;
}

// The K attempts from state x on: uniforms, rsq; returns the accept count.
template <int K>
__device__ __forceinline__ int gauss_attempts(uint64_t x, double (&v1)[K], double (&v2)[K], double (&rsq)[K])
{
    // no FMA contraction in these functions (the pragma covers only expressions written
    // here, not inlined helpers): v1*v1 + v2*v2 must round exactly as on the host
#pragma clang fp contract(off)
    int acc = 0;
#pragma unroll
    for (int q = 0; q < K; ++q) {
        x = lcg_step(x);
        v1[q] = 2.0 * u48(x) - 1.0;
        x = lcg_step(x);
        v2[q] = 2.0 * u48(x) - 1.0;
        rsq[q] = v1[q] * v1[q] + v2[q] * v2[q];
        acc += (rsq[q] < 1.0 && rsq[q] != 0.0);
    }
    return acc;
}

// The accepted attempts' pairs p, p + 1, .. below npairs into o; last(q) for attempt q that gives
// the last pair.
template <int K, typename Last>
__device__ __forceinline__ void gauss_pairs(const double (&v1)[K], const double (&v2)[K], const double (&rsq)[K],
                                            long long p, long long npairs, long long count, double* __restrict__ o,
                                            Last&& last)
{
#pragma clang fp contract(off)
#pragma unroll
    for (int q = 0; q < K; ++q) {
        if (rsq[q] < 1.0 && rsq[q] != 0.0) {
            if (p < npairs) {
                // near 1 the library log is accurate only in absolute terms; the series
                // keeps the relative error at the ulp level where log(rsq) -> 0
                const double lg = rsq[q] > 0.5 ? log_near_one(rsq[q]) : log(rsq[q]);
                double fac = sqrt(-2.0 * lg / rsq[q]);
                o[2 * p] = v2[q] * fac;
                if (2 * p + 1 < count) o[2 * p + 1] = v1[q] * fac;
                if (p == npairs - 1) last(q);
            }
            ++p;
        }
    }
}

// Inclusive sum over the lanes of a wavefront.
__device__ __forceinline__ int wave_scan(int v)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) {
        const int u = __shfl_up(v, w);
        if (lane >= w) v += u;
    }
    return v;
}

// `count` values of the stream at `base` into o by one workgroup; returns the state after them.
template <int THREADS, int K>
__device__ __forceinline__ uint64_t gauss_rounds(uint64_t base, double* __restrict__ o, long long count,
                                                 int* __restrict__ status, int (&s_wave)[THREADS / 64],
                                                 long long& s_last)
{
    const int t = threadIdx.x, wave = t >> 6;
    const long long npairs = (count + 1) / 2;
    long long produced = 0;
    for (int round = 0; produced < npairs; ++round) {
        if (round > 1 << 20) {  // cannot happen (acceptance pi/4); keeps the loop finite
            if (t == 0) status[0] = 1;
            break;
        }
        double v1[K], v2[K], rsq[K];
        const int acc = gauss_attempts<K>(lcg_jump(base, 2ull * (uint64_t)t * K), v1, v2, rsq);
        const int incl = wave_scan(acc);
        if ((t & 63) == 63) s_wave[wave] = incl;
        __syncthreads();
        int before = 0, total = 0;
#pragma unroll
        for (int w = 0; w < THREADS / 64; ++w) {
            before += w < wave ? s_wave[w] : 0;
            total += s_wave[w];
        }
        gauss_pairs<K>(v1, v2, rsq, produced + before + incl - acc, npairs, count, o,
                       [&](int q) { s_last = (long long)t * K + q; });   // index within the round
        __syncthreads();
        if (produced + total >= npairs) {
            base = lcg_jump(base, 2ull * (uint64_t)(s_last + 1));
            produced = npairs;
        } else {
            base = lcg_jump(base, 2ull * (uint64_t)THREADS * K);
            produced += total;
        }
        __syncthreads();
    }
    return base;
}

__global__ void __launch_bounds__(RNG_THREADS)
gauss_streams_kernel(uint64_t* __restrict__ states, double* __restrict__ out,
                     const long long* __restrict__ offsets, const int* __restrict__ counts,
                     int* __restrict__ status)
{
    __shared__ int s_wave[RNG_THREADS / 64];
    __shared__ long long s_last;
    const int s = blockIdx.x;
    const uint64_t base = gauss_rounds<RNG_THREADS, 8>(states[s], out + offsets[s], counts[s], status, s_wave, s_last);
    if (threadIdx.x == 0) states[s] = base;
}

// A short call of one stream: one launch.
template <int K>
__global__ void __launch_bounds__(RNG_THREADS)
gauss_one_kernel(uint64_t* __restrict__ state, double* __restrict__ out, int count, int* __restrict__ status)
{
    __shared__ int s_wave[RNG_THREADS / 64];
    __shared__ long long s_last;
    const uint64_t base = gauss_rounds<RNG_THREADS, K>(*state, out, count, status, s_wave, s_last);
    if (threadIdx.x == 0) *state = base;
}

// ------------------------------------------------------------------ one stream, many workgroups
// A long call of one stream (the m steps' noise of one system) in two launches instead of one
// workgroup's rounds: (1) workgroup w evaluates attempts [w GW_THREADS K, (w + 1) GW_THREADS K)
// of the call and counts its accepts; (2) every workgroup adds up the counts before its own,
// evaluates its attempts again and writes the accepted pairs below the needed count, the thread of
// the last needed pair setting the stream state after its attempt.  In the (never observed) case
// that all attempts hold too few accepts, workgroup 0 draws the rest.  The values and the final
// state are those of gauss_rounds, attempt for attempt.
constexpr int GW_THREADS = 256;

struct GaussPlan {
    uint64_t base;      // stream state at the start of the call
    uint64_t pad;
};

template <int K>
__global__ void __launch_bounds__(GW_THREADS)
gauss_wide_count_kernel(const uint64_t* __restrict__ state, int* __restrict__ wg_count, GaussPlan* __restrict__ plan)
{
    __shared__ int s_red[GW_THREADS / 64];
    double v1[K], v2[K], rsq[K];
    const uint64_t base = *state;
    const long long g = (long long)blockIdx.x * GW_THREADS + threadIdx.x;
    int acc = gauss_attempts<K>(lcg_jump(base, 2ull * (uint64_t)g * K), v1, v2, rsq);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < GW_THREADS / 64; ++w) sum += s_red[w];
        wg_count[blockIdx.x] = sum;
        if (blockIdx.x == 0) plan->base = base;
    }
}

template <int K>
__global__ void __launch_bounds__(GW_THREADS)
gauss_wide_write_kernel(uint64_t* __restrict__ state, double* __restrict__ out, const int* __restrict__ wg_count,
                        int count, const GaussPlan* __restrict__ plan, int* __restrict__ status)
{
    constexpr int WAVES = GW_THREADS / 64;
    __shared__ int s_wave[WAVES];
    __shared__ long long s_sum[2][WAVES];
    __shared__ long long s_last;
    const int t = threadIdx.x, wave = t >> 6, G = gridDim.x;
    const uint64_t base = plan->base;
    const long long npairs = ((long long)count + 1) / 2;
    const long long g = (long long)blockIdx.x * GW_THREADS + t;
    double v1[K], v2[K], rsq[K];
    const int acc = gauss_attempts<K>(lcg_jump(base, 2ull * (uint64_t)g * K), v1, v2, rsq);
    const int incl = wave_scan(acc);
    long long before = 0, total = 0;   // pairs before this workgroup; of all of them
    for (int w = t; w < G; w += GW_THREADS) {
        const int c = wg_count[w];
        before += w < (int)blockIdx.x ? c : 0;
        total += c;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        before += __shfl_xor(before, off);
        total += __shfl_xor(total, off);
    }
    if ((t & 63) == 63) {
        s_wave[wave] = incl;
        s_sum[0][wave] = before;
        s_sum[1][wave] = total;
    }
    __syncthreads();
    before = 0;
    total = 0;
    for (int w = 0; w < WAVES; ++w) {
        before += s_sum[0][w] + (w < wave ? s_wave[w] : 0);
        total += s_sum[1][w];
    }
    gauss_pairs<K>(v1, v2, rsq, before + incl - acc, npairs, count, out,
                   [&](int q) { *state = lcg_jump(base, 2ull * (uint64_t)(g * K + q + 1)); });
    if (blockIdx.x == 0 && total < npairs) {
        __syncthreads();   // s_wave is free
        const uint64_t next = gauss_rounds<GW_THREADS, K>(lcg_jump(base, 2ull * (uint64_t)G * GW_THREADS * K),
                                                          out + 2 * total, count - 2 * total, status, s_wave, s_last);
        if (t == 0) *state = next;
    }
}

bool g_jumps_ready[64] = {false};

int ensure_jumps()
{
    int dev = 0;
    BDH_HIP(hipGetDevice(&dev));
    if (dev >= 0 && dev < 64 && g_jumps_ready[dev]) return 0;
    uint64_t A[48], C[48];
    A[0] = LCG_A;
    C[0] = LCG_C;
    for (int b = 1; b < 48; ++b) {  // J_{b} = J_{b-1} o J_{b-1}
        A[b] = (A[b - 1] * A[b - 1]) & MASK48;
        C[b] = (A[b - 1] * C[b - 1] + C[b - 1]) & MASK48;
    }
    BDH_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_jumpA), A, sizeof(A)));
    BDH_HIP(hipMemcpyToSymbol(HIP_SYMBOL(c_jumpC), C, sizeof(C)));
    if (dev >= 0 && dev < 64) g_jumps_ready[dev] = true;
    return 0;
}

}  // namespace

uint64_t lcg_seed(uint32_t seed) { return (((uint64_t)seed) << 16) | 0x330Eu; }

int gauss_prepare() { return ensure_jumps(); }

// Calls of at most this many values take one workgroup: its first round (two attempts a thread)
// holds them, 5.9 us at 60 values and 6.7 at 768, where the two launches take 10.6 (26655 values)
// and a second round would cost one workgroup 5 more.  With four launches (count, plan, write,
// remainder; eight attempts a thread) 768 values took 22 us, 26655 19 us.
constexpr int GAUSS_ONE_MAX = 2800;

// Attempts per thread: few, so that a call spreads over the chip and a thread has few logarithms
// one after the other, until the workgroups' summing of each other's counts costs more.
int gauss_wide_k(long long attempts) { return attempts <= (1 << 20) ? 2 : 8; }

long long gauss_attempts_for(long long count)
{
    // 1.34 per pair (acceptance pi / 4 = 0.785: 1.273) plus a margin of 2048
    return (long long)(1.34 * (double)((count + 1) / 2)) + 2048;
}

int gauss_wide_workgroups(long long count)
{
    const long long need = gauss_attempts_for(count), per = (long long)GW_THREADS * gauss_wide_k(need);
    return (int)((need + per - 1) / per);
}

size_t gauss_wide_scratch_bytes(long long max_count)
{
    // the largest grid of K = 2 may belong to a smaller count than max_count
    const long long wgs = std::max<long long>(gauss_wide_workgroups(max_count), (1 << 20) / (2 * GW_THREADS));
    return sizeof(GaussPlan) + sizeof(int) * (size_t)wgs;
}

int launch_gauss_wide(uint64_t* d_state, double* d_out, int count, void* d_scratch, size_t scratch_bytes,
                      int* d_status, hipStream_t st)
{
    if (count <= 0) return 0;
    if (ensure_jumps()) return -1;
    if (count <= GAUSS_ONE_MAX) {
        hipLaunchKernelGGL(gauss_one_kernel<2>, dim3(1), dim3(RNG_THREADS), 0, st, d_state, d_out, count, d_status);
        BDH_LAUNCH_CHECK();
        return 0;
    }
    const int G = gauss_wide_workgroups(count);
    BDH_CHECK(sizeof(GaussPlan) + sizeof(int) * (size_t)G <= scratch_bytes, "gauss: scratch too small for the count");
    GaussPlan* plan = static_cast<GaussPlan*>(d_scratch);
    int* wg = reinterpret_cast<int*>(plan + 1);
    auto launch = [&](auto k) {
        constexpr int K = decltype(k)::value;
        hipLaunchKernelGGL(gauss_wide_count_kernel<K>, dim3(G), dim3(GW_THREADS), 0, st, (const uint64_t*)d_state, wg,
                           plan);
        BDH_LAUNCH_CHECK();
        hipLaunchKernelGGL(gauss_wide_write_kernel<K>, dim3(G), dim3(GW_THREADS), 0, st, d_state, d_out,
                           (const int*)wg, count, (const GaussPlan*)plan, d_status);
        BDH_LAUNCH_CHECK();
        return 0;
    };
    return gauss_wide_k(gauss_attempts_for(count)) == 2 ? launch(std::integral_constant<int, 2>{})
                                                        : launch(std::integral_constant<int, 8>{});
}

int launch_gauss_streams(uint64_t* d_states, double* d_out, const long long* d_offsets,
                         const int* d_counts, int nstreams, int* d_status, hipStream_t st)
{
    if (nstreams <= 0) return 0;
    if (ensure_jumps()) return -1;
    hipLaunchKernelGGL(gauss_streams_kernel, dim3(nstreams), dim3(RNG_THREADS), 0, st,
                       d_states, d_out, d_offsets, d_counts, d_status);
    BDH_LAUNCH_CHECK();
    return 0;
}

}  // namespace bdh
