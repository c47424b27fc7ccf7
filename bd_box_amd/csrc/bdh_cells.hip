// Cell lists built on the GPU and the nonbonded forces evaluated over them.
//
// The reference builds its neighbour structures on the host at every force call
// (calc_func.c:114-115): hashed spatial buckets (nb_list bucket_space, bucket.c:471-509)
// or sorted corner keys (bucket_list, bucket.c:173-379), both of cell edge
// max_force_cutoff (pre_func.c:197-231: the largest potential cutoff, or twice the
// largest bead radius, plus 0.01).  Pairs found there go through force_single, whose
// per-potential cutoffs select the interacting pairs -- the same set the brute-force
// loop selects (calc_func.c:188-228).  Here, all on the device and rebuilt every call:
//   grid          the bounding box (bc none) or the periodic cube in cubic cells of edge >=
//                 the cell cutoff, at most CELL_MAX_DIM per axis
//   count, scan   beads of every cell, and the cells' first slots
//   place         bead indices, ascending within a cell, and the positions beside them: the
//                 lists -- and the order of every force sum -- do not depend on the order the
//                 counting atomics ran in
// Few beads take one launch (cell_build_kernel<false>), up to CELL_ONE_MAX_N two or three (the
// cells first), more a launch per stage.  A bead's neighbours are the beads of the 27 surrounding cells (each distinct cell
// once when a periodic axis has fewer than 3 cells): cells adjacent in x are adjacent in the
// list, so these are at most nine runs of it and, at a periodic x boundary, nine single cells.
// The pair and bond terms are the brute-force kernel's (bdh_pairterm.hpp); with the cell edge
// at least the largest cutoff, every pair the brute-force kernel finds interacting is visited,
// so the set of interacting pairs is identical.
#include "bdh_common.hpp"
#include "bdh_kernels.hpp"
#include "bdh_pairterm.hpp"

namespace bdh {

struct CellGrid {
    double ox, oy, oz;  // origin
    double h, inv_h;    // cell edge
    int nx, ny, nz;
    int ncell;
};

// Cubic cells of edge >= cutoff, at most CELL_MAX_DIM per axis: tiling the periodic cube, or
// covering the bounding box lo..hi.
__device__ CellGrid make_grid(double lx, double ly, double lz, double hx, double hy, double hz,
                              double cutoff, int pbc, double box)
{
    CellGrid G;
    if (pbc) {
        int n = (int)floor(box / cutoff);
        if (n < 1) n = 1;
        if (n > CELL_MAX_DIM) n = CELL_MAX_DIM;
        G.nx = G.ny = G.nz = n;
        G.h = box / n;
        G.ox = G.oy = G.oz = -0.5 * box;
    } else {
        // extents of the finite coordinates (none finite, e.g. after a failed step: one cell)
        double ex = hx - lx, ey = hy - ly, ez = hz - lz;
        const bool ok = ex >= 0.0 && ey >= 0.0 && ez >= 0.0 && ex < 1e30 && ey < 1e30 && ez < 1e30;
        if (!ok) { ex = ey = ez = 0.0; lx = ly = lz = 0.0; }
        const double h = fmax(cutoff, fmax(fmax(ex, ey), ez) / (CELL_MAX_DIM - 1));
        G.h = h;
        G.ox = lx; G.oy = ly; G.oz = lz;
        G.nx = max(1, min(CELL_MAX_DIM, (int)(ex / h) + 1));
        G.ny = max(1, min(CELL_MAX_DIM, (int)(ey / h) + 1));
        G.nz = max(1, min(CELL_MAX_DIM, (int)(ez / h) + 1));
    }
    G.inv_h = 1.0 / G.h;
    G.ncell = G.nx * G.ny * G.nz;
    return G;
}

// Cell index along one axis, always in [0, n): non-finite coordinates go to cell 0.
__device__ __forceinline__ int cell_coord(double x, double o, double inv_h, int n, int pbc)
{
    double f = floor((x - o) * inv_h);
    if (pbc && !(f >= 0.0 && f < (double)n)) f -= (double)n * floor(f / (double)n);
    if (!(f >= 0.0)) return 0;
    return f >= (double)n ? n - 1 : (int)f;
}

__device__ __forceinline__ int cell_of(const CellGrid& G, double4 p, int pbc)
{
    return (cell_coord(p.z, G.oz, G.inv_h, G.nz, pbc) * G.ny + cell_coord(p.y, G.oy, G.inv_h, G.ny, pbc)) * G.nx +
           cell_coord(p.x, G.ox, G.inv_h, G.nx, pbc);
}

// lo[k], hi[k]: the extremes of every thread's over the workgroup, in thread 0
template <int WAVES>
__device__ __forceinline__ void block_box(double (&lo)[3], double (&hi)[3], double (*s_red)[WAVES])
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int w = 32; w > 0; w >>= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            lo[k] = fmin(lo[k], __shfl_xor(lo[k], w));
            hi[k] = fmax(hi[k], __shfl_xor(hi[k], w));
        }
    if (lane == 0)
        for (int k = 0; k < 3; ++k) { s_red[k][wave] = lo[k]; s_red[3 + k][wave] = hi[k]; }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < WAVES; ++w)
            for (int k = 0; k < 3; ++k) {
                lo[k] = fmin(lo[k], s_red[k][w]);
                hi[k] = fmax(hi[k], s_red[3 + k][w]);
            }
}

__device__ __forceinline__ void add_box(double4 p, double (&lo)[3], double (&hi)[3])
{
    lo[0] = fmin(lo[0], p.x); hi[0] = fmax(hi[0], p.x);
    lo[1] = fmin(lo[1], p.y); hi[1] = fmax(hi[1], p.y);
    lo[2] = fmin(lo[2], p.z); hi[2] = fmax(hi[2], p.z);
}

// box[6 w ..]: the bounding box of the positions workgroup w of CELL_BOXES reads
constexpr int CELL_BOXES = 64;

__global__ void __launch_bounds__(256)
cell_box_kernel(const double4* __restrict__ pos, int N, double* __restrict__ box)
{
    __shared__ double s_red[6][4];
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int i = blockIdx.x * 256 + threadIdx.x; i < N; i += CELL_BOXES * 256) add_box(pos[i], lo, hi);
    block_box<4>(lo, hi, s_red);
    if (threadIdx.x == 0)
        for (int k = 0; k < 3; ++k) { box[6 * blockIdx.x + k] = lo[k]; box[6 * blockIdx.x + 3 + k] = hi[k]; }
}

// Cell of every bead; every workgroup forms the grid for itself.
__global__ void __launch_bounds__(256)
cell_key_kernel(const double4* __restrict__ pos, int N, double cutoff, int pbc, double box,
                const double* __restrict__ boxes, CellGrid* __restrict__ g, int* __restrict__ key)
{
    __shared__ CellGrid s_g;
    const int t = threadIdx.x, i = blockIdx.x * 256 + t;
    const double4 p = pos[min(i, N - 1)];
    if (t < 64) {
        static_assert(CELL_BOXES == 64, "one box a lane");
        double lo[3] = {0.0, 0.0, 0.0}, hi[3] = {0.0, 0.0, 0.0};
        if (!pbc) {
            for (int k = 0; k < 3; ++k) { lo[k] = boxes[6 * t + k]; hi[k] = boxes[6 * t + 3 + k]; }
#pragma unroll
            for (int w = 32; w > 0; w >>= 1)
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    lo[k] = fmin(lo[k], __shfl_xor(lo[k], w));
                    hi[k] = fmax(hi[k], __shfl_xor(hi[k], w));
                }
        }
        if (t == 0) {
            s_g = make_grid(lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], cutoff, pbc, box);
            if (blockIdx.x == 0) *g = s_g;
        }
    }
    __syncthreads();
    if (i < N) key[i] = cell_of(s_g, p, pbc);
}

__global__ void cell_zero_kernel(const CellGrid* __restrict__ g, int* __restrict__ count,
                                 int* __restrict__ fill)
{
    const int ncell = g->ncell;
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < ncell; c += gridDim.x * blockDim.x) {
        count[c] = 0;
        fill[c] = 0;
    }
}

__global__ void cell_count_kernel(int N, const int* __restrict__ key, int* __restrict__ count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) atomicAdd(&count[key[i]], 1);
}

// exclusive scan of count[0..ncell) into start[0..ncell]; one block of 1024 threads
__global__ void __launch_bounds__(1024)
cell_scan_kernel(const int* __restrict__ count, const CellGrid* __restrict__ g,
                 int* __restrict__ start)
{
    __shared__ int s[1024];
    const int ncell = g->ncell;
    const int t = threadIdx.x;
    const int per = (ncell + 1023) / 1024;
    const int b = min(ncell, t * per), e = min(ncell, b + per);
    int sum = 0;
    for (int c = b; c < e; ++c) sum += count[c];
    s[t] = sum;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const int v = (t >= off) ? s[t - off] : 0;
        __syncthreads();
        s[t] += v;
        __syncthreads();
    }
    int run = s[t] - sum;
    for (int c = b; c < e; ++c) { start[c] = run; run += count[c]; }
    if (t == 1023) start[ncell] = s[1023];
}

__global__ void cell_scatter_kernel(int N, const int* __restrict__ key, const int* __restrict__ start,
                                    int* __restrict__ fill, int* __restrict__ list)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int c = key[i];
    list[start[c] + atomicAdd(&fill[c], 1)] = i;
}

// Bead i among the beads list[b, e) of its cell (in any order): its slot by index.
__device__ __forceinline__ void cell_place(int i, double4 p, int b, int e, const int* list, int* __restrict__ sorted,
                                           double4* __restrict__ pos_s)
{
    int k = b;
    for (int m = b; m < e; ++m) k += list[m] < i;
    sorted[k] = i;
    pos_s[k] = p;
}

__global__ void cell_place_kernel(const double4* __restrict__ pos, int N, const int* __restrict__ key,
                                  const int* __restrict__ start, const int* __restrict__ list,
                                  int* __restrict__ sorted, double4* __restrict__ pos_s)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int c = key[i];
    cell_place(i, pos[i], start[c], start[c + 1], list, sorted, pos_s);
}

// Counts, first slots and order of the beads in one launch, without a word between workgroups:
// workgroup w owns the cells [w ncell / CELL_GROUPS, (w + 1) ncell / CELL_GROUPS), looks at
// every bead's cell, counts the beads below its cells (its first slot) and those in them (in
// LDS), and places its own, which a thread remembers as bits, one for each bead it looked at.
// KEYS: the cells come from cell_key_kernel, 4 bytes a bead; otherwise each workgroup forms the
// grid and the cells from the positions, 32 bytes a bead, and the whole build is this launch.
// Bound by each workgroup's reading of every bead, then by latency.  20000 periodic beads: 46 us
// in one workgroup (24^3 cells), now 12 us with cell_key_kernel; 1000 beads 5.4 us.  128
// workgroups instead of 32 place 20000 beads 2.3 us sooner and cost the small builds nothing.
constexpr int CELL_ONE_THREADS = 1024;
constexpr int CELL_ONE_MAX_N = 64 * CELL_ONE_THREADS;
constexpr int CELL_GROUPS = 128;
constexpr int CELL_OWN_MAX = (CELL_MAX + CELL_GROUPS - 1) / CELL_GROUPS;

template <bool KEYS>
__global__ void __launch_bounds__(CELL_ONE_THREADS)
cell_build_kernel(const double4* __restrict__ pos, int N, double cutoff, int pbc, double box,
                  CellGrid* __restrict__ g, int* __restrict__ key, int* __restrict__ start, int* __restrict__ list,
                  int* __restrict__ sorted, double4* __restrict__ pos_s)
{
    constexpr int WAVES = CELL_ONE_THREADS / 64;
    __shared__ int s_cnt[CELL_OWN_MAX];
    __shared__ int s_wave[2][WAVES];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int ncells;
    CellGrid G;
    if constexpr (KEYS) {
        ncells = g->ncell;
    } else {
        __shared__ double s_red[6][WAVES];
        __shared__ CellGrid s_g;
        double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
        if (!pbc) {
            for (int i = t; i < N; i += CELL_ONE_THREADS) add_box(pos[i], lo, hi);
            block_box<WAVES>(lo, hi, s_red);
        }
        if (t == 0) {
            s_g = make_grid(lo[0], lo[1], lo[2], hi[0], hi[1], hi[2], cutoff, pbc, box);
            if (blockIdx.x == 0) *g = s_g;
        }
        __syncthreads();
        G = s_g;
        ncells = G.ncell;
    }
    const int c0 = (int)((long long)ncells * blockIdx.x / CELL_GROUPS);
    const int c1 = (int)((long long)ncells * (blockIdx.x + 1) / CELL_GROUPS);
    if (c0 == c1) return;
    for (int c = t; c < c1 - c0; c += CELL_ONE_THREADS) s_cnt[c] = 0;
    __syncthreads();
    int below = 0;
    unsigned long long own = 0;
    auto look = [&](int bit, int c) {
        below += c < c0;
        if (c >= c0 && c < c1) {
            own |= 1ull << bit;
            atomicAdd(&s_cnt[c - c0], 1);
        }
    };
    // bit b of thread t: bead bead_of(b)
    auto bead_of = [&](int b) { return KEYS ? 4 * (t + (b >> 2) * CELL_ONE_THREADS) + (b & 3) : t + b * CELL_ONE_THREADS; };
    if constexpr (KEYS) {
#pragma unroll 4
        for (int q = 0; q < (N + 4 * CELL_ONE_THREADS - 1) / (4 * CELL_ONE_THREADS); ++q) {
            const int i = bead_of(4 * q);
            int4 c = reinterpret_cast<const int4*>(key)[min(i, (N - 1) & ~3) >> 2];
            if (i < N) look(4 * q, c.x);
            if (i + 1 < N) look(4 * q + 1, c.y);
            if (i + 2 < N) look(4 * q + 2, c.z);
            if (i + 3 < N) look(4 * q + 3, c.w);
        }
    } else {
        for (int q = 0, i = t; i < N; ++q, i += CELL_ONE_THREADS) {
            const int c = cell_of(G, pos[i], pbc);
            if (c >= c0 && c < c1) key[i] = c;
            look(q, c);
        }
    }
    __syncthreads();
    // exclusive scan of the own cells: a run of cells a thread, then the threads' sums
    const int ncell = c1 - c0, per = (ncell + CELL_ONE_THREADS - 1) / CELL_ONE_THREADS;
    const int b = min(ncell, t * per), e = min(ncell, b + per);
    int sum = 0;
    for (int c = b; c < e; ++c) sum += s_cnt[c];
    int run = sum;
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) {
        const int v = __shfl_up(run, w);
        if (lane >= w) run += v;
        below += __shfl_xor(below, w);
    }
    if (lane == 63) { s_wave[0][wave] = run; s_wave[1][wave] = below; }
    __syncthreads();
    run -= sum;
    int first = 0;  // slot of the first own bead
    for (int w = 0; w < WAVES; ++w) {
        first += s_wave[1][w];
        if (w < wave) run += s_wave[0][w];
    }
    run += first;
    for (int c = b; c < e; ++c) {
        const int n = s_cnt[c];
        s_cnt[c] = run;
        start[c0 + c] = run;
        run += n;
    }
    if (c1 == ncells && t == 0) start[c1] = N;
    __syncthreads();
    for (unsigned long long m = own; m; m &= m - 1) {
        const int i = bead_of(__ffsll(m) - 1);
        list[atomicAdd(&s_cnt[key[i] - c0], 1)] = i;
    }
    __syncthreads();
    // s_cnt[c] is now the end of cell c0 + c
    for (unsigned long long m = own; m; m &= m - 1) {
        const int i = bead_of(__ffsll(m) - 1);
        const double4 p = pos[i];
        const int c = key[i] - c0;
        cell_place(i, p, c ? s_cnt[c - 1] : first, s_cnt[c], list, sorted, pos_s);
    }
}

int launch_cell_build(const double4* d_pos, int N, double cutoff, int pbc, double box,
                      const CellList& cl, hipStream_t st)
{
    BDH_CHECK(cutoff > 0.0, "cell list: cutoff must be positive");
    CellGrid* g = (CellGrid*)cl.grid;
    double* boxes = reinterpret_cast<double*>(g + 1);
    const dim3 beads(ceil_div(N, 256));
    // one launch while reading the positions in every workgroup costs less than the extra
    // launches (us, one launch / two or three): periodic 4000 beads 8.4 / 9.6, 8000 10.7 / 10.9,
    // 12000 13.3 / 11.9; free space, which reads them twice, 4000 13.2 / 13.2, 6000 15.0 / 14.0
    if (N <= (pbc ? 8192 : 4096)) {
        hipLaunchKernelGGL(cell_build_kernel<false>, dim3(CELL_GROUPS), dim3(CELL_ONE_THREADS), 0, st, d_pos, N,
                           cutoff, pbc, box, g, cl.key, cl.start, cl.list, cl.sorted, cl.pos);
        BDH_LAUNCH_CHECK();
        return 0;
    }
    if (!pbc) {
        hipLaunchKernelGGL(cell_box_kernel, dim3(CELL_BOXES), dim3(256), 0, st, d_pos, N, boxes);
        BDH_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(cell_key_kernel, beads, dim3(256), 0, st, d_pos, N, cutoff, pbc, box, (const double*)boxes, g,
                       cl.key);
    BDH_LAUNCH_CHECK();
    if (N <= CELL_ONE_MAX_N) {
        hipLaunchKernelGGL(cell_build_kernel<true>, dim3(CELL_GROUPS), dim3(CELL_ONE_THREADS), 0, st, d_pos, N,
                           cutoff, pbc, box, g, cl.key, cl.start, cl.list, cl.sorted, cl.pos);
        BDH_LAUNCH_CHECK();
        return 0;
    }
    hipLaunchKernelGGL(cell_zero_kernel, dim3(256), dim3(256), 0, st, (const CellGrid*)g, cl.count,
                       cl.fill);
    BDH_LAUNCH_CHECK();
    hipLaunchKernelGGL(cell_count_kernel, beads, dim3(256), 0, st, N, (const int*)cl.key, cl.count);
    BDH_LAUNCH_CHECK();
    hipLaunchKernelGGL(cell_scan_kernel, dim3(1), dim3(1024), 0, st, cl.count, (const CellGrid*)g,
                       cl.start);
    BDH_LAUNCH_CHECK();
    hipLaunchKernelGGL(cell_scatter_kernel, beads, dim3(256), 0, st, N, cl.key, cl.start, cl.fill, cl.list);
    BDH_LAUNCH_CHECK();
    hipLaunchKernelGGL(cell_place_kernel, beads, dim3(256), 0, st, d_pos, N, cl.key, cl.start, cl.list, cl.sorted,
                       cl.pos);
    BDH_LAUNCH_CHECK();
    return 0;
}

// The neighbours of a bead as runs of the list: candidate row q = ky + my kz of the cells
// around its own, and in it the cells x0..x1 and, at a periodic boundary, the wrapped cell xw.
struct NbrRows {
    int cy, cz;
    int my, mz;      // candidates per axis: 3, or n for a periodic axis of n < 3 cells
    int x0, x1, xw;  // xw < 0: none
};

__device__ __forceinline__ NbrRows nbr_rows(const CellGrid& G, double4 p, int pbc)
{
    NbrRows r;
    const int cx = cell_coord(p.x, G.ox, G.inv_h, G.nx, pbc);
    r.cy = cell_coord(p.y, G.oy, G.inv_h, G.ny, pbc);
    r.cz = cell_coord(p.z, G.oz, G.inv_h, G.nz, pbc);
    r.my = (pbc && G.ny < 3) ? G.ny : 3;
    r.mz = (pbc && G.nz < 3) ? G.nz : 3;
    r.x0 = max(cx - 1, 0);
    r.x1 = min(cx + 1, G.nx - 1);
    r.xw = (!pbc || G.nx <= 3) ? -1 : cx == 0 ? G.nx - 1 : cx == G.nx - 1 ? 0 : -1;
    if (pbc && G.nx <= 3) { r.x0 = 0; r.x1 = G.nx - 1; }
    return r;
}

// axis coordinate of candidate k, or -1 if it lies outside a non-periodic grid
__device__ __forceinline__ int nbr_axis(int c, int k, int m, int n, int pbc)
{
    if (pbc) {
        if (m < 3) return k;
        const int v = c + k - 1;
        return v < 0 ? v + n : (v >= n ? v - n : v);
    }
    const int v = c + k - 1;
    return (v < 0 || v >= n) ? -1 : v;
}

// f(k) for every list slot k of candidate row q
template <typename F>
__device__ __forceinline__ void each_in_row(const CellGrid& G, const NbrRows& r, int q, int pbc,
                                            const int* __restrict__ start, F&& f)
{
    const int kz = q / r.my;
    const int y = nbr_axis(r.cy, q - kz * r.my, r.my, G.ny, pbc);
    const int z = nbr_axis(r.cz, kz, r.mz, G.nz, pbc);
    if (y < 0 || z < 0) return;
    const int* row = start + (z * G.ny + y) * G.nx;
    const int e = row[r.x1 + 1];
    for (int k = row[r.x0]; k < e; ++k) f(k);
    if (r.xw >= 0) {
        const int ew = row[r.xw + 1];
        for (int k = row[r.xw]; k < ew; ++k) f(k);
    }
}

// ------------------------------------------------------------------------ forces
// Row beads in list order, so that a workgroup's rows share their neighbours; CELL_LANES lanes
// a bead, lane l taking neighbour row l (of at most nine), and the lanes' sums meeting in a
// fixed shuffle tree (deterministic).  Full rows: no atomics.  Bound by the chain of dependent
// loads (row bounds, positions, charges): 20000 spheres 17 us with 27 cells over 8 lanes and
// positions read through the index list, 9.4 us with runs of adjacent cells and listed positions.
constexpr int CELL_LANES = 16;
constexpr int CF_THREADS = 128;

template <typename T>
__global__ void __launch_bounds__(CF_THREADS)
forces_cells_kernel(const double4* __restrict__ pos, const double* __restrict__ Q,
                    const double2* __restrict__ LJ, int N, Topology topo, ForceParams fp,
                    const CellGrid* __restrict__ g, const int* __restrict__ start,
                    const int* __restrict__ sorted, const double4* __restrict__ pos_s,
                    double* __restrict__ F, double* __restrict__ PE, int* __restrict__ flags)
{
    __shared__ double s_e[3][CF_THREADS / CELL_LANES];
    const int sub = threadIdx.x % CELL_LANES;
    const int slot = threadIdx.x / CELL_LANES;
    const int row = blockIdx.x * (CF_THREADS / CELL_LANES) + slot;
    PairAcc a{0, 0, 0, 0, 0, 0};
    double e_b = 0.0;
    int i = 0;
    if (row < N) {
        i = sorted[row];
        const CellGrid G = *g;
        const double4 pi = pos_s[row];
        const double qi = Q[i];
        const double2 lji = LJ[i];
        const int nb0 = fp.use_conn ? topo.conn_off[i] : 0;
        const int nb1 = fp.use_conn ? topo.conn_off[i + 1] : 0;
        const NbrRows nr = nbr_rows(G, pi, fp.pbc);
        if (sub < nr.my * nr.mz)
            each_in_row(G, nr, sub, fp.pbc, start, [&](int k) {
                if (k == row) return;
                const double4 pj = pos_s[k];
                const int j = sorted[k];
                double dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
                const double r2 = pair_r2(dx, dy, dz, fp.pbc, fp.box);
                if (r2 <= fp.far_r2)
                    pair_term<T>(dx, dy, dz, r2, qi, Q[j], lji, LJ[j], bonded(topo, nb0, nb1, j), fp, a);
            });
        if (sub == CELL_LANES - 1) e_b = bond_terms(pos, i, pi, topo, fp, a, PE != nullptr);
    }
#pragma unroll
    for (int w = CELL_LANES / 2; w > 0; w >>= 1) {
        a.fx += __shfl_xor(a.fx, w, CELL_LANES);
        a.fy += __shfl_xor(a.fy, w, CELL_LANES);
        a.fz += __shfl_xor(a.fz, w, CELL_LANES);
        a.e_lj += __shfl_xor(a.e_lj, w, CELL_LANES);
        a.e_c += __shfl_xor(a.e_c, w, CELL_LANES);
        a.rep |= __shfl_xor(a.rep, w, CELL_LANES);
    }
    e_b = __shfl(e_b, CELL_LANES - 1, CELL_LANES);
    if (sub == 0) {
        if (row < N) {
            F[3 * i] = a.fx;
            F[3 * i + 1] = a.fy;
            F[3 * i + 2] = a.fz;
        }
        s_e[0][slot] = a.e_lj;
        s_e[1][slot] = a.e_c;
        s_e[2][slot] = e_b;
    }
    __syncthreads();
    if (PE && threadIdx.x < 3) {
        double s = 0;
        for (int k = 0; k < CF_THREADS / CELL_LANES; ++k) s += s_e[threadIdx.x][k];
        PE[3 * blockIdx.x + threadIdx.x] = 0.5 * s;
    }
    if (a.rep && fp.check_overlap) atomicOr(flags, 1);
    if (a.rep & 2) atomicOr(flags, 2);
}

int cell_force_blocks(int N) { return ceil_div(N, CF_THREADS / CELL_LANES); }

template <typename T>
int launch_forces_cells(const double4* d_pos, const double* d_Q, const double2* d_LJ, int N,
                        const Topology& topo, const ForceParams& fp, const CellList& cl,
                        double* d_F, double* d_PE, int* d_flags, hipStream_t st)
{
    hipLaunchKernelGGL(forces_cells_kernel<T>, dim3(cell_force_blocks(N)), dim3(CF_THREADS), 0, st,
                       d_pos, d_Q, d_LJ, N, topo, fp, (const CellGrid*)cl.grid, cl.start, cl.sorted,
                       (const double4*)cl.pos, d_F, d_PE, d_flags);
    BDH_LAUNCH_CHECK();
    return 0;
}

// ------------------------------------------------------------------- pair export
// Pairs i < j with |r_j - r_i| <= cutoff (FP64, pair_r2) found through the cell list,
// written in whatever order the atomics give (the caller sorts).  count may exceed cap:
// then only cap pairs were stored.
__global__ void cell_pairs_kernel(const double4* __restrict__ pos, int N,
                                  const CellGrid* __restrict__ g, const int* __restrict__ start,
                                  const int* __restrict__ sorted, double cutoff, int pbc,
                                  double box, int* __restrict__ pairs, long long cap,
                                  unsigned long long* __restrict__ count)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const CellGrid G = *g;
    const double4 pi = pos[i];
    const NbrRows nr = nbr_rows(G, pi, pbc);
    for (int q = 0; q < nr.my * nr.mz; ++q)
        each_in_row(G, nr, q, pbc, start, [&](int k) {
            const int j = sorted[k];
            if (j <= i) return;
            const double4 pj = pos[j];
            double dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
            const double r = sqrt(pair_r2(dx, dy, dz, pbc, box));
            if (r <= cutoff) {
                const unsigned long long s = atomicAdd(count, 1ull);
                if ((long long)s < cap) {
                    pairs[2 * s] = i;
                    pairs[2 * s + 1] = j;
                }
            }
        });
}

__global__ void clear_u64_kernel(unsigned long long* p) { *p = 0ull; }

int launch_cell_pairs(const double4* d_pos, int N, const CellList& cl, double cutoff, int pbc,
                      double box, int* d_pairs, long long cap, unsigned long long* d_count,
                      hipStream_t st)
{
    hipLaunchKernelGGL(clear_u64_kernel, dim3(1), dim3(1), 0, st, d_count);
    BDH_LAUNCH_CHECK();
    hipLaunchKernelGGL(cell_pairs_kernel, dim3(ceil_div(N, 128)), dim3(128), 0, st, d_pos, N,
                       (const CellGrid*)cl.grid, cl.start, cl.sorted, cutoff, pbc, box, d_pairs, cap,
                       d_count);
    BDH_LAUNCH_CHECK();
    return 0;
}

size_t cell_grid_bytes() { return sizeof(CellGrid) + sizeof(double) * 6 * CELL_BOXES; }

template int launch_forces_cells<float>(const double4*, const double*, const double2*, int, const Topology&, const ForceParams&, const CellList&, double*, double*, int*, hipStream_t);
template int launch_forces_cells<double>(const double4*, const double*, const double2*, int, const Topology&, const ForceParams&, const CellList&, double*, double*, int*, hipStream_t);

}  // namespace bdh
