// sf_m2g.hip -- deterministic marker -> grid interpolation for gfx950.
//
// Reference: bilinearMarkerToGrid! (MarkerToGrid.jl:18-38).  The reference's GPU path adds
// 8 float64 atomics per marker (:58-100) and is order-nondeterministic; its CPU path
// (:110-155) adds the markers sequentially in index order m = 1..Nm.  This
// implementation reproduces the CPU path bit for bit:
//
//   1. key:     per marker the top-left node (ix, iy) of common.jl:22-33 with the same
//               IEEE operations; markers outside [0,Nx]x[0,Ny] are counted ("erroneous
//               marker position") and dropped.  cell = ix*(Ny+1) + iy (column-major: see m2g_keys).
//   2. count + exclusive scan of markers per cell (integer atomics: exact).
//   3. scatter marker indices into their cell segment (each marker's place in its cell comes from
//               the counting atomic: runs of markers in no fixed order).
//   4. tiles: node (A, B) (1-based) receives contributions from cells (A,B) as top-left,
//               (A-1,B) as top-right, (A,B-1) as bottom-left and (A-1,B-1) as bottom-right
//               (:124-151).  A workgroup takes the cells of a tile of nodes into LDS, sorts each
//               cell's markers by index, and merges the four cells of each node by index: that
//               replays exactly the CPU accumulation order, so wt_sum and val_wt_sum are the CPU
//               sums; safeDivision (:164-172) keeps the old value where wt == 0.
//   5. tiles whose markers do not fit into LDS are done in pieces of fewer rows; rows that do not fit alone,
//               and all of a grid with very many markers per cell, from global memory, a wave per node.
#include <algorithm>

#include "sf_device.h"
#include "sf_internal.h"

namespace sf {

enum { CNT_BAD = 0, CNT_EMPTY = 1, CNT_NONFINITE = 2, CNT_OVERFLOW = 3 };  // CNT_OVERFLOW: tiles listed in step 5
#define SCAN_ITEMS 8
#define SCAN_BLOCK 256
#define SCAN_TILE (SCAN_ITEMS * SCAN_BLOCK)
#define SCAN_TOP 1024
#define M2G_EMPTY ((M2G_SPREAD) / 16 - 1)  // counters of empty nodes, one to a 128-byte line
#define M2G_FAR 80.0

// floor(Int, v) in the reference throws unless v fits an Int64.
__device__ inline bool key_ok(double v) { return __builtin_isfinite(v) && v > -9.2e18 && v < 9.2e18; }

// Workgroup k of n in the order that gives each of the 8 XCDs (to which the hardware hands workgroups
// round robin) a contiguous band.
__device__ inline int xcd_band(int k, int n)
{
    const int x = k % 8, i = k / 8, per = n / 8, rem = n % 8;
    return (x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per) + i;
}

// topleftIndexRelDist (common.jl:22-33), 1-based ix/iy.
__device__ inline void topleft(double xmin, double ymin, double x, double y, double dx, double dy, int64_t& ix,
                               int64_t& iy, double& dxij, double& dyij)
{
    ix = (int64_t)floor((x - xmin) / dx) + 1;
    iy = (int64_t)floor((y - ymin) / dy) + 1;
    const double x_ix = xmin + (double)(ix - 1) * dx;
    const double y_iy = ymin + (double)(iy - 1) * dy;
    dxij = (x - x_ix) / dx;
    dyij = (y - y_iy) / dy;
}

__global__ __launch_bounds__(256) void fill_int(int* __restrict__ a, int64_t n, int v)
{
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) a[k] = v;
}

__global__ __launch_bounds__(256) void fill_dbl(double* __restrict__ a, int64_t n, double v)
{
    for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) a[k] = v;
}

__global__ void zero_counters(unsigned long long* c, unsigned long long* spread)
{
    if (threadIdx.x < 4) c[threadIdx.x] = 0ull;
    if (!spread) return;
    for (int k = threadIdx.x; k < M2G_SPREAD; k += blockDim.x) spread[k] = 0ull;
}

// Runs of equal keys in consecutive lanes (markers in index order share cells: the x-outer /
// y-inner set-up puts md consecutive markers in one cell): per lane, whether it heads a run, the
// run length (heads only) and the lane of its run's head.  Every lane of the wave calls this.
struct KeyRun {
    bool head;
    int len, head_lane;
};
__device__ inline KeyRun key_run(int k)
{
    const int lane = (int)__lane_id();
    const int kp = dpp_i32<0x138>(k);  // the key of lane - 1 (wave_shr:1; lane 0 reads 0)
    const bool valid = k >= 0;
    const bool head = valid && (lane == 0 || kp != k);
    const unsigned long long heads = __ballot(head);
    const unsigned long long brk = __ballot(head || !valid);  // a run ends where the next one starts
    KeyRun r;
    r.head = head;
    const unsigned long long after = lane == 63 ? 0ull : (brk >> (lane + 1));
    r.len = head ? (after ? __builtin_ctzll(after) + 1 : 64 - lane) : 0;
    const unsigned long long upto = heads & (lane == 63 ? ~0ull : ((2ull << lane) - 1ull));
    r.head_lane = upto ? 63 - __builtin_clzll(upto) : lane;
    return r;
}

// The keys and the scatter wait for memory (the counting atomic above all): with U markers to a thread U
// atomics and 2 U loads are in flight at once.  268 M markers, ms, U = 1, 2, 4, 8: keys 2.38, 2.32, 1.76, 1.68,
// scatter 0.99, 0.75, 0.73, 0.92.  Up to some 10 M markers the waves in flight cover the waits, and U = 4
// costs 3 to 5% of a whole pass (4.2 M: 0.191 against 0.204 ms; 12 M equal; 19 M 0.957 against 0.948).
#define M2G_MANY (1 << 24)
#define M2G_PER_THREAD 4
template <int U>
__global__ __launch_bounds__(256) void m2g_keys(const double* __restrict__ x_m, const double* __restrict__ y_m, int64_t nm,
                                                double xmin, double ymin, double dx, double dy, int gnx, int gny,
                                                int* __restrict__ key, int* __restrict__ count, int* __restrict__ loc,
                                                unsigned long long* __restrict__ counters)
{
    const int lane = (int)__lane_id();
    const int64_t m0 = ((int64_t)blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64) * (64 * U) + lane;
    if (m0 - lane >= nm) return;
    double x[U], y[U];
    int k[U], base[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t m = min(m0 + 64 * u, nm - 1);
        x[u] = x_m[m];
        y[u] = y_m[m];
    }
    KeyRun run[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        k[u] = -1;
        if (m0 + 64 * u < nm) {
            if (!key_ok((x[u] - xmin) / dx) || !key_ok((y[u] - ymin) / dy)) {
                atomicAdd(&counters[CNT_NONFINITE], 1ull);
            } else {
                int64_t ix, iy;
                double dxij, dyij;
                topleft(xmin, ymin, x[u], y[u], dx, dy, ix, iy, dxij, dyij);
                if (!(ix >= 0 && ix <= gnx && iy >= 0 && iy <= gny)) {
                    atomicAdd(&counters[CNT_BAD], 1ull);
                } else {
                    // the sort numbers cells column-major (ix slowest), the order in which the x-outer /
                    // y-inner marker set-up visits them, so the per-cell gathers below read nearly in
                    // order; the exported keys are row-major (sf_marker_cell_keys)
                    k[u] = loc ? (int)(ix * (int64_t)(gny + 1) + iy) : (int)(iy * (int64_t)(gnx + 1) + ix);
                }
            }
            key[m0 + 64 * u] = k[u];
        }
        // one counter atomic per run of equal keys instead of one per marker; for the sort it also gives
        // the run its places in the cell, in index order within the run
        run[u] = key_run(k[u]);
    }
    if (loc) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            base[u] = 0;
            if (run[u].head) base[u] = atomicAdd(&count[k[u]], run[u].len);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            base[u] = __shfl(base[u], run[u].head_lane);
            if (k[u] >= 0) loc[m0 + 64 * u] = base[u] + (lane - run[u].head_lane);
        }
    } else {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (run[u].head) atomicAdd(&count[k[u]], run[u].len);
    }
}

__global__ __launch_bounds__(SCAN_BLOCK) void scan_block_sums(const int* __restrict__ cnt, int64_t n,
                                                              int* __restrict__ bsum)
{
    __shared__ int sh[SCAN_BLOCK];
    const int t = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)t * SCAN_ITEMS;
    int s = 0;
    for (int i = 0; i < SCAN_ITEMS; ++i)
        if (base + i < n) s += cnt[base + i];
    sh[t] = s;
    __syncthreads();
    for (int w = SCAN_BLOCK / 2; w > 0; w >>= 1) {
        if (t < w) sh[t] += sh[t + w];
        __syncthreads();
    }
    if (t == 0) bsum[blockIdx.x] = sh[0];
}

// Exclusive scan of the (few thousand) block sums by one workgroup: each thread a chunk, then a scan
// of the chunk sums (one thread for all took 0.81 ms for the 8,200 sums of 4096^2 cells).
__global__ __launch_bounds__(SCAN_TOP) void scan_top(int* __restrict__ bsum, int nblk)
{
    __shared__ int sh[SCAN_TOP];
    const int t = threadIdx.x;
    const int per = (nblk + SCAN_TOP - 1) / SCAN_TOP;
    const int lo = min(t * per, nblk), hi = min(lo + per, nblk);
    int s = 0;
    for (int b = lo; b < hi; ++b) s += bsum[b];
    sh[t] = s;
    __syncthreads();
    for (int w = 1; w < SCAN_TOP; w <<= 1) {
        const int add = (t >= w) ? sh[t - w] : 0;
        __syncthreads();
        sh[t] += add;
        __syncthreads();
    }
    int acc = sh[t] - s;
    for (int b = lo; b < hi; ++b) {
        const int v = bsum[b];
        bsum[b] = acc;
        acc += v;
    }
}

__global__ __launch_bounds__(SCAN_BLOCK) void scan_apply(const int* __restrict__ cnt, int64_t n,
                                                         const int* __restrict__ bsum, int* __restrict__ off)
{
    __shared__ int sh[SCAN_BLOCK];
    const int t = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)t * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    int s = 0;
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        v[i] = (base + i < n) ? cnt[base + i] : 0;
        s += v[i];
    }
    sh[t] = s;
    __syncthreads();
    // Hillis-Steele inclusive scan of thread sums
    for (int w = 1; w < SCAN_BLOCK; w <<= 1) {
        int add = (t >= w) ? sh[t - w] : 0;
        __syncthreads();
        sh[t] += add;
        __syncthreads();
    }
    int run = bsum[blockIdx.x] + sh[t] - s;
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        if (base + i < n) {
            off[base + i] = run;
            if (base + i == n - 1) off[n] = run + v[i];
        }
        run += v[i];
    }
}

template <int U>
__global__ __launch_bounds__(256) void m2g_scatter(const int* __restrict__ key, const int* __restrict__ loc, int64_t nm,
                                                   const int* __restrict__ off, int* __restrict__ rec_idx)
{
    const int64_t m0 = (int64_t)blockIdx.x * (256 * U) + threadIdx.x;
    int k[U], l[U], o[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t m = min(m0 + 256 * u, nm - 1);
        k[u] = m0 + 256 * u < nm ? key[m] : -1;
        l[u] = loc[m];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) o[u] = off[max(k[u], 0)];
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (k[u] >= 0) rec_idx[o[u] + l[u]] = (int)(m0 + 256 * u);
}

__device__ inline double corner_weight(int corner, double dxij, double dyij)
{
    // MarkerToGrid.jl:127,133,141,147 -- 0 TL, 1 TR, 2 BL, 3 BR
    switch (corner) {
        case 0: return (1.0 - dxij) * (1.0 - dyij);
        case 1: return dxij * (1.0 - dyij);
        case 2: return (1.0 - dxij) * dyij;
        default: return dxij * dyij;
    }
}

// What the node kernels share: the sorted cells, the markers, the grid and its outputs.
struct M2GNodes {
    const int* off;
    int* rec_idx;
    const double *x_m, *y_m, *val_m;
    double xmin, ymin, dx, dy;
    int gnx, gny;
    int tx, ty, ntx, nty;  // nodes per tile, tiles
    double *val_grid, *val_wt_sum, *wt_sum;
    int ws_nx;
    unsigned long long *counters, *spread;
    int *list, *list2;  // parts of tiles that did not fit (first row, rows), rows of these that did not either;
                        // a row is tile * ty + its place in the tile
    bool all;           // all rows are taken as listed
};

__device__ inline void m2g_store(const M2GNodes& g, int a, int b, double wt, double vw)
{
    if (g.wt_sum) {
        g.wt_sum[(int64_t)a + (int64_t)b * g.ws_nx] = wt;
        g.val_wt_sum[(int64_t)a + (int64_t)b * g.ws_nx] = vw;
    }
    if (wt != 0.0)
        g.val_grid[(int64_t)a + (int64_t)b * g.gnx] = vw / wt;
    else
        atomicAdd(&g.spread[(1 + blockIdx.x % M2G_EMPTY) * 16], 1ull);
}

// The empty nodes, from the counters they were spread over: on one counter the atomics of a sparse grid
// took turns (0.8 of 1.1 ms at 2048^2 nodes and 262144 markers).
__global__ __launch_bounds__(M2G_EMPTY) void m2g_count_empty(unsigned long long* counters, const unsigned long long* spread)
{
    const unsigned long long n = spread[(1 + threadIdx.x) * 16];
    if (n) atomicAdd(&counters[CNT_EMPTY], n);
}

// A tile's markers in LDS, column of cells by column (the cells of a column are contiguous in slot
// order), each column where the one before ends: its markers, at most one per thread, plus a spare slot
// per cell that ends the cell's list.  28 bytes a slot, 40 KB: four workgroups per CU.  What bounds the
// kernel is latency, so the workgroups in flight count (at the size below): 6.8 ms with four; 8.4 with
// three, columns of a fixed 204 slots and 52 KB; 10.1 with five and tiles of 8 x 5 nodes.  256 threads and
// two workgroups took 9.2, 128 threads and four, on smaller tiles, 9.5.
#define M2G_THREADS 192
#define M2G_COLS 9   // columns of cells, one more than of nodes
#define M2G_ROWS 12  // most cells of a column
#define M2G_SLOTS 1440
#define M2G_MARGIN 1.04
#define M2G_END 0x7fffffff
struct M2GTile {
    double dx[M2G_SLOTS], dy[M2G_SLOTS], v[M2G_SLOTS];
    int idx[M2G_SLOTS];
    int cell[M2G_COLS * (M2G_ROWS + 1)];  // first slot of a cell; per column one past its last cell
};

// One tile of nodes (a0..a1-1, b0..b1-1; cells a0..a1, b0..b1), by a workgroup.  0, or the rows of it that
// should fit if it does not.
// Each marker is read once per tile (coalesced in slot order) and its relative position computed once;
// the per-node merges then run on LDS.  Reading 32-byte records from global memory per node instead
// spread every load of a wave over 64 lines: 18.8 ms at 4096^2 nodes and 268 M markers, after 5.0 ms of
// sorting the cells and 3.3 ms of writing the records, where this takes 6.8.  With three workgroups per
// CU, 3.6 of 8.4 went to the loads (2.1 GB of indices and 7.9 GB of markers with the tiles' overlap), 1.5 to
// the sorting and 3.3 to the merges (one wave of a workgroup, a chain of LDS reads).  It is bound by
// latency: the loads of a tile are issued together, column by column without branches, and the cells are
// sorted by counting smaller indices, all columns in step.  Merging run by run of consecutive indices
// (fewer choices, uneven loops) took 9.8.
__device__ inline int m2g_tile(const M2GNodes& g, M2GTile& s, int a0, int a1, int b0, int b1)
{
    const int t = threadIdx.x;
    const int ncx = a1 - a0 + 1, ncy = b1 - b0 + 1, nce = ncy + 1;
    const int64_t ld = g.gny + 1;
    // the columns' segments of rec_idx
    int beg[M2G_COLS], num[M2G_COLS], most = 0, total = 0;
#pragma unroll
    for (int i = 0; i < M2G_COLS; ++i) {
        const int64_t k = (int64_t)(a0 + min(i, ncx - 1)) * ld + b0;
        beg[i] = g.off[k];
        num[i] = i < ncx ? g.off[k + ncy] - beg[i] : 0;
    }
#pragma unroll
    for (int i = 0; i < M2G_COLS; ++i) {
        most = max(most, num[i]);
        total += num[i];
    }
    if (most > M2G_THREADS || total + ncx * ncy > M2G_SLOTS)  // the same for every thread
        return max(1, min((int)(M2G_THREADS * ncy / (1.1f * most)), (int)(M2G_SLOTS * ncy / (1.1f * total + ncx * ncy))) - 1);
    int base[M2G_COLS];  // the columns' first slots
#pragma unroll
    for (int i = 0; i < M2G_COLS; ++i) base[i] = i ? base[i - 1] + num[i - 1] + ncy : 0;
    if (t < ncx * nce) {
        const int i = t / nce, j = t % nce;
        const int64_t k = (int64_t)(a0 + i) * ld + b0;
        int first = 0;
#pragma unroll
        for (int u = 1; u < M2G_COLS; ++u) first = u == i ? base[u] : first;
        s.cell[t] = first + g.off[k + j] - g.off[k] + j;
    }
    int m[M2G_COLS], place[M2G_COLS], lo[M2G_COLS], n[M2G_COLS];
    double rx[M2G_COLS], ry[M2G_COLS], rv[M2G_COLS];
    if (total > 0) {
        // marker indices, then positions and values: every load in bounds (a thread without a
        // marker reads the first one's), so that all are in flight together
#pragma unroll
        for (int u = 0; u < M2G_COLS; ++u) {
            m[u] = g.rec_idx[t < num[u] ? beg[u] + t : 0];
        }
#pragma unroll
        for (int u = 0; u < M2G_COLS; ++u) {
            rx[u] = g.x_m[m[u]];
            ry[u] = g.y_m[m[u]];
            rv[u] = g.val_m[m[u]];
        }
#pragma unroll
        for (int u = 0; u < M2G_COLS; ++u)
            if (t < num[u]) s.idx[base[u] + t] = m[u];
    }
    __syncthreads();
    int longest = 0;
    if (total > 0) {
#pragma unroll
        for (int u = 0; u < M2G_COLS; ++u) {
            place[u] = lo[u] = n[u] = 0;
            if (t - t % 64 >= num[u]) {  // nothing for the whole wave
                m[u] = -1;
                continue;
            }
            int64_t ix, iy;
            double dxij, dyij;
            topleft(g.xmin, g.ymin, rx[u], ry[u], g.dx, g.dy, ix, iy, dxij, dyij);
            rx[u] = dxij;
            ry[u] = dyij;
            // the marker's cell: its first slot (place) and its markers in the unsorted column
            const bool have = t < num[u];
            const int c = u * nce + (have ? (int)(iy - b0) : 0);
            place[u] = s.cell[c];
            lo[u] = have ? place[u] - (c - u * nce) : 0;
            n[u] = have ? lo[u] + s.cell[c + 1] - 1 - place[u] : 0;  // one past its last
            longest = max(longest, n[u] - lo[u]);
            if (!have) m[u] = -1;
        }
    }
    __syncthreads();
    if (total > 0) {
        // the marker's place in its cell: its markers of smaller index (a thread without a marker has n = lo)
        for (int q = 0; q < longest; ++q) {
#pragma unroll
            for (int u = 0; u < M2G_COLS; ++u) {
                const int other = s.idx[min(lo[u] + q, M2G_SLOTS - 1)];
                place[u] += (int)(lo[u] + q < n[u]) & (int)(other < m[u]);
            }
        }
    }
    __syncthreads();
    if (t < ncx * nce && t % nce > 0) s.idx[s.cell[t] - 1] = M2G_END;
    if (total > 0) {
#pragma unroll
        for (int u = 0; u < M2G_COLS; ++u) {
            if (m[u] < 0) continue;
            s.dx[place[u]] = rx[u];
            s.dy[place[u]] = ry[u];
            s.v[place[u]] = rv[u];
            s.idx[place[u]] = m[u];
        }
    }
    __syncthreads();
    // the nodes' merges, x fastest
    const int na = a1 - a0, nodes = na * (b1 - b0);
    for (int n = t; n < nodes; n += M2G_THREADS) {
        const int aa = n % na, bb = n / na;
        // cells: 0 TL (A,B), 1 TR (A-1,B), 2 BL (A,B-1), 3 BR (A-1,B-1)
        int p0 = s.cell[(aa + 1) * nce + bb + 1], p1 = s.cell[aa * nce + bb + 1];
        int p2 = s.cell[(aa + 1) * nce + bb], p3 = s.cell[aa * nce + bb];
        int h0 = s.idx[p0], h1 = s.idx[p1], h2 = s.idx[p2], h3 = s.idx[p3];
        double wt = 0.0, vw = 0.0;
        while (true) {
            const int best = min(min(h0, h1), min(h2, h3));
            if (best == M2G_END) break;
            const bool c0 = best == h0, c1 = best == h1, c2 = best == h2, c3 = best == h3;
            int p = p0;
            p = c1 ? p1 : p;
            p = c2 ? p2 : p;
            p = c3 ? p3 : p;
            const int nxt = s.idx[p + 1];
            const double dxij = s.dx[p], dyij = s.dy[p], val = s.v[p];
            const double wx = (c1 || c3) ? dxij : 1.0 - dxij;
            const double wy = (c2 || c3) ? dyij : 1.0 - dyij;
            const double w = wx * wy;
            wt = wt + w;
            vw = vw + w * val;
            ++p;
            p0 = c0 ? p : p0;
            p1 = c1 ? p : p1;
            p2 = c2 ? p : p2;
            p3 = c3 ? p : p3;
            h0 = c0 ? nxt : h0;
            h1 = c1 ? nxt : h1;
            h2 = c2 ? nxt : h2;
            h3 = c3 ? nxt : h3;
        }
        m2g_store(g, a0 + aa, b0 + bb, wt, vw);
    }
    return 0;
}

__global__ __launch_bounds__(M2G_THREADS) void m2g_tiles(M2GNodes g)
{
    __shared__ M2GTile s;
    const int tile = xcd_band(blockIdx.x, gridDim.x);
    const int a0 = (tile / g.nty) * g.tx, b0 = (tile % g.nty) * g.ty;
    const int a1 = min(a0 + g.tx, g.gnx), b1 = min(b0 + g.ty, g.gny);
    const int rows = m2g_tile(g, s, a0, a1, b0, b1);
    if (rows > 0 && threadIdx.x == 0) {
        if (g.ty > 1) {
            int* l = g.list + 2 * atomicAdd(&g.counters[CNT_OVERFLOW], (unsigned long long)((b1 - b0 + rows - 1) / rows));
            for (int b = b0; b < b1; b += rows, l += 2) {
                l[0] = tile * g.ty + b - b0;
                l[1] = rows;
            }
        } else {
            g.list2[atomicAdd(&g.spread[0], 1ull)] = tile;
        }
    }
}

// Step 5: the tiles that did not fit, in parts, and these in pieces of fewer rows where they do not fit.
__global__ __launch_bounds__(M2G_THREADS) void m2g_parts(M2GNodes g)
{
    __shared__ M2GTile s;
    const int n = (int)g.counters[CNT_OVERFLOW];
    for (int w = blockIdx.x; w < n; w += gridDim.x) {
        const int row = g.list[2 * w], tile = row / g.ty, row0 = (tile % g.nty) * g.ty, b0 = row0 + row % g.ty;
        const int a0 = (tile / g.nty) * g.tx, a1 = min(a0 + g.tx, g.gnx);
        int h = g.list[2 * w + 1];
        const int b1 = min(min(b0 + h, row0 + g.ty), g.gny);
        for (int b = b0; b < b1;) {
            const int to = min(b + h, b1);
            if (m2g_tile(g, s, a0, a1, b, to) > 0) {
                if (h > 1) {
                    h = (h + 1) / 2;
                    continue;
                }
                if (threadIdx.x == 0) g.list2[atomicAdd(&g.spread[0], 1ull)] = tile * g.ty + b - row0;
            }
            b = to;
            __syncthreads();
        }
    }
}

// Step 5, the cells of the rows that did not fit: each sorted in place by marker index by one workgroup, runs of
// M2G_RUN by counting smaller indices in LDS, longer cells by merging the runs through tmp (as long as
// rec_idx).  A cell that several rows share is sorted by the workgroup that first takes its mark in
// count.
#define M2G_RUN 1024
__device__ inline int m2g_far_rows(const M2GNodes& g)
{
    return g.all ? g.ntx * g.nty * g.ty : (int)g.spread[0];
}

__device__ inline void m2g_far_row(const M2GNodes& g, int l, int& a0, int& a1, int& b0, int& b1)
{
    const int w = g.all ? l : g.list2[l], tile = w / g.ty;
    a0 = (tile / g.nty) * g.tx;
    a1 = min(a0 + g.tx, g.gnx);
    b0 = (tile % g.nty) * g.ty + w % g.ty;
    b1 = min(b0 + 1, g.gny);  // none past the grid
}

__global__ __launch_bounds__(256) void m2g_far_sort(M2GNodes g, int* count, int* tmp)
{
    __shared__ int4 s_run[M2G_RUN / 4];
    __shared__ int s_mark;
    int* const s_idx = (int*)s_run;
    const int t = threadIdx.x;
    const int nl = m2g_far_rows(g), most = (g.tx + 1) * 2;
    const int64_t ld = g.gny + 1;
    for (int64_t w = blockIdx.x; w < (int64_t)nl * most; w += gridDim.x) {
        const int c = (int)(w % most);
        int a0, a1, b0, b1;
        m2g_far_row(g, (int)(w / most), a0, a1, b0, b1);
        const int ncy = b1 - b0 + 1;
        if (b0 >= b1 || c >= (a1 - a0 + 1) * ncy) continue;
        const int64_t k = (int64_t)(a0 + c / ncy) * ld + b0 + c % ncy;
        const int b = g.off[k], n = g.off[k + 1] - b;
        if (n < 2) continue;
        if (t == 0) s_mark = atomicExch(&count[k], -1);
        __syncthreads();
        const int mark = s_mark;
        __syncthreads();
        if (mark < 0) continue;
        for (int r = 0; r < n; r += M2G_RUN) {
            const int len = min(M2G_RUN, n - r);
            int mine[M2G_RUN / 256], rank[M2G_RUN / 256];
#pragma unroll
            for (int u = 0; u < M2G_RUN / 256; ++u) {
                const int i = u * 256 + t;
                mine[u] = i < len ? g.rec_idx[b + r + i] : M2G_END;
                s_idx[i] = mine[u];
                rank[u] = 0;
            }
            __syncthreads();
            for (int i = 0; i < (len + 3) / 4; ++i) {
                const int4 o = s_run[i];
#pragma unroll
                for (int u = 0; u < M2G_RUN / 256; ++u)
                    rank[u] += (int)(o.x < mine[u]) + (int)(o.y < mine[u]) + (int)(o.z < mine[u]) + (int)(o.w < mine[u]);
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < M2G_RUN / 256; ++u)
                if (u * 256 + t < len) g.rec_idx[b + r + rank[u]] = mine[u];
        }
        int *src = g.rec_idx + b, *dst = tmp + b;
        for (int64_t run = M2G_RUN; run < n; run *= 2) {
            __syncthreads();
            for (int i = t; i < n; i += 256) {
                const int v = src[i];
                const int64_t r = i / run, m0 = (r ^ 1) * run;
                int lo = (int)min((int64_t)n, m0), hi = (int)min((int64_t)n, m0 + run);
                const int first = lo;
                while (lo < hi) {
                    const int mid = lo + (hi - lo) / 2;
                    if (src[mid] < v) lo = mid + 1;
                    else hi = mid;
                }
                dst[(r & ~(int64_t)1) * run + (i - r * run) + (lo - first)] = v;
            }
            int* const other = src;
            src = dst;
            dst = other;
        }
        if (src != g.rec_idx + b) {
            __syncthreads();
            for (int i = t; i < n; i += 256) dst[i] = src[i];
        }
    }
}

// Orders a wave's LDS writes before its LDS reads of other lanes' values.
__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Step 5, their nodes: one wave per node.  Of each of the four cells the next 64 indices go to LDS; the
// markers up to the smallest last index of a cell that goes on are complete, find their place among the
// other cells' by binary search and leave their weights there, and two lanes add the two sums in that
// order.  At 64^2 nodes and 1024 markers per cell all passes take 1.3 ms; one thread per node, merging
// from global memory after one thread per cell had sorted, took 17 to 21.
__global__ __launch_bounds__(256) void m2g_far_nodes(M2GNodes g)
{
    __shared__ int s_idx[4][4][64];
    __shared__ double s_w[4][2][256];
    const int lane = threadIdx.x % 64, wv = threadIdx.x / 64;
    const int nl = m2g_far_rows(g), most = g.tx;
    const int64_t ld = g.gny + 1;
    for (int64_t w = (int64_t)blockIdx.x * 4 + wv; w < (int64_t)nl * most; w += (int64_t)gridDim.x * 4) {
        const int n = (int)(w % most);
        int a0, a1, b0, b1;
        m2g_far_row(g, (int)(w / most), a0, a1, b0, b1);
        const int na = a1 - a0;
        if (b0 >= b1 || n >= na * (b1 - b0)) continue;
        const int A = a0 + n % na + 1, B = b0 + n / na + 1;  // 1-based node
        const int64_t kc[4] = {(int64_t)A * ld + B, (int64_t)(A - 1) * ld + B, (int64_t)A * ld + (B - 1),
                               (int64_t)(A - 1) * ld + (B - 1)};
        int h[4], e[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            h[q] = g.off[kc[q]];
            e[q] = g.off[kc[q] + 1];
        }
        double sum = 0.0;  // of the weights in even lanes, of the weighted values in odd ones
        while (true) {
            int idx[4], end = M2G_END - 1, got = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                idx[q] = lane < e[q] - h[q] ? g.rec_idx[h[q] + lane] : M2G_END;
                s_idx[wv][q][lane] = idx[q];
                if (e[q] - h[q] > 64) end = min(end, __shfl(idx[q], 63));
            }
            wave_sync();
            double x[4], y[4], val[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int taken = __popcll(__ballot(idx[q] <= end));
                got += taken;
                h[q] += taken;
                if (idx[q] <= end) {
                    x[q] = g.x_m[idx[q]];
                    y[q] = g.y_m[idx[q]];
                    val[q] = g.val_m[idx[q]];
                }
            }
            if (got == 0) break;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (idx[q] > end) continue;
                int place = lane;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (r == q) continue;
                    int p = 0;
#pragma unroll
                    for (int step = 32; step > 0; step /= 2) p += s_idx[wv][r][p + step - 1] < idx[q] ? step : 0;
                    place += p + (int)(s_idx[wv][r][p] < idx[q]);
                }
                int64_t ix, iy;
                double dxij, dyij;
                topleft(g.xmin, g.ymin, x[q], y[q], g.dx, g.dy, ix, iy, dxij, dyij);
                const double wt = corner_weight(q, dxij, dyij);
                s_w[wv][0][place] = wt;
                s_w[wv][1][place] = wt * val[q];
            }
            wave_sync();
            const double* const add = s_w[wv][lane & 1];
            int i = 0;
            for (; i + 8 <= got; i += 8) {
                double a[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) a[u] = add[i + u];
#pragma unroll
                for (int u = 0; u < 8; ++u) sum = sum + a[u];
            }
            for (; i < got; ++i) sum = sum + add[i];
            wave_sync();
        }
        const double wt = __shfl(sum, 0), vw = __shfl(sum, 1);
        if (lane == 0) m2g_store(g, A - 1, B - 1, wt, vw);
    }
}

static int grid1d(int64_t n, int bs) { return (int)((n + bs - 1) / bs); }

static void launch_keys(const double* x_m, const double* y_m, int64_t nm, double xmin, double ymin, double dx, double dy,
                        int gnx, int gny, int* key, int* count, int* loc, unsigned long long* counters, hipStream_t st)
{
    if (nm >= M2G_MANY)
        hipLaunchKernelGGL(m2g_keys<M2G_PER_THREAD>, dim3(grid1d(nm, 256 * M2G_PER_THREAD)), dim3(256), 0, st, x_m, y_m, nm,
                           xmin, ymin, dx, dy, gnx, gny, key, count, loc, counters);
    else if (nm > 0)
        hipLaunchKernelGGL(m2g_keys<1>, dim3(grid1d(nm, 256)), dim3(256), 0, st, x_m, y_m, nm, xmin, ymin, dx, dy, gnx, gny,
                           key, count, loc, counters);
}

hipError_t m2g_cell_keys(M2GScratch& S, double xmin, double ymin, int gnx, int gny, const double* x_m,
                         const double* y_m, int64_t nm, double dx, double dy, int* keys, int* counts, hipStream_t st)
{
    const int64_t ncells = (int64_t)(gnx + 1) * (gny + 1);
    hipLaunchKernelGGL(zero_counters, dim3(1), dim3(1024), 0, st, S.counters, (unsigned long long*)nullptr);
    hipLaunchKernelGGL(fill_int, dim3(1024), dim3(256), 0, st, counts, ncells, 0);
    launch_keys(x_m, y_m, nm, xmin, ymin, dx, dy, gnx, gny, keys, counts, nullptr, S.counters, st);
    return hipGetLastError();
}

hipError_t m2g_run(M2GScratch& S, double xmin, double ymin, double* val_grid, int gnx, int gny, const double* x_m,
                   const double* y_m, const double* val_m, int64_t nm, double dx, double dy, double* val_wt_sum,
                   double* wt_sum, int ws_nx, int ws_ny, hipStream_t st)
{
    const int64_t ncells = (int64_t)(gnx + 1) * (gny + 1);
    const int nblk = (int)((ncells + SCAN_TILE - 1) / SCAN_TILE);
    const int fillgrid = 1024;
    hipLaunchKernelGGL(zero_counters, dim3(1), dim3(1024), 0, st, S.counters, S.spread);
    hipLaunchKernelGGL(fill_int, dim3(fillgrid), dim3(256), 0, st, S.count, ncells, 0);
    if (wt_sum) {
        hipLaunchKernelGGL(fill_dbl, dim3(fillgrid), dim3(256), 0, st, wt_sum, (int64_t)ws_nx * ws_ny, 0.0);
        hipLaunchKernelGGL(fill_dbl, dim3(fillgrid), dim3(256), 0, st, val_wt_sum, (int64_t)ws_nx * ws_ny, 0.0);
    }
    launch_keys(x_m, y_m, nm, xmin, ymin, dx, dy, gnx, gny, S.key, S.count, S.loc, S.counters, st);
    hipLaunchKernelGGL(scan_block_sums, dim3(nblk), dim3(SCAN_BLOCK), 0, st, S.count, ncells, S.blocksums);
    hipLaunchKernelGGL(scan_top, dim3(1), dim3(SCAN_TOP), 0, st, S.blocksums, nblk);
    hipLaunchKernelGGL(scan_apply, dim3(nblk), dim3(SCAN_BLOCK), 0, st, S.count, ncells, S.blocksums, S.offset);
    if (nm >= M2G_MANY)
        hipLaunchKernelGGL(m2g_scatter<M2G_PER_THREAD>, dim3(grid1d(nm, 256 * M2G_PER_THREAD)), dim3(256), 0, st, S.key,
                           S.loc, nm, S.offset, S.rec_idx);
    else if (nm > 0)
        hipLaunchKernelGGL(m2g_scatter<1>, dim3(grid1d(nm, 256)), dim3(256), 0, st, S.key, S.loc, nm, S.offset, S.rec_idx);
    M2GNodes g{S.offset, S.rec_idx, x_m, y_m, val_m, xmin, ymin, dx, dy, gnx, gny, 8, 1, 0, 0,
               val_grid, val_wt_sum, wt_sum, ws_nx, S.counters, S.spread, S.loc, S.loc + nm / 2, false};
    // Tiles of 8 columns (a row of values is half a 128-byte line; fewer where 9 x 2 cells do not fit), at
    // most M2G_ROWS - 1 rows, as high as fit at the mean density: a column fills three quarters of the
    // threads, the tile the slots with M2G_MARGIN to spare (1.15 makes tiles of 8 x 7 at 16 markers per
    // cell: 7.5 ms at the size above against 6.8).  Advection by a continuous flow keeps lattice markers
    // that even (512^2 to 1500^2 nodes 6 to 13% faster than with three quarters of 1836 slots); in random
    // order about a tile in twenty goes in parts at 16 per cell (512^2: 0.61 ms, 0.60 before), and where
    // markers cluster many do, each in as many as it needs (a normal distribution in x 0.86 ms, 0.87 before,
    // in x and y 1.16, 1.24).  (A listed tile has more than M2G_THREADS markers and a marker lies in at most
    // four tiles; a tile has at most M2G_ROWS - 1 parts of two words each: both lists fit S.loc.)  Above
    // M2G_FAR markers per cell all nodes take the kernels of step 5: 4.2 M markers in random order take
    // 0.98 ms by tiles and 1.42 by step 5 at 72 per cell, 1.43 and 1.38 at 86 (in lattice order 0.78 and 0.73 at
    // 76).
    const double per_cell = std::max(1.0, (double)nm / ((double)gnx * gny));
    g.all = per_cell > M2G_FAR;
    if (!g.all) {
        const double slots = M2G_MARGIN * per_cell + 1.0;  // of a cell, the spare one included
        const int rows = std::min(0.75 * M2G_THREADS / per_cell, M2G_SLOTS / (M2G_COLS * slots));
        g.ty = std::max(1, std::min(M2G_ROWS - 1, rows - 1));
        g.tx = std::min(M2G_COLS, (int)(M2G_SLOTS / ((g.ty + 1) * slots))) - 1;
    }
    g.ntx = (gnx + g.tx - 1) / g.tx;
    g.nty = (gny + g.ty - 1) / g.ty;
    if (!g.all) {
        hipLaunchKernelGGL(m2g_tiles, dim3(g.ntx * g.nty), dim3(M2G_THREADS), 0, st, g);
    }
    // No tile can be listed where all markers fit into one: three launches less, 22 us of kernel time instead of
    // 28 for nine markers.
    if (g.all || nm > M2G_THREADS) {
        if (!g.all && g.ty > 1) hipLaunchKernelGGL(m2g_parts, dim3(1024), dim3(M2G_THREADS), 0, st, g);
        hipLaunchKernelGGL(m2g_far_sort, dim3(2048), dim3(256), 0, st, g, S.count, S.key);
        hipLaunchKernelGGL(m2g_far_nodes, dim3(2048), dim3(256), 0, st, g);
    }
    hipLaunchKernelGGL(m2g_count_empty, dim3(1), dim3(M2G_EMPTY), 0, st, S.counters, S.spread);
    return hipGetLastError();
}

}  // namespace sf
