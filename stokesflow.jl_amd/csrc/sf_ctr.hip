// sf_ctr.hip -- launches of the register-resident FP32 correction pass (sf_ctr_tile.h) for gfx950.
#include <algorithm>
#include <cmath>

#include "sf_ctr_tile.h"

namespace sf {

#define CTR_MAX_WAVES 16

__device__ inline int ctr_xcd_remap(int k, int total)
{
    const int xcd = k % 8, idx = k / 8, per = total / 8, rem = total % 8;
    return (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
}

template <int R>
__global__ __launch_bounds__(64 * CTR_MAX_WAVES) void ctr_tile_f32(CorrParams p, int k)
{
    __shared__ float lds[CTR_LDS(CTR_MAX_WAVES)];
    const int logical = ctr_xcd_remap(blockIdx.x, gridDim.x);
    const int nstrips = p.nstrips;
    ctr_tile<R>(p, k, p.seg, logical % nstrips, logical / nstrips, lds);
}

static int64_t ctr_tiles(int nx, int ny, int rows, int k)
{
    const int out = SF_WAVE - 2 * k, seg = rows - 2 * k;
    return (int64_t)((nx - 1 + out - 1) / out) * ((ny + seg - 1) / seg);
}

// The passes of n grids (one launch for all): one shape, and per grid the sweeps k[i].  A tile takes a
// fixed part (loads, pseudo-time steps, stores) and K sweeps; workgroups that share a CU slow each
// other by CTR_SHARE each, and no pass is faster than its bytes.  One grid: the launch and the rounds of
// workgroups; several: a launch, the tiles' time spread over the chip, and half a tile's until the last
// workgroup ends, each grid with the k that serves the sum best.
//
// Measured (us per sweep, best shape, the plan's, and the one-wave passes): 64^2 0.93, 0.93, 2.4; 256^2
// 1.12, 1.16, 2.5; 512^2 1.76, 1.96, 3.8; 768^2 2.57, 2.59, 5.4; 1000x777 3.35, 3.45, 5.6; 1400^2 6.7, 7.0, 9.9;
// 2048^2 12.3, 13.0, 14.6; 3000^2 27.1, 28.0, 32.8; 4096^2 51.5, 51.8, 60.9.  The last are 8 waves of six
// rows at the memory's rate: a pass moves 86 bytes per node, halos included, 5.6 TB/s.  Taking the tiles
// in square panels, for the halos' sake, gained nothing (4 wide: 5% slower).  Above 3072 nodes per side
// a pass keeps the documented five sweeps (six would be 8% faster per sweep at 4096^2).
#define CTR_SHARE 0.45
CorrPlan corr_plan(const int* nx, const int* ny, int n, int* k)
{
    struct Shape {
        int r, waves, per_cu;  // rows per wave, waves, workgroups a CU holds
        double fixed, iter;    // us
    };
    static const Shape shapes[] = {{1, 8, 4, 0.8, 0.40},  {1, 16, 2, 1.1, 0.45}, {2, 8, 4, 0.9, 0.55},  {2, 12, 2, 2.1, 0.60},
                                   {2, 16, 2, 2.4, 0.68}, {3, 8, 3, 1.5, 0.78},  {3, 12, 2, 2.4, 0.95}, {4, 12, 1, 3.5, 1.10},
                                   {3, 16, 1, 3.1, 1.10}, {4, 16, 1, 4.7, 1.33}, {5, 8, 2, 2.8, 1.18},  {6, 8, 2, 3.7, 1.30},
                                   {5, 16, 1, 5.5, 1.75}, {6, 16, 1, 6.6, 2.03}};
    const int cus = 256;
    const double launch_us = n == 1 ? 2.5 : 5.0;
    CorrPlan best{};
    double best_us = 1e300;
    int kk[WIDE_MAX];
    double nodes = 0.0;
    for (int i = 0; i < n; ++i) nodes += (double)nx[i] * ny[i];
    const double bytes_per_us = nodes * 64.0 > 260e6 ? 5.6e6 : 6.5e6;  // from HBM or cached
    for (const Shape& sh : shapes) {
        const int rows = sh.r * sh.waves;
        int64_t least = 0;
        for (int i = 0; i < n; ++i) least += ctr_tiles(nx[i], ny[i], rows, 2);  // workgroups of a short pass
        double sum = 0.0, slowest = 0.0;
        for (int i = 0; i < n; ++i) {
            const bool five = std::max(nx[i], ny[i]) > 3072;
            double us = 1e300, share = 0.0, alone = 0.0;
            for (int c = five ? 5 : 2; c <= (five ? 5 : CORR_MAX_K) && 2 * c < rows; ++c) {
                const double load = 64.0 * rows * 44.0, bytes = load + (SF_WAVE - 2.0 * c) * (rows - 2.0 * c) * 20.0;
                const int64_t wgs = ctr_tiles(nx[i], ny[i], rows, c);
                const int shared = (int)std::min<int64_t>(sh.per_cu, ((n == 1 ? wgs : least) + cus - 1) / cus);
                // what the first round's loads take beyond the fixed part; later rounds' too if nothing
                // else runs on the CU meanwhile
                const int64_t first = n == 1 ? std::min<int64_t>(wgs, cus * shared) : cus * shared;
                const double wait = n > 1 && least <= cus ? 0.0 : std::max(0.0, first * load / bytes_per_us - sh.fixed);
                const double tile = sh.fixed + c * sh.iter + (shared == 1 ? wait : 0.0);
                const double rounds = (double)wgs / (cus * shared);
                double own = n > 1 ? rounds : (sh.per_cu == 1 ? std::ceil(rounds) : std::max(1.0, rounds));
                own *= tile * (1.0 + CTR_SHARE * (shared - 1));
                own = std::max(own, wgs * bytes / bytes_per_us) / c;
                const double rest = (launch_us + (shared > 1 ? wait : 0.0) + (n == 1 ? 0.0 : 0.5 * tile)) / c;
                if (own + rest / n < us) {
                    us = own + rest / n;
                    share = own;
                    alone = rest;
                    kk[i] = c;
                }
            }
            if (us == 1e300) share = 1e300;
            sum += share;
            slowest = std::max(slowest, alone);
        }
        if (sum + slowest < best_us) {
            best_us = sum + slowest;
            best = CorrPlan{sh.r, sh.waves};
            std::copy(kk, kk + n, k);
        }
    }
    return best;
}

int corr_plan_tiles(const CorrPlan& plan, int nx, int ny, int k) { return (int)ctr_tiles(nx, ny, plan.r * plan.waves, k); }

hipError_t launch_corr_resident(const CorrParams& p0, int k, int r, int waves, hipStream_t s)
{
    if (waves < 1 || waves > CTR_MAX_WAVES || k < 1 || 2 * k >= SF_WAVE || waves * r <= 2 * k) return hipErrorInvalidValue;
    CorrParams p = p0;
    p.seg = waves * r - 2 * k;
    const int out = SF_WAVE - 2 * k;
    p.nstrips = (p.nx - 1 + out - 1) / out;
    p.ntiles = p.nstrips * ((p.ny + p.seg - 1) / p.seg);
    const dim3 grid(p.ntiles), block(64 * waves);
    switch (r) {
        case 1: hipLaunchKernelGGL(ctr_tile_f32<1>, grid, block, 0, s, p, k); break;
        case 2: hipLaunchKernelGGL(ctr_tile_f32<2>, grid, block, 0, s, p, k); break;
        case 3: hipLaunchKernelGGL(ctr_tile_f32<3>, grid, block, 0, s, p, k); break;
        case 4: hipLaunchKernelGGL(ctr_tile_f32<4>, grid, block, 0, s, p, k); break;
        case 5: hipLaunchKernelGGL(ctr_tile_f32<5>, grid, block, 0, s, p, k); break;
        case 6: hipLaunchKernelGGL(ctr_tile_f32<6>, grid, block, 0, s, p, k); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// One launch of the wide refined mode: slot i runs slot_k[i] sweeps.
template <int R>
__global__ __launch_bounds__(64 * CTR_MAX_WAVES) void wide_ctr_kernel(WideCorrArgs a)
{
    __shared__ float lds[CTR_LDS(CTR_MAX_WAVES)];
    const int t_glob = ctr_xcd_remap(blockIdx.x, gridDim.x);
    if (t_glob >= a.tile_start[a.n_active]) return;
    int lo = 0, hi = a.n_active - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.tile_start[mid] <= t_glob) lo = mid;
        else hi = mid - 1;
    }
    const int t = t_glob - a.tile_start[lo], k = a.slot_k[lo];
    const CorrParams __attribute__((address_space(4)))& p = ((const CorrParams __attribute__((address_space(4)))*)a.desc)[a.slot_desc[lo]];
    const int out = SF_WAVE - 2 * k, nstrips = (p.nx - 1 + out - 1) / out;
    ctr_tile<R>(p, k, (int)(blockDim.x >> 6) * R - 2 * k, t % nstrips, t / nstrips, lds);
}

hipError_t launch_wide_corr(const WideCorrArgs& a, const CorrPlan& plan, hipStream_t s)
{
    const int total = a.tile_start[a.n_active];
    if (total <= 0) return hipSuccess;
    for (int i = 0; i < a.n_active; ++i)
        if (a.slot_k[i] < 1 || a.slot_k[i] > CORR_MAX_K || 2 * a.slot_k[i] >= plan.waves * plan.r) return hipErrorInvalidValue;
    const dim3 grid(total), block(64 * plan.waves);
    switch (plan.r) {
        case 1: hipLaunchKernelGGL(wide_ctr_kernel<1>, grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL(wide_ctr_kernel<2>, grid, block, 0, s, a); break;
        case 3: hipLaunchKernelGGL(wide_ctr_kernel<3>, grid, block, 0, s, a); break;
        case 4: hipLaunchKernelGGL(wide_ctr_kernel<4>, grid, block, 0, s, a); break;
        case 5: hipLaunchKernelGGL(wide_ctr_kernel<5>, grid, block, 0, s, a); break;
        case 6: hipLaunchKernelGGL(wide_ctr_kernel<6>, grid, block, 0, s, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace sf
