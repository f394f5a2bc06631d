// sf_ptr.hip -- launches of the register-resident PT pass (sf_ptr_tile.h) for gfx950, and the choice
// between it and the wave-pipelined pass.
#include <algorithm>
#include <cmath>

#include "sf_ptr_tile.h"

namespace sf {

#define PTR_MAX_WAVES 16

template <int R>
__global__ __launch_bounds__(64 * PTR_MAX_WAVES) void ptr_tile_f64(PTParams p, int k)
{
    __shared__ double lds[PTR_LDS(PTR_MAX_WAVES)];
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int nstrips = p.nstrips;
    PTROnce once;
    ptr_tile<R>(p, k, p.seg, logical % nstrips, logical / nstrips, lds, once);
}

hipError_t launch_pt_resident(const PTParams& p0, int k, int r, int waves, hipStream_t s)
{
    if (waves < 1 || waves > PTR_MAX_WAVES || k < 1 || 2 * k >= SF_WAVE || waves * r <= 2 * k) return hipErrorInvalidValue;
    if ((int64_t)(p0.nx + 2) * (p0.ny + 2) >= PTR_MAX_NODES) return hipErrorInvalidValue;  // 32-bit byte offsets
    PTParams p = p0;
    p.seg = waves * r - 2 * k;
    p.nstrips = (p.nx - 1 + (SF_WAVE - 2 * k) - 1) / (SF_WAVE - 2 * k);  // columns 0..nx-2 carry outputs
    p.ntiles = p.nstrips * ((p.ny + p.seg - 1) / p.seg);
    const dim3 grid(p.ntiles), block(64 * waves);
    switch (r) {
        case 1: hipLaunchKernelGGL(ptr_tile_f64<1>, grid, block, 0, s, p, k); break;
        case 2: hipLaunchKernelGGL(ptr_tile_f64<2>, grid, block, 0, s, p, k); break;
        case 3: hipLaunchKernelGGL(ptr_tile_f64<3>, grid, block, 0, s, p, k); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

struct Shape {
    int waves, r;
    double fixed, iter;  // us, see pt_plan_resident
};
static const Shape shapes[] = {{8, 1, 0.6, 0.54},  {12, 1, 1.1, 0.61}, {16, 1, 1.6, 0.72}, {8, 2, 1.7, 0.79},
                               {12, 2, 2.3, 1.01}, {16, 2, 2.9, 1.26}, {12, 3, 3.1, 1.5},  {16, 3, 4.2, 1.85}};

static const double pipe_step[3] = {0.55, 0.72, 0.94};  // us per row step, workgroups per CU

#define WIDE_PIPE_MARGIN 1.15  // see wide_plan

static int wide_pipe_rows(int ny, int h)
{
    const int nseg = (ny + h - 1) / h;
    return (ny + nseg - 1) / nseg;
}

static int64_t resident_tiles(int nx, int ny, int rows, int k)
{
    const int out = SF_WAVE - 2 * k, seg = rows - 2 * k;
    return (int64_t)((nx - 1 + out - 1) / out) * ((ny + seg - 1) / seg);
}

// The pass of a grid: the shape with the least modelled time per iteration.  Both models are fits
// to sweeps on MI355X (back-to-back launches, us), for a chip of 256 CUs.
//
// Resident: a launch (2.5) plus rounds of one workgroup per CU, each a fixed part (loads, pseudo-time
// steps, stores; more where most CUs load at once) and K iterations.  Fixed part / iteration: 8 x 1
// rows 0.6 / 0.54, 12 x 1 1.1 / 0.61, 16 x 1 1.6 / 0.72, 8 x 2 1.7 / 0.79, 12 x 2 2.3 / 1.01, 16 x 2 2.9 /
// 1.26, 12 x 3 3.1 / 1.5, 16 x 3 4.2 / 1.85 (four rows per wave spill).
// Pipelined: rows + K + lag steps of 0.55, 0.72 and 0.94 us with one, two and three workgroups
// per CU (up to L2- and MALL-sized grids; 0.58, 0.82, 1.06 from HBM, in the same proportions).
//
// Measured against the passes before (us per iteration): 64^2 1.30 (2.6), 301x257 1.64 (3.1), 512^2 2.6
// (4.65), 700^2 3.85 (about 6.5) resident; 1024^2 6.3 (9.1), 2048^2 18.7 (28), 4096^2 64-66 (109)
// pipelined.  They cross near 730^2: resident 800^2 5.3 against 4.7, pipelined 600^2 3.6 against 2.95.
PTPlan pt_plan_resident(int nx, int ny, int kmax, double launch_us, double kept_us, double* us_per_iter)
{
    const int cus = 256;
    PTPlan best{};
    double best_us = 1e300;
    if ((int64_t)(nx + 2) * (ny + 2) < PTR_MAX_NODES)
        for (const Shape& sh : shapes)
            for (int k = 2; k <= kmax && 2 * k < sh.waves * sh.r; ++k) {
                const int64_t wgs = resident_tiles(nx, ny, sh.waves * sh.r, k);
                const double rounds = (double)((wgs + cus - 1) / cus);
                const double fixed = sh.fixed * (1.0 + 0.5 * std::min(1.0, (double)wgs / cus));
                double us = (launch_us + rounds * (fixed + k * sh.iter)) / k;
                if (kept_us > 0.0 && wgs <= cus) us = (kept_us + k * sh.iter) / k;
                if (us < best_us) {
                    best_us = us;
                    best = PTPlan{PT_PLAN_RESIDENT, k, 0, sh.r, sh.waves};
                }
            }
    *us_per_iter = best_us;
    return best;
}

PTPlan pt_plan(int nx, int ny)
{
    const int cus = 256;
    double best_us;
    PTPlan best = pt_plan_resident(nx, ny, PT_PLAN_MAX_K, 2.5, 0.0, &best_us);
    const int k = PT_PLAN_MAX_K, lag = 9;
    const int strips = (nx - 1 + SF_WAVE - 2 * k - 1) / (SF_WAVE - 2 * k);
    for (int nseg = 1; nseg <= ny && (int64_t)strips * (nseg - 1) < 12 * cus; ++nseg) {
        const int rows = (ny + nseg - 1) / nseg;
        const int64_t wgs = (int64_t)strips * ((ny + rows - 1) / rows);
        const int64_t full = (wgs - 1) / (3 * cus);  // whole rounds of three per CU before the last
        const int per_cu = (int)((wgs - full * 3 * cus + cus - 1) / cus);
        const double us = (2.5 + (rows + k + lag) * (full * pipe_step[2] + pipe_step[per_cu - 1])) / k;
        if (us < best_us) {
            best_us = us;
            best = PTPlan{PT_PLAN_PIPE, k, rows, 0, 0};
        }
    }
    // Flat grids: a wave of the one-wave passes of four iterations marches over the whole height (from 16
    // rows on the two are equal within 5%).  Its row step takes 2.2 us with two waves per SIMD and 1.6 with one (ptk_default_rows); the pipelined
    // model is 15% short there (WIDE_PIPE_MARGIN).  us per iteration, one-wave and the plan: 100000x4
    // 6.9, 9.2; 100000x8 8.9, 9.9; 250000x6 16.5, 20.1; 50000x4 5.2, 5.8; but 50000x11 7.7, 6.7.
    if (ny < 16) {
        const double waves = (nx - 1 + 55) / 56;
        const double ow_us = (2.5 + (ny + 7) * (waves <= 4 * cus ? 1.6 : 2.2 * std::max(1.0, waves / (8 * cus)))) / 4;
        if (ow_us < best_us * (best.kind == PT_PLAN_PIPE ? WIDE_PIPE_MARGIN : 1.0)) best = PTPlan{};
    }
    return best;
}

// The wide passes of n grids, one launch for all.  Resident: one shape, and per grid the iterations
// k[i].  A pass is a launch, the tiles' time spread over the CUs, and on average half a tile's time until
// the last workgroup ends; each grid takes the k that serves that sum best, and the shape is the one
// whose slowest grid gets on fastest.  The fixed part is the single grid's while the tiles fit the chip
// at once; beyond, the CUs load in step and it is the tile's bytes at the memory's rate (2048^2: 15 us of
// 24 per round).  Pipelined (K = 7): as pt_plan, with one height for all grids.
//
// Measured (us per iteration of the whole set; resident, pipelined, one-wave passes of up to four
// before): one 64^2 1.9, 3.1, 3.1; 64 x 64^2 7.2, 8.1, 9.9; 4 x 100x90 2.1, 3.2, 3.4; 16 x 256^2 11.2, 8.5, 11.2;
// 64 x 256^2 48, 32, 43; 8 x 512^2 17.6, 12.9, 18.0; one 2048^2 34, 24, 32.  The pipelined model gains
// WIDE_PIPE_MARGIN too much on sets near the line (it has the row steps but not the pipeline's start).
WidePlan wide_plan(const int* nx, const int* ny, int n, int* k, int* rows)
{
    const int cus = 256;
    const double launch_us = 5.0;
    WidePlan best{};
    double best_us = 1e300, nodes = 0.0;
    for (int i = 0; i < n; ++i) nodes += (double)nx[i] * ny[i];
    const double bytes_per_us = nodes * 144.0 < 200e6 ? 10e6 : 5.5e6;  // cached or from HBM
    int kk[WIDE_MAX];
    for (const Shape& sh : shapes) {
        const int h = sh.waves * sh.r;
        const double load = std::max(1.5 * sh.fixed, 64.0 * h * 104.0 * cus / bytes_per_us);
        double sum = 0.0, slowest = 0.0;
        int64_t least = 0;
        for (int i = 0; i < n; ++i) least += resident_tiles(nx[i], ny[i], h, 2);
        const double fixed = least > cus ? load : 1.5 * sh.fixed;
        for (int i = 0; i < n; ++i) {
            double us = 1e300, share = 0.0, alone = 0.0;
            for (int c = 2; c <= WIDE_RESIDENT_MAX_K && 2 * c < h; ++c) {
                const double tile = fixed + c * sh.iter;
                const double own = (double)resident_tiles(nx[i], ny[i], h, c) * tile / (cus * c);
                const double rest = (launch_us + 0.5 * tile) / c;
                if (own + rest / n < us) {
                    us = own + rest / n;
                    share = own;
                    alone = rest;
                    kk[i] = c;
                }
            }
            sum += share;
            slowest = std::max(slowest, alone);
        }
        if (sum + slowest < best_us) {
            best_us = sum + slowest;
            best = WidePlan{0, sh.r, sh.waves};
            std::copy(kk, kk + n, k);
        }
    }
    int height = 0;
    for (int h = 16; h <= 4096; h += h / 4) {
        int64_t wgs = 0;
        double work = 0.0;
        int longest = 0;
        for (int i = 0; i < n; ++i) {
            const int seg = wide_pipe_rows(ny[i], h), tiles = wide_pipe_tiles(nx[i], ny[i], seg);
            wgs += tiles;
            work += (double)tiles * (seg + 16);
            longest = std::max(longest, seg + 16);
        }
        const int per_cu = (int)std::min<int64_t>(3, (wgs + cus - 1) / cus);
        double us = longest * pipe_step[per_cu - 1];
        if (wgs > 3 * cus) us = work * pipe_step[2] / (3 * cus) + 0.5 * us;
        us = WIDE_PIPE_MARGIN * (launch_us + us) / WIDE_PIPE_K;
        if (us < best_us) {
            best_us = us;
            height = h;
        }
    }
    if (height)
        for (int i = 0; i < n; ++i) {
            best = WidePlan{1, 3, PTR_MAX_WAVES};  // what is left before a check: resident
            k[i] = WIDE_PIPE_K;
            rows[i] = wide_pipe_rows(ny[i], height);
        }
    return best;
}

// Slot i runs slot_pf[i] >> 1 iterations.
template <int R>
__global__ __launch_bounds__(64 * PTR_MAX_WAVES) void wide_ptr_kernel(WideArgs a)
{
    __shared__ double lds[PTR_LDS(PTR_MAX_WAVES)];
    int t;
    const int i = wide_slot(a, &t);
    if (i < 0) return;
    const int k = a.slot_pf[i] >> 1;
    const auto& pp = ((WideInstC*)a.desc)[a.slot_inst[i]].wpt[a.slot_pf[i] & 1];
    const int out = SF_WAVE - 2 * k, nstrips = (pp.nx - 1 + out - 1) / out;
    PTROnce once;
    ptr_tile<R>(pp, k, (int)(blockDim.x >> 6) * R - 2 * k, t % nstrips, t / nstrips, lds, once);
}

int wide_resident_tiles(const WidePlan& plan, int nx, int ny, int k)
{
    return (int)resident_tiles(nx, ny, plan.waves * plan.r, k);
}

hipError_t launch_wide_resident(const WideArgs& a, const WidePlan& plan, hipStream_t s)
{
    const int total = a.tile_start[a.n_active];
    if (total <= 0) return hipSuccess;
    for (int i = 0; i < a.n_active; ++i) {
        const int k = a.slot_pf[i] >> 1;
        if (k < 1 || k > WIDE_RESIDENT_MAX_K || 2 * k >= plan.waves * plan.r) return hipErrorInvalidValue;
    }
    const dim3 grid(total), block(64 * plan.waves);
    switch (plan.r) {
        case 1: hipLaunchKernelGGL(wide_ptr_kernel<1>, grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL(wide_ptr_kernel<2>, grid, block, 0, s, a); break;
        case 3: hipLaunchKernelGGL(wide_ptr_kernel<3>, grid, block, 0, s, a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_pt_plan(const PTParams& p, const PTPlan& plan, int k, hipStream_t s)
{
    if (plan.kind == PT_PLAN_RESIDENT) return launch_pt_resident(p, k, plan.r, plan.waves, s);
    if (k >= 5) return launch_pt_pipe(p, k, plan.rows, s);
    PTParams q = p;
    q.seg = 0;  // what is left before a check: the one-wave passes' own tiles
    return launch_pt_multi(q, k, s);
}

}  // namespace sf
