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
    ptr_tile<R>(p, k, p.seg, logical % nstrips, logical / nstrips, lds);
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
// (4.65), 700^2 3.85 (about 6.5) resident; 1024^2 6.3 (9.1), 2048^2 19.4 (29.4), 4096^2 69.7 (112)
// pipelined.  They cross near 730^2: resident 800^2 5.3 against 4.7, pipelined 600^2 3.6 against 2.95.
PTPlan pt_plan_resident(int nx, int ny, int kmax, double launch_us, double* us_per_iter)
{
    struct Shape {
        int waves, r;
        double fixed, iter;
    };
    static const Shape shapes[] = {{8, 1, 0.6, 0.54},  {12, 1, 1.1, 0.61}, {16, 1, 1.6, 0.72}, {8, 2, 1.7, 0.79},
                                   {12, 2, 2.3, 1.01}, {16, 2, 2.9, 1.26}, {12, 3, 3.1, 1.5},  {16, 3, 4.2, 1.85}};
    const int cus = 256;
    PTPlan best{};
    double best_us = 1e300;
    if ((int64_t)(nx + 2) * (ny + 2) < PTR_MAX_NODES)
        for (const Shape& sh : shapes)
            for (int k = 2; k <= kmax && 2 * k < sh.waves * sh.r; ++k) {
                const int out = SF_WAVE - 2 * k, seg = sh.waves * sh.r - 2 * k;
                const int64_t wgs = (int64_t)((nx - 1 + out - 1) / out) * ((ny + seg - 1) / seg);
                const double rounds = (double)((wgs + cus - 1) / cus);
                const double fixed = sh.fixed * (1.0 + 0.5 * std::min(1.0, (double)wgs / cus));
                const double us = (launch_us + rounds * (fixed + k * sh.iter)) / k;
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
    static const double step[3] = {0.55, 0.72, 0.94};
    const int cus = 256;
    double best_us;
    PTPlan best = pt_plan_resident(nx, ny, PT_PLAN_MAX_K, 2.5, &best_us);
    const int k = PT_PLAN_MAX_K, lag = 9;
    const int strips = (nx - 1 + SF_WAVE - 2 * k - 1) / (SF_WAVE - 2 * k);
    for (int nseg = 1; nseg <= ny && (int64_t)strips * (nseg - 1) < 12 * cus; ++nseg) {
        const int rows = (ny + nseg - 1) / nseg;
        const int64_t wgs = (int64_t)strips * ((ny + rows - 1) / rows);
        const int64_t full = (wgs - 1) / (3 * cus);  // whole rounds of three per CU before the last
        const int per_cu = (int)((wgs - full * 3 * cus + cus - 1) / cus);
        const double us = (2.5 + (rows + k + lag) * (full * step[2] + step[per_cu - 1])) / k;
        if (us < best_us) {
            best_us = us;
            best = PTPlan{PT_PLAN_PIPE, k, rows, 0, 0};
        }
    }
    return best;
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
