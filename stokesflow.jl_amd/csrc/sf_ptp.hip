// sf_ptp.hip -- launches of the wave-pipelined PT pass (sf_ptp_tile.h) for gfx950.
#include "sf_ptp_tile.h"

namespace sf {

// One workgroup per tile, XCD-banded tile order (as the one-wave passes).
template <int K>
__global__ __launch_bounds__(64 * PTPShape<K>::WAVES, 3) void ptp_tile_f64(PTParams p)
{
    __shared__ double lds[PTPShape<K>::LDS];
    const int logical = xcd_remap(blockIdx.x, gridDim.x);
    const int nstrips = p.nstrips;
    // the kernel's only argument, read in place
    ptp_tile<K>(*(PTParamsC*)__builtin_amdgcn_kernarg_segment_ptr(), p.seg, logical % nstrips, logical / nstrips, lds);
}

template <int K>
static hipError_t launch_k(const PTParams& p0, int rows, hipStream_t s)
{
    PTParams p = p0;
    p.seg = rows;
    p.nstrips = (p.nx - 1 + PTPShape<K>::OUT - 1) / PTPShape<K>::OUT;  // columns 0..nx-2 carry outputs
    p.ntiles = p.nstrips * ((p.ny + rows - 1) / rows);
    hipLaunchKernelGGL(ptp_tile_f64<K>, dim3(p.ntiles), dim3(64 * PTPShape<K>::WAVES), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_pt_pipe(const PTParams& p, int k, int rows, hipStream_t s)
{
    if (rows < 1) return hipErrorInvalidValue;
    switch (k) {
        case 5: return launch_k<5>(p, rows, s);
        case 6: return launch_k<6>(p, rows, s);
        case 7: return launch_k<7>(p, rows, s);
        default: return hipErrorInvalidValue;
    }
}

// The tiles of several grids (the wide batched mode): slot i in tiles of slot_rows[i] rows.
template <int K>
__global__ __launch_bounds__(64 * PTPShape<K>::WAVES, 3) void wide_ptp_kernel(WideArgs a)
{
    __shared__ double lds[PTPShape<K>::LDS];
    int t;
    const int i = wide_slot(a, &t);
    if (i < 0) return;
    PTParamsC& pp = ((WideInstC*)a.desc)[a.slot_inst[i]].wpt[a.slot_pf[i] & 1];
    const int nstrips = (pp.nx - 1 + PTPShape<K>::OUT - 1) / PTPShape<K>::OUT;
    ptp_tile<K>(pp, a.slot_rows[i], t % nstrips, t / nstrips, lds);
}

int wide_pipe_tiles(int nx, int ny, int rows)
{
    return ((nx - 1 + PTPShape<WIDE_PIPE_K>::OUT - 1) / PTPShape<WIDE_PIPE_K>::OUT) * ((ny + rows - 1) / rows);
}

hipError_t launch_wide_pipe(const WideArgs& a, hipStream_t s)
{
    const int total = a.tile_start[a.n_active];
    if (total <= 0) return hipSuccess;
    for (int i = 0; i < a.n_active; ++i)
        if (a.slot_rows[i] < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(wide_ptp_kernel<WIDE_PIPE_K>, dim3(total), dim3(64 * PTPShape<WIDE_PIPE_K>::WAVES), 0, s, a);
    return hipGetLastError();
}

}  // namespace sf
