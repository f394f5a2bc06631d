// sf_corr.h -- the FP32 correction sweep's arithmetic and stores, shared by its kernels
// (sf_refine.hip, sf_ctr_tile.h).
#pragma once

#include "sf_device.h"
#include "sf_internal.h"

namespace sf {

// The FP32 sweeps' pseudo-time steps (dtauP, dtauVx, dtauVy of compute_timesteps!,
// StokesSolver_multixpu.jl:128-133) take the hardware reciprocal (v_rcp_f32, 1 ulp) in place of
// IEEE division.  The steps only scale the correction sweeps and convergence is decided on FP64
// residuals, so their last bits do not matter; the five divisions per node were a tenth of the
// sweep's VALU work (2048^2: 21.9 -> 19.8 us per sweep).  Every FP32 kernel uses the same
// expressions, so all sweep groupings stay bit-identical to each other.
__device__ __forceinline__ float tau_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// The FP32 sweep's arithmetic, shared by every FP32 kernel so that all sweep groupings give the
// same bits.  It is the PT iteration's (StokesSolver_multixpu.jl:140-234) on the correction, in an
// order of its own: products with a common factor are grouped, constants folded and a*b+c fused,
// which the FP64 kernels may not do (they reproduce the reference bit for bit) but the correction
// sweeps may: they only have to drive the FP64 residual down, and convergence is decided in FP64.
struct CorrC {
    float rdx, rdy;
    float kx, ky;  // g dt / 8 / dx and g dt / 2 / dy: the free-surface term's factors
    float dampx, dampy;
};

template <class PP>
__device__ __forceinline__ CorrC corr_consts(const PP& p, float dt)
{
    const float gdt = p.g * dt;
    return CorrC{p.rdx, p.rdy, (gdt * 0.125f) * p.rdx, (gdt * 0.5f) * p.rdy, p.dampx, p.dampy};
}

// The P update and the stresses at one node (compute_P_tau!, :140-169): m2 = 2 mu_p, taup = dtauP.
struct CorrPT {
    float dvxdx, dvydy, cres, pn, txx, tyy, txy;
};

__device__ __forceinline__ CorrPT corr_ptau(const CorrC& k, float vx1, float vx1_p1, float vx_r, float vy1_p1,
                                            float vy_r, float vy_r_p1, float m2, float mub, float fc, float pold,
                                            float taup)
{
    CorrPT o;
    o.dvxdx = (vx1_p1 - vx1) * k.rdx;
    o.dvydy = (vy1_p1 - vy_r_p1) * k.rdy;
    const float div = o.dvxdx + o.dvydy;
    o.cres = div + fc;  // continuity residual of the full state
    o.pn = __builtin_fmaf(-taup, o.cres, pold);
    const float d3 = div * (1.0f / 3.0f);
    o.txx = m2 * (o.dvxdx - d3);
    o.tyy = m2 * (o.dvydy - d3);
    o.txy = mub * __builtin_fmaf(vx1 - vx_r, k.rdy, (vy_r_p1 - vy_r) * k.rdx);
    return o;
}

// x momentum residual (compute_ResX, :176-182) plus the forcing.
__device__ __forceinline__ float corr_rx(const CorrC& k, float txx_p1, float txx, float pn_p1, float pn, float txy_p1,
                                         float txy_prev_p1, float fx)
{
    return __builtin_fmaf((txx_p1 - txx) - (pn_p1 - pn), k.rdx, __builtin_fmaf(txy_p1 - txy_prev_p1, k.rdy, fx));
}

// y momentum residual with the free-surface term (compute_ResY, :189-202) plus the forcing;
// av4 is four times the Vx average, d_xi and d_yi the two rho differences.
__device__ __forceinline__ float corr_ry(const CorrC& k, float tyy, float tyy_prev, float pn, float pn_prev,
                                         float txy_p1, float txy, float av4, float d_xi, float vy, float d_yi,
                                         float fy)
{
    const float stab = __builtin_fmaf(av4 * d_xi, k.kx, (vy * d_yi) * k.ky);
    return __builtin_fmaf((tyy - tyy_prev) - (pn - pn_prev), k.rdy, __builtin_fmaf(txy_p1 - txy, k.rdx, fy)) - stab;
}

// The pseudo-time steps (compute_timesteps!, :128-133) from mu_p.
template <class PP>
__device__ __forceinline__ float corr_taup(const PP& p, float mup)
{
    return (p.ptsc41 * mup) * tau_rcp(p.max_nxy);
}
template <class PP>
__device__ __forceinline__ float corr_tauv(const PP& p, float mup_a, float mup_b)
{
    return p.vsc_mdxy2 * tau_rcp((mup_a + mup_b) * 2.05f);
}

struct CorrRow {
    float pn, mx, my, vx, vy;
};

// Stores of a pass's last sweep for row step r, with corr_tile's conditions and (homogeneous) BC writes.
template <class PP>
__device__ __forceinline__ void corr2_store(const PP& p, const CorrRow& o, int c, int r, int r0, bool out_lane)
{
    const int nx = p.nx, ny = p.ny;
    const int64_t lvx = nx, lvy = nx + 1, lp = nx - 1;
    if (!out_lane || r < r0) return;
    if (c < nx - 1 && r <= ny - 2) p.p_b[ix2(c, r, lp)] = o.pn;
    const int j = r - 1;
    if (j < 0) return;
    if (c < nx - 2) {
        p.mx_o[ix2(c, j, nx - 2)] = o.mx;
        p.vx_b[ix2(c + 1, j + 1, lvx)] = o.vx;
        if (j == 0) p.vx_b[ix2(c + 1, 0, lvx)] = o.vx;
        if (j == ny - 2) p.vx_b[ix2(c + 1, ny, lvx)] = o.vx;
    }
    if (c == 0 || c == nx - 2) {
        const int col = (c == 0) ? 0 : nx - 1;
        p.vx_b[ix2(col, j + 1, lvx)] = 0.f;
        if (j == 0) p.vx_b[ix2(col, 0, lvx)] = 0.f;
        if (j == ny - 2) p.vx_b[ix2(col, ny, lvx)] = 0.f;
    }
    if (c < nx - 1 && j <= ny - 3) {
        p.my_o[ix2(c, j, nx - 1)] = o.my;
        p.vy_b[ix2(c + 1, j + 1, lvy)] = o.vy;
        if (c == 0) p.vy_b[ix2(0, j + 1, lvy)] = o.vy;
        if (c == nx - 2) p.vy_b[ix2(nx, j + 1, lvy)] = o.vy;
    }
    if (c < nx - 1 && (j == 0 || j == ny - 2)) {
        const int row = (j == 0) ? 0 : ny - 1;
        p.vy_b[ix2(c + 1, row, lvy)] = 0.f;
        if (c == 0) p.vy_b[ix2(0, row, lvy)] = 0.f;
        if (c == nx - 2) p.vy_b[ix2(nx, row, lvy)] = 0.f;
    }
}

}  // namespace sf
