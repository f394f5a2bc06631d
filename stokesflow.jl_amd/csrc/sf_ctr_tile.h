// sf_ctr_tile.h -- K FP32 correction sweeps per pass on a tile that stays in registers.
//
// The FP32 counterpart of sf_ptr_tile.h, with its layout, exchanges and boundary rules: a workgroup holds
// 64 columns by WAVES * R rows, wave i the rows rb + i R .. + R - 1, reads the tile once, sweeps it K times
// and writes its inner 64 - 2K columns and WAVES * R - 2K rows.  A node takes 15 registers (state, momentum,
// materials, forcing), so a wave holds up to six rows where FP64 holds three.  The expressions are sf_corr.h's:
// the same bits as K sweeps of any other grouping.
#pragma once

#include "sf_corr.h"

namespace sf {

#define CTR_ROW 66  // one quantity of a row in LDS: lane l at l + 1
#define CTR_LDS(waves) (((waves) + 1) * 6 * CTR_ROW)

__device__ __forceinline__ int ctr_row(int r, int nrows) { return min(max(r, 0), nrows - 1); }
// Element at a byte offset from a row's start: the row is uniform, so its address is scalar.
__device__ __forceinline__ const float& ctr_at(const float* a, int64_t row, unsigned off) { return *(const float*)((const char*)(a + row) + off); }
__device__ __forceinline__ float& ctr_at(float* a, int64_t row, unsigned off) { return *(float*)((char*)(a + row) + off); }

// Workgroup barrier that orders LDS accesses only.
__device__ __forceinline__ void ctr_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int R, class PP>
__device__ __forceinline__ void ctr_tile(const PP& p, int K, int seg, int strip, int segid, float* lds)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nwaves = blockDim.x >> 6;
    const int nx = p.nx, ny = p.ny;
    const int c0 = strip * (SF_WAVE - 2 * K) - K;
    const int c = c0 + lane;
    const int r0 = segid * seg, r1 = min(r0 + seg, ny);
    const int rw = r0 - K + wave * R;  // the wave's first row
    const CorrC kc = corr_consts(p, p.dt);
    const bool edge_col = c0 < 0 || c0 + SF_WAVE + 1 >= nx;
    const bool vx_zero = (c + 1 == 0) || (c + 1 == nx - 1), vy_left = c + 1 == 0, vy_right = c + 1 == nx;

    // the tile's rows: V and rho at column c + 1, the rest at column c, all clamped into the arrays
    const int cc = c < 0 ? 0 : c, c1 = c + 1 < 0 ? 0 : c + 1;
    const unsigned lvx = 4u * (unsigned)min(c1, nx - 1), lvy = 4u * (unsigned)min(c1, nx), lp = 4u * (unsigned)min(cc, nx - 2);
    const unsigned lmb = 4u * (unsigned)min(cc, nx - 1), ldx = 4u * (unsigned)min(cc, nx - 3);
    const int64_t svx = nx, svy = nx + 1, sp = nx - 1, sdx = nx - 2;  // row strides
    float vxp[R], vyp[R], pn[R], mx[R], my[R], m2[R], mub[R], taup[R], tauvx[R], tauvy[R], dxi[R], dyi[R], fx[R], fy[R], fc[R];
    float mup[R + 1], rho[R + 2];
#pragma unroll
    for (int q = 0; q < R + 1; ++q) mup[q] = ctr_at(p.mu_p, ctr_row(rw + q - 1, ny - 1) * sp, lp);
#pragma unroll
    for (int q = 0; q < R + 2; ++q) rho[q] = ctr_at(p.rho, ctr_row(rw + q - 1, ny) * svy, lvy);
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int r = rw + q;
        const int64_t op = ctr_row(r, ny - 1) * sp, ox = ctr_row(r - 1, ny - 1) * sdx, oy = ctr_row(r - 1, ny - 2) * sp;
        vxp[q] = ctr_at(p.vx_a, ctr_row(r, ny + 1) * svx, lvx);
        vyp[q] = ctr_at(p.vy_a, ctr_row(r, ny) * svy, lvy);
        mub[q] = ctr_at(p.mu_b, ctr_row(r, ny) * svx, lmb);
        pn[q] = ctr_at(p.p_a, op, lp);
        fc[q] = ctr_at(p.fc, op, lp);
        mx[q] = ctr_at((const float*)p.mx, ox, ldx);
        fx[q] = ctr_at(p.fx, ox, ldx);
        my[q] = ctr_at((const float*)p.my, oy, lp);
        fy[q] = ctr_at(p.fy, oy, lp);
    }
    // LDS rows: V of wave i at vrow + i, cells of wave i at crow + i + 1
    float* const vmine = lds + 1 + wave * (2 * CTR_ROW) + lane;
    const float* const vnext = vmine + 2 * CTR_ROW;
    float* const cmine = lds + (nwaves + 1) * (2 * CTR_ROW) + (wave + 1) * (4 * CTR_ROW) + lane;
    const float* const cprev = cmine - 4 * CTR_ROW;
    vmine[0] = vxp[0];
    vmine[CTR_ROW] = vyp[0];
#pragma unroll
    for (int q = 0; q < R; ++q) {
        m2[q] = 2.0f * mup[q + 1];
        taup[q] = corr_taup(p, mup[q + 1]);
        tauvx[q] = corr_tauv(p, mup[q], lane_down(mup[q], 1));
        tauvy[q] = corr_tauv(p, mup[q], mup[q + 1]);
        dxi[q] = lane_down(rho[q + 1], 1) - lane_up(rho[q + 1], 1);
        dyi[q] = rho[q + 2] - rho[q];
    }

    const bool edge = rw <= 0 || rw + R >= ny;  // the wave has boundary rows
    for (int it = 0; it < K; ++it) {
        const bool bc = edge && it > 0;  // (the first sweep reads the boundary rows from memory)
        ctr_barrier();
        // V of the row below the wave's last one: column c at lane - 1
        float nvx = vnext[-1], nvxp = vnext[0], nvyp = vnext[CTR_ROW];
        const int rl = rw + R - 1;
        if (bc && rl == ny - 1) {  // V row ny: Vx row ny = row ny-1, Vy zero
            nvxp = vxp[R - 1];
            nvx = lane_up(vxp[R - 1], 1);
            nvyp = 0.f;
        }
        // V of the row of the wave's last row step (row 0: Vx row 0 = row 1, Vy row 0 zero)
        float lvxp = vxp[R - 1], lvyp = vyp[R - 1];
        if (bc && rl == 0) {
            lvxp = nvxp;
            lvyp = 0.f;
        }
        const float lvxc = lane_up(lvxp, 1), lvyc = lane_up(lvyp, 1);
        const CorrPT last = corr_ptau(kc, nvx, nvxp, lvxc, nvyp, lvyc, lvyp, m2[R - 1], mub[R - 1], fc[R - 1], pn[R - 1],
                                      taup[R - 1]);
        cmine[0] = last.pn;
        cmine[CTR_ROW] = last.txx;
        cmine[2 * CTR_ROW] = last.txy;
        cmine[3 * CTR_ROW] = last.tyy;
        ctr_barrier();
        // the row above the wave's first one
        float w_pn = cprev[0], w_tyy = cprev[3 * CTR_ROW], w_txyp = cprev[2 * CTR_ROW + 1];
        float w_txx = cprev[CTR_ROW], w_txxp = cprev[CTR_ROW + 1], w_pnp = cprev[1];
        // V of the current row at columns c, c + 1
        float cvxp = vxp[0], cvyp = vyp[0], cvx, cvy;
        if (R == 1) {
            cvxp = lvxp;
            cvyp = lvyp;
            cvx = lvxc;
            cvy = lvyc;
        } else {
            if (bc && rw == 0) {
                cvxp = vxp[R > 1 ? 1 : 0];
                cvyp = 0.f;
            }
            cvx = lane_up(cvxp, 1);
            cvy = lane_up(cvyp, 1);
        }
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int r = rw + q;
            float bvx, bvxp, bvy = 0.f, bvyp = 0.f;  // V of the row below
            CorrPT s;
            if (q == R - 1) {
                bvx = nvx;
                bvxp = nvxp;
                s = last;
            } else {
                bvxp = vxp[q + 1 < R ? q + 1 : 0];
                bvyp = vyp[q + 1 < R ? q + 1 : 0];
                if (bc && r == ny - 1) {
                    bvxp = cvxp;
                    bvyp = 0.f;
                }
                if (bc && r + 1 == 0) {  // the row below is row 0
                    bvxp = q + 2 < R ? vxp[q + 2 < R ? q + 2 : 0] : nvxp;
                    bvyp = 0.f;
                }
                bvx = lane_up(bvxp, 1);
                bvy = lane_up(bvyp, 1);
                s = corr_ptau(kc, bvx, bvxp, cvx, bvyp, cvy, cvyp, m2[q], mub[q], fc[q], pn[q], taup[q]);
            }
            const float txyp = lane_down(s.txy, 1);
            const float rx = corr_rx(kc, w_txxp, w_txx, w_pnp, w_pn, txyp, w_txyp, fx[q]);
            const float av4 = ((cvx + cvxp) + bvx) + bvxp;
            const float ry = corr_ry(kc, s.tyy, w_tyy, s.pn, w_pn, txyp, s.txy, av4, dxi[q], cvyp, dyi[q], fy[q]);
            mx[q] = __builtin_fmaf(kc.dampx, mx[q], rx);
            my[q] = __builtin_fmaf(kc.dampy, my[q], ry);
            pn[q] = s.pn;
            vxp[q] = __builtin_fmaf(tauvx[q], mx[q], cvxp);
            vyp[q] = __builtin_fmaf(tauvy[q], my[q], cvyp);
            if (it < K - 1) {  // V as the last sweep stores it: free-slip columns, Vy zero on row ny - 1
                if (edge_col) {
                    asm volatile("");  // a branch, not selects on every strip
                    const float dn = lane_down(vyp[q], 1), up = lane_up(vyp[q], 1);
                    vxp[q] = vx_zero ? 0.f : vxp[q];
                    vyp[q] = vy_left ? dn : (vy_right ? up : vyp[q]);
                }
                if (r == ny - 1) vyp[q] = 0.f;
            }
            if (q < R - 1) {
                w_txx = s.txx;
                w_txxp = lane_down(s.txx, 1);
                w_pnp = lane_down(s.pn, 1);
                w_pn = s.pn;
                w_tyy = s.tyy;
                w_txyp = txyp;
                cvx = bvx;
                cvxp = bvxp;
                cvy = bvy;
                cvyp = bvyp;
            }
        }
        vmine[0] = vxp[0];
        vmine[CTR_ROW] = vyp[0];
    }
    const bool out_lane = lane >= K && lane < SF_WAVE - K;
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int r = rw + q;
        if (r < r0 || r >= r1) continue;
        if (!edge_col && r >= 2 && r <= ny - 2) {  // no boundary row or column
            if (out_lane) {
                const unsigned cb = 4u * (unsigned)c;
                ctr_at(p.p_b, r * sp, cb) = pn[q];
                ctr_at(p.mx_o, (r - 1) * sdx, cb) = mx[q];
                ctr_at(p.vx_b, r * svx + 1, cb) = vxp[q];
                ctr_at(p.my_o, (r - 1) * sp, cb) = my[q];
                ctr_at(p.vy_b, r * svy + 1, cb) = vyp[q];
            }
        } else {
            const CorrRow o{pn[q], mx[q], my[q], vxp[q], vyp[q]};
            corr2_store(p, o, c, r, r0, out_lane);
        }
    }
}

}  // namespace sf
