// sf_ptr_tile.h -- K PT iterations per pass on a tile that stays in registers, FP64.
//
// A workgroup holds a tile of 64 columns by WAVES * R rows: wave i the rows rb + i R .. + R - 1, lane
// l the column c0 + l, everything a node needs (state and materials) in registers.  The tile is read
// once, iterated K times in place and its inner 64 - 2K columns and WAVES * R - 2K rows are written.
// An iteration needs two exchanges between neighbouring waves through LDS: the V of a wave's first
// row goes up, then P and the stresses of a wave's last row go down, with a workgroup barrier each.
//
// An iteration costs the two barriers and R rows of arithmetic in a chain, so a pass is far
// shorter than one that marches down the rows (sf_ptk_tile.h, sf_ptp_tile.h): the shape for grids
// that the chip holds in about one round of workgroups, where latency bounds the pass.
//
// Lanes.  A row step produces P and dV at column c and V at column c + 1, so a lane keeps V at
// column c + 1; V at column c comes from the lane above.  The valid lanes shrink by one on either
// side per iteration, 1..62 after the first, K..63-K after the last; so do the rows.  What lies
// outside is computed from whatever is there and not stored.  Boundaries and expressions are
// pt_tile's (a product with a power of two may be folded: exact), so the stored iteration k+K is
// bit-identical to K pt_tile launches.
#pragma once

#include "sf_ptp_tile.h"

namespace sf {

#define PTR_VROW 66   // one V component of a row in LDS: lane l at l + 1
#define PTR_CROW 66   // one cell quantity of a row in LDS
// doubles of LDS for a workgroup of `waves` waves: one V row per wave and one past the last, one
// cell row per wave and one before the first
#define PTR_LDS(waves) (((waves) + 1) * (2 * PTR_VROW + 4 * PTR_CROW))

// The window of the row above while a wave marches down its rows.
struct PTRWin {
    double dtxx, dpn, pn, tyy, txyp;
};
struct PTRCell {
    double pn, txx, tyy, txy;
};

// P and the stresses of a row (compute_P_tau!, StokesSolver_multixpu.jl:140-169).
__device__ __forceinline__ PTRCell ptr_cell(const PTPConst& k, double vx, double vxp, double vy, double vyp, double vx1,
                                            double vx1p, double vy1p, double m2, double mub, double taup, double pold)
{
    const double dvxdx = (vx1p - vx1) * k.rdx;
    const double dvydy = (vy1p - vyp) * k.rdy;
    const double div = dvxdx + dvydy;
    const double d3 = (1.0 / 3.0) * div;
    PTRCell o;
    o.pn = pold - taup * div;
    o.txx = m2 * (dvxdx - d3);
    o.tyy = m2 * (dvydy - d3);
    o.txy = mub * ((vx1 - vx) * k.rdy + (vyp - vy) * k.rdx);
    return o;
}

// No exchange: one pass.
struct PTROnce {
    static constexpr bool RUN = false;
    int passes = 1;
    __device__ void put(int, int, double, double, double, double, double) const {}
    __device__ void get(int, int, double&, double&, double&, double&, double&) const {}
    __device__ bool swap() { return true; }
};

// ex: what happens between passes where the caller runs several on the same tile (ex.passes of them): the
// inner nodes stay in registers, those within K of another tile go out (put), the waves meet and
// wait for the other tiles (swap; false ends the run), and the outer nodes come in (get).
template <int R, class PP, class EX>
__device__ __forceinline__ bool ptr_tile(const PP& p, int K, int seg, int strip, int segid, double* lds, EX& ex)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nwaves = blockDim.x >> 6;
    const int nx = p.nx, ny = p.ny;
    const int OUT = SF_WAVE - 2 * K;
    const int c0 = strip * OUT - K;
    const int c = c0 + lane;
    const int r0 = segid * seg, r1 = min(r0 + seg, ny);
    const int rw = r0 - K + wave * R;  // the wave's first row
    PTPConst kc;
    kc.rdx = p.rdx;
    kc.rdy = p.rdy;
    kc.rdx8 = 0.125 * p.rdx;
    kc.rdy2 = 0.5 * p.rdy;
    kc.g = p.g;
    kc.dt = *p.dt;
    kc.dampx = p.dampx;
    kc.dampy = p.dampy;
    PTPEdge e;
    e.any = c0 < 0 || c0 + SF_WAVE + 1 >= nx;
    e.vx_zero = (c + 1 == 0) || (c + 1 == nx - 1);
    e.vy_left = c + 1 == 0;
    e.vy_right = c + 1 == nx;

    // the tile's rows: V and rho at column c + 1, the rest at column c, all clamped into the arrays
    const int cc = c < 0 ? 0 : c, c1 = c + 1 < 0 ? 0 : c + 1;
    const unsigned lvx = 8u * (unsigned)min(c1, nx - 1), lvy = 8u * (unsigned)min(c1, nx), lp = 8u * (unsigned)min(cc, nx - 2);
    const unsigned lmb = 8u * (unsigned)min(cc, nx - 1), ldx = 8u * (unsigned)min(cc, nx - 3);
    const unsigned svx = 8u * (unsigned)nx, svy = svx + 8u, sp = svx - 8u, sdx = svx - 16u;  // row strides
    double vxp[R], vyp[R], pn[R], dvx[R], dvy[R], m2[R], mub[R], taup[R], tauvx[R], tauvy[R], rho1[R], dxi[R], dyi[R];
    double mup[R + 1], rho[R + 2];
#pragma unroll
    for (int q = 0; q < R + 1; ++q) mup[q] = ptp_at(p.mu_p, (unsigned)crow(rw + q - 1, ny - 1) * sp + lp);
#pragma unroll
    for (int q = 0; q < R + 2; ++q) rho[q] = ptp_at(p.rho, (unsigned)crow(rw + q - 1, ny) * svy + lvy);
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int r = rw + q;
        vxp[q] = ptp_at(p.vx_a, (unsigned)crow(r, ny + 1) * svx + lvx);
        vyp[q] = ptp_at(p.vy_a, (unsigned)crow(r, ny) * svy + lvy);
        mub[q] = ptp_at(p.mu_b, (unsigned)crow(r, ny) * svx + lmb);
        pn[q] = ptp_at(p.p_a, (unsigned)crow(r, ny - 1) * sp + lp);
        dvx[q] = ptp_at((const double*)p.dvx, (unsigned)crow(r - 1, ny - 1) * sdx + ldx);
        dvy[q] = ptp_at((const double*)p.dvy, (unsigned)crow(r - 1, ny - 2) * sp + lp);
    }
    // LDS rows: V of wave i at vrow + i, cells of wave i at crow + i + 1
    double* const vrows = lds + 1;
    double* const crows = lds + (nwaves + 1) * (2 * PTR_VROW);
    double* const vmine = vrows + wave * (2 * PTR_VROW) + lane;
    const double* const vnext = vmine + 2 * PTR_VROW;
    double* const cmine = crows + (wave + 1) * (4 * PTR_CROW) + lane;
    const double* const cprev = cmine - 4 * PTR_CROW;
    vmine[0] = vxp[0];
    vmine[PTR_VROW] = vyp[0];
    const double vsc = p.vsc_mdxy2, ptsc41 = p.ptsc41, max_nxy = p.max_nxy;
    bool plain = ptp_plain(vsc) && ptp_plain(ptsc41) && ptp_plain(max_nxy);
#pragma unroll
    for (int q = 0; q < R + 1; ++q) plain = plain && ptp_plain_row(mup[q]);
    const double y41 = ptp_recip(4.1), ymax = ptp_recip(max_nxy);
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const double mu = mup[q + 1], mm = mup[q];
        const double dx2 = (mm + lane_down(mm, 1)) * 0.5, dy2 = (mm + mu) * 0.5;
        m2[q] = 2.0 * mu;
        mub[q] = (2.0 * mub[q]) * 0.5;
        if (plain) {
            taup[q] = ptp_div_by(ptsc41 * mu, max_nxy, ymax);
            tauvx[q] = ptp_div_by(ptp_div_by(vsc, dx2, ptp_recip(dx2)), 4.1, y41);
            tauvy[q] = ptp_div_by(ptp_div_by(vsc, dy2, ptp_recip(dy2)), 4.1, y41);
        } else {
            taup[q] = (ptsc41 * mu) / max_nxy;
            tauvx[q] = (vsc / dx2) / 4.1;
            tauvy[q] = (vsc / dy2) / 4.1;
        }
        rho1[q] = rho[q + 1];
        dxi[q] = lane_down(rho[q + 1], 1) - lane_up(rho[q + 1], 1);
        dyi[q] = rho[q + 2] - rho[q];
    }

    // the wave's boundary rows, if any: the special cases below are skipped in one test
    const bool edge = rw <= 0 || rw + R >= ny;
    const bool out_lane = lane >= K && lane < SF_WAVE - K;
    for (int pass = 0;; ++pass) {
        const bool final_pass = !EX::RUN || pass == ex.passes - 1;
        for (int it = 0; it < K; ++it) {
            const bool bc = edge && (it > 0 || pass > 0);  // (the first iteration reads the boundary rows from memory)
            ptp_barrier();
            // V of the row below the wave's last one: column c at lane - 1
            double nvx = vnext[-1], nvxp = vnext[0], nvyp = vnext[PTR_VROW];
            const int rl = rw + R - 1;
            if (bc && rl == ny - 1) {  // V row ny: Vx row ny = row ny-1, Vy zero
                nvxp = vxp[R - 1];
                nvx = lane_up(vxp[R - 1], 1);
                nvyp = 0.0;
            }
            // V of the row of the wave's last row step (row 0: Vx row 0 = row 1, Vy row 0 zero)
            double lvxp = vxp[R - 1], lvyp = vyp[R - 1];
            if (bc && rl == 0) {
                lvxp = nvxp;
                lvyp = 0.0;
            }
            const double lvxc = lane_up(lvxp, 1), lvyc = lane_up(lvyp, 1);
            const PTRCell last = ptr_cell(kc, lvxc, lvxp, lvyc, lvyp, nvx, nvxp, nvyp, m2[R - 1], mub[R - 1], taup[R - 1], pn[R - 1]);
            cmine[0] = last.pn;
            cmine[PTR_CROW] = last.txx;
            cmine[2 * PTR_CROW] = last.txy;
            cmine[3 * PTR_CROW] = last.tyy;
            ptp_barrier();
            PTRWin w;
            w.pn = cprev[0];
            w.dpn = (cprev[1] - w.pn) * kc.rdx;
            w.dtxx = (cprev[PTR_CROW + 1] - cprev[PTR_CROW]) * kc.rdx;
            w.txyp = cprev[2 * PTR_CROW + 1];
            w.tyy = cprev[3 * PTR_CROW];
            // V of the current row at columns c, c + 1
            double cvxp = vxp[0], cvyp = vyp[0], cvx, cvy;
            if (R == 1) {
                cvxp = lvxp;
                cvyp = lvyp;
                cvx = lvxc;
                cvy = lvyc;
            } else {
                if (bc && rw == 0) {
                    cvxp = vxp[R > 1 ? 1 : 0];
                    cvyp = 0.0;
                }
                cvx = lane_up(cvxp, 1);
                cvy = lane_up(cvyp, 1);
            }
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int r = rw + q;
                double bvx, bvxp, bvy = 0.0, bvyp = 0.0;  // V of the row below
                PTRCell s;
                if (q == R - 1) {
                    bvx = nvx;
                    bvxp = nvxp;
                    s = last;
                } else {
                    bvxp = vxp[q + 1 < R ? q + 1 : 0];
                    bvyp = vyp[q + 1 < R ? q + 1 : 0];
                    if (bc && r == ny - 1) {
                        bvxp = cvxp;
                        bvyp = 0.0;
                    }
                    if (bc && r + 1 == 0) {  // the row below is row 0
                        bvxp = q + 2 < R ? vxp[q + 2 < R ? q + 2 : 0] : nvxp;
                        bvyp = 0.0;
                    }
                    bvx = lane_up(bvxp, 1);
                    bvy = lane_up(bvyp, 1);
                    s = ptr_cell(kc, cvx, cvxp, cvy, cvyp, bvx, bvxp, bvyp, m2[q], mub[q], taup[q], pn[q]);
                }
                const double txyp = lane_down(s.txy, 1);
                const double rx = (w.dtxx + (txyp - w.txyp) * kc.rdy) - w.dpn;
                const double av4 = ((cvx + cvxp) + bvx) + bvxp;
                const double ry = (((s.tyy - w.tyy) * kc.rdy + (txyp - s.txy) * kc.rdx) - (s.pn - w.pn) * kc.rdy) +
                                  kc.g * (rho1[q] - kc.dt * ((av4 * dxi[q]) * kc.rdx8 + (cvyp * dyi[q]) * kc.rdy2));
                dvx[q] = kc.dampx * dvx[q] + rx;
                dvy[q] = kc.dampy * dvy[q] + ry;
                pn[q] = s.pn;
                vxp[q] = cvxp + tauvx[q] * dvx[q];
                vyp[q] = cvyp + tauvy[q] * dvy[q];
                if (it < K - 1 || !final_pass) ptp_bc(e, r == ny - 1, vxp[q], vyp[q]);
                if (q < R - 1) {
                    w.dtxx = (lane_down(s.txx, 1) - s.txx) * kc.rdx;
                    w.dpn = (lane_down(s.pn, 1) - s.pn) * kc.rdx;
                    w.pn = s.pn;
                    w.tyy = s.tyy;
                    w.txyp = txyp;
                    cvx = bvx;
                    cvxp = bvxp;
                    cvy = bvy;
                    cvyp = bvyp;
                }
            }
            vmine[0] = vxp[0];
            vmine[PTR_VROW] = vyp[0];
        }
        if (final_pass) break;
        if constexpr (EX::RUN) {
            const bool in_col = c >= 0 && c <= nx - 2, rim_lane = lane < 2 * K || lane >= SF_WAVE - 2 * K;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int r = rw + q;
                if (r >= r0 && r < r1 && out_lane && in_col && (rim_lane || r < r0 + K || r >= r1 - K))
                    ex.put(r, c, vxp[q], vyp[q], pn[q], dvx[q], dvy[q]);
            }
            if (!ex.swap()) return false;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int r = rw + q;
                if (r >= 0 && r < ny && in_col && !(r >= r0 && r < r1 && out_lane))
                    ex.get(r, c, vxp[q], vyp[q], pn[q], dvx[q], dvy[q]);
            ptp_bc(e, r == ny - 1, vxp[q], vyp[q]);  // the boundary columns of the outer rows
            }
            vmine[0] = vxp[0];
            vmine[PTR_VROW] = vyp[0];
        }
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int r = rw + q;
        if (r < r0 || r >= r1) continue;
        if (!e.any && r >= 2 && r <= ny - 2) {  // no boundary row or column
            if (out_lane) {
                const unsigned j = (unsigned)r, cb = 8u * (unsigned)c;
                ptp_at(p.p_b, j * sp + cb) = pn[q];
                ptp_at(p.dvx_o, (j - 1) * sdx + cb) = dvx[q];
                ptp_at(p.vx_b, j * svx + cb + 8u) = vxp[q];
                ptp_at(p.dvy_o, (j - 1) * sp + cb) = dvy[q];
                ptp_at(p.vy_b, j * svy + cb + 8u) = vyp[q];
            }
        } else {
            const PTRow o{pn[q], dvx[q], dvy[q], vxp[q], vyp[q]};
            pt2_store(p, o, c, r, r0, out_lane);
        }
    }
    return true;
}

}  // namespace sf
