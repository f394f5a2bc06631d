// sf_ptp_tile.h -- K PT iterations per pass, pipelined over the waves of a workgroup, FP64.
//
// ptk_tile (sf_ptk_tile.h) keeps all K iterations of a tile in one wave's registers, so K is
// bounded by the register file (four iterations at 251 VGPRs, two waves per SIMD) and the wave
// issues the lane shifts, register copies and range tests of all of them.  Here the K stages are
// spread over the 1 + K/2 waves of a workgroup: wave 0 runs stage 0 (iteration k+1, the loads and
// the five FP64 divisions of the pseudo-time steps), wave w >= 1 the stages 2w-1 and 2w (the last
// wave of an even K only 2w-1), and the last wave stores.  All waves march down the same strip of
// 64 columns, one row per step, with one workgroup barrier per step; each wave holds the row
// windows of one or two stages only (three waves per SIMD), so K can be seven.
//
// Rows.  Stage s of a wave runs one row behind the wave's first stage (as in ptk_tile), and a
// wave's first stage two rows behind the previous wave's last one: the row that wave w - 1 writes
// to LDS in step t is read by wave w in step t + 1.  So at step t wave 0 runs row rstart + t, wave
// w's stages rows rstart + t - (3w - 1) and rstart + t - 3w.
//
// LDS.  The materials of a row do not change from stage to stage: wave 0 puts the seven values
// per node that the stages need (2 mu_p, mu_b, the three pseudo-time steps, rho one column over,
// the x difference of rho) into a ring of rows that every later stage reads.  Between two waves a
// double-buffered row of V, P and dV is handed over; V is written one lane up (a stage's lane l
// produces V at column c + 1, which is the next stage's lane l + 1) and read at lanes l and l + 1,
// so a handed-over row needs no lane shifts.
//
// Lanes, strips, boundaries and the halo shrinking by one lane and row per stage are ptk_tile's,
// and every stage evaluates pt_row's expressions on the same operands (a product with a power of
// two may be folded: exact), so the stored iteration k+K is bit-identical to K pt_tile launches.
//
// What bounds it: FP64 issue.  A row and stage takes 54 additions and multiplications, 6 to 10 DPP
// moves and little else (77 VALU instructions against 126 in ptk_tile<4>, with 1.28 strip overlap
// against 1.14 x 1.13), and seven iterations share one pass over memory (1.87 GB at 4096^2).  Measured
// at 4096^2, us per iteration: 64.0, 448 per pass (ptk_tile<4> 108.6-112); in the solver's loop 66 (109);
// 2048^2 18.7 (28), 1024^2 6.4 (9.1).  With the barriers, the loads or the stores taken out a pass of
// 500 us (before the short divisions and the wave priorities) took 457, 430 and 470, with all of them
// out 383: the rest is arithmetic.  Two rows in flight in wave 0 did as well as three or four
// (which spill); one stage per wave (more waves, shorter steps) was no faster, wave 0 being the
// longest; three workgroups per CU fit (48 KB of LDS, 157 VGPRs) and want to be resident together:
// a fourth round costs a whole one (pt_plan).
#pragma once

#include <type_traits>

#include "sf_pt2_tile.h"

namespace sf {

#define PTP_MATS 7
#define PTP_VROW 66                            // V rows: lanes 0..64 used
#define PTP_HAND (2 * PTP_VROW + 3 * SF_WAVE)  // doubles of one handed-over row

template <int K>
struct PTPShape {
    static constexpr int WAVES = 1 + K / 2;
    static constexpr int OUT = SF_WAVE - 2 * K;  // output columns per strip
    // first stage of wave w >= 1 and the rows it runs behind stage 0
    __device__ static constexpr int stage(int w) { return 2 * w - 1; }
    __device__ static constexpr int lag(int w) { return 3 * w - 1; }
    static constexpr bool LAST_TWO = K % 2 == 1;  // the last wave has two stages
    static constexpr int LAG = lag(WAVES - 1) + (LAST_TWO ? 1 : 0);  // the last stage's
    static constexpr int RING = lag(WAVES - 1) + 1;  // material rows kept: up to the last wave's first stage
    static constexpr int LDS = RING * PTP_MATS * SF_WAVE + 2 * (WAVES - 1) * PTP_HAND;  // doubles
};

// Constants of a pass: rdx, rdy, and the free-surface term's factors 0.25 * 0.5 * rdx and
// 0.5 * rdy.
struct PTPConst {
    double rdx, rdy, rdx8, rdy2, g, dt, dampx, dampy;
};

// The row window of one stage: V of the current row (and one lane down), and of the row above the
// x differences of txx and P, and P, tyy and txy.
struct PTPWin {
    double vx, vxp, vy, vyp;
    double dtxx, dpn, pn, tyy, txyp;
};

// The materials of a row at the lane's column (rho1: rho one column over; dxi: the x difference of
// rho; dyi its y difference, formed from rho1 of the rows around).
struct PTPMat {
    double m2, mub, taup, tauvx, tauvy, rho1, dxi, dyi;
};

// One row of one stage with pt_row's expressions; the window slides down one row.
__device__ __forceinline__ PTRow ptp_row(const PTPConst& k, PTPWin& w, double vx1, double vx1p, double vy1, double vy1p,
                                         const PTPMat& m, double pold, double dvx, double dvy)
{
    const double dvxdx = (vx1p - vx1) * k.rdx;
    const double dvydy = (vy1p - w.vyp) * k.rdy;
    const double div = dvxdx + dvydy;
    const double d3 = (1.0 / 3.0) * div;
    const double pn = pold - m.taup * div;
    const double txx = m.m2 * (dvxdx - d3);
    const double tyy = m.m2 * (dvydy - d3);
    const double txy = m.mub * ((vx1 - w.vx) * k.rdy + (w.vyp - w.vy) * k.rdx);
    const double txyp = lane_down(txy, 1);
    const double rx = (w.dtxx + (txyp - w.txyp) * k.rdy) - w.dpn;
    const double av4 = ((w.vx + w.vxp) + vx1) + vx1p;
    const double ry = (((tyy - w.tyy) * k.rdy + (txyp - txy) * k.rdx) - (pn - w.pn) * k.rdy) +
                      k.g * (m.rho1 - k.dt * ((av4 * m.dxi) * k.rdx8 + (w.vyp * m.dyi) * k.rdy2));
    PTRow o;
    o.pn = pn;
    o.dvx = k.dampx * dvx + rx;
    o.dvy = k.dampy * dvy + ry;
    o.vx = w.vxp + m.tauvx * o.dvx;
    o.vy = w.vyp + m.tauvy * o.dvy;
    w.dtxx = (lane_down(txx, 1) - txx) * k.rdx;
    w.dpn = (lane_down(pn, 1) - pn) * k.rdx;
    w.pn = pn;
    w.tyy = tyy;
    w.txyp = txyp;
    w.vx = vx1;
    w.vxp = vx1p;
    w.vy = vy1;
    w.vyp = vy1p;
    return o;
}

// Column boundaries of a strip: V at column c + 1 of the lane.
struct PTPEdge {
    bool any;  // the strip holds a boundary column (uniform)
    bool vx_zero, vy_left, vy_right;
};

// V as pt_tile would have stored it: free-slip columns, and Vy zero on row ny - 1.
__device__ __forceinline__ void ptp_bc(const PTPEdge& e, bool last_row, double& vx, double& vy)
{
    if (e.any) {
        asm volatile("");  // a branch: as selects the boundary would cost every strip 16 instructions
        const double dn = lane_down(vy, 1), up = lane_up(vy, 1);
        vx = e.vx_zero ? 0.0 : vx;
        vy = e.vy_left ? dn : (e.vy_right ? up : vy);
    }
    if (last_row) vy = 0.0;
}

// Whether the divisions of the pseudo-time steps stay in that range: mu_p of the row and the
// constants within 2^+-200 on every lane (a uniform test; else the divisions are full ones).  Wave 0
// issues 131 instead of 162 VALU instructions per row: 79.2 -> 71.2 us per iteration at 4096^2 together
// with the wave priorities below.
__device__ __forceinline__ bool ptp_plain(double v) { return v > 0x1p-200 && v < 0x1p200; }
__device__ __forceinline__ bool ptp_plain_row(double mup) { return __ballot(ptp_plain(mup)) == ~0ull; }

// Element at a byte offset from a uniform row pointer (32-bit: rows are shorter than 4 GiB).
__device__ __forceinline__ const double& ptp_at(const double* row, unsigned off) { return *(const double*)((const char*)row + off); }
__device__ __forceinline__ double& ptp_at(double* row, unsigned off) { return *(double*)((char*)row + off); }

// Workgroup barrier that orders LDS accesses only: global loads and stores stay in flight.
__device__ __forceinline__ void ptp_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Rows that stage s of a tile computes.
struct PTPRange {
    int lo, hi;
};
template <int K>
__device__ __forceinline__ PTPRange ptp_range(int s, int r0, int r1, int ny)
{
    return PTPRange{max(r0 - (K - s), 0), min(r1 - 1 + (K - 1 - s), ny - 1)};
}

__device__ __forceinline__ void ptp_put(double* hand, int lane, const PTRow& o)
{
    hand[lane + 1] = o.vx;
    hand[PTP_VROW + lane + 1] = o.vy;
    hand[2 * PTP_VROW + lane] = o.pn;
    hand[2 * PTP_VROW + SF_WAVE + lane] = o.dvx;
    hand[2 * PTP_VROW + 2 * SF_WAVE + lane] = o.dvy;
}

// Wave 0: stage 0, from memory; rows PF ahead are in flight.
template <int K, class PP>
__device__ __forceinline__ void ptp_first(const PP& p, const PTPConst& kc, const PTPEdge& e, double* mats, double* hand,
                                          int c, int r0, int r1, int rstart, int steps)
{
    constexpr int PF = 2;
    const int lane = threadIdx.x & 63;
    const int nx = p.nx, ny = p.ny;
    const int cc = c < 0 ? 0 : c;
    LaneCols lc;
    lc.vx = (unsigned)min(cc, nx - 1);
    lc.vy = (unsigned)min(cc, nx);
    lc.p = (unsigned)min(cc, nx - 2);
    lc.dvx = (unsigned)min(cc, nx - 3);
    lc.dvy = (unsigned)min(cc, nx - 2);
    const LaneCols lb{8 * lc.vx, 8 * lc.vy, 8 * lc.p, 8 * lc.dvx, 8 * lc.dvy};  // byte offsets
    const PTPRange rg = ptp_range<K>(0, r0, r1, ny);
    const double vsc = p.vsc_mdxy2, ptsc41 = p.ptsc41, max_nxy = p.max_nxy;
    const double y41 = ptp_recip(4.1), ymax = ptp_recip(max_nxy);
    const bool const_plain = ptp_plain(vsc) && ptp_plain(ptsc41) && ptp_plain(max_nxy);
    bool plain_m = false;  // the row above passed ptp_plain_row
    PTPWin w{};
    w.vx = (p.vx_a + (int64_t)rstart * nx)[lc.vx];
    w.vy = (p.vy_a + (int64_t)rstart * (nx + 1))[lc.vy];
    double rho_r = (p.rho + (int64_t)rstart * (nx + 1))[lc.vy];
    RowIn in[PF];
#pragma unroll
    for (int u = 0; u < PF; ++u) in[u] = load_row(p, lc, rstart + u, true);
    w.vxp = lane_down(w.vx, 1);
    w.vyp = lane_down(w.vy, 1);
    double rho1 = lane_down(rho_r, 1), rho1_m = 0.0, mup_m = 0.0;
    int slot = 0, t = 0;
    PTRow o{};
    // Row pointers of the row PF ahead, for the steps where no row index needs a clamp.
    struct Rows {
        const double *vx, *vy, *rho, *p, *mup, *mub, *dvx, *dvy;
    } q;
    auto step = [&](RowIn& next, auto plain_tag) {
        const int r = rstart + t;
        const RowIn a = next;
        if constexpr (decltype(plain_tag)::value) {
            next = RowIn{ptp_at(q.vx, lb.vx), ptp_at(q.vy, lb.vy), ptp_at(q.rho, lb.vy), ptp_at(q.p, lb.p),
                         ptp_at(q.mup, lb.p), ptp_at(q.mub, lb.vx), ptp_at(q.dvx, lb.dvx), ptp_at(q.dvy, lb.dvy)};
            q.vx += nx;
            q.vy += nx + 1;
            q.rho += nx + 1;
            q.p += nx - 1;
            q.mup += nx - 1;
            q.mub += nx;
            q.dvx += nx - 2;
            q.dvy += nx - 1;
        } else if (r + PF <= rg.hi) {
            next = load_row(p, lc, r + PF, true);
        }
        const double rho_n1 = lane_down(a.rho1, 1);
        PTPMat m;
        m.m2 = 2.0 * a.mup;
        m.mub = (2.0 * a.mub) * 0.5;
        const double dx2 = (mup_m + lane_down(mup_m, 1)) * 0.5, dy2 = (mup_m + a.mup) * 0.5;
        const bool plain = const_plain && ptp_plain_row(a.mup);
        if (plain && plain_m) {
            m.taup = ptp_div_by(ptsc41 * a.mup, max_nxy, ymax);
            m.tauvx = ptp_div_by(ptp_div_by(vsc, dx2, ptp_recip(dx2)), 4.1, y41);
            m.tauvy = ptp_div_by(ptp_div_by(vsc, dy2, ptp_recip(dy2)), 4.1, y41);
        } else {
            m.taup = (ptsc41 * a.mup) / max_nxy;
            m.tauvx = (vsc / dx2) / 4.1;
            m.tauvy = (vsc / dy2) / 4.1;
        }
        plain_m = plain;
        m.rho1 = rho1;
        m.dxi = lane_down(rho1, 1) - rho_r;
        m.dyi = rho_n1 - rho1_m;
        double* const ms = mats + slot * (PTP_MATS * SF_WAVE) + lane;
        ms[0] = m.m2;
        ms[SF_WAVE] = m.mub;
        ms[2 * SF_WAVE] = m.taup;
        ms[3 * SF_WAVE] = m.tauvx;
        ms[4 * SF_WAVE] = m.tauvy;
        ms[5 * SF_WAVE] = m.rho1;
        ms[6 * SF_WAVE] = m.dxi;
        o = ptp_row(kc, w, a.vx1, lane_down(a.vx1, 1), a.vy1, lane_down(a.vy1, 1), m, a.pold, a.dvx, a.dvy);
        ptp_bc(e, r == ny - 1, o.vx, o.vy);
        ptp_put(hand + (t & 1) * PTP_HAND, lane, o);
        mup_m = a.mup;
        rho1_m = rho1;
        rho1 = rho_n1;
        rho_r = a.rho1;
        slot = slot + 1 == PTPShape<K>::RING ? 0 : slot + 1;
        ++t;
        ptp_barrier();
    };
    const int n0 = rg.hi - rstart + 1;                            // rows of stage 0; steps > n0
    const int n1 = min(rg.hi, ny - 2) - PF - rstart + 1;          // of them, rows whose load is a plain one
    {
        const int64_t r = min(rstart + PF, ny - 2);
        q = Rows{p.vx_a + (r + 1) * nx, p.vy_a + (r + 1) * (nx + 1), p.rho + (r + 1) * (nx + 1), p.p_a + r * (nx - 1),
                 p.mu_p + r * (nx - 1), p.mu_b + r * nx, p.dvx + (r - 1) * (nx - 2), p.dvy + (r - 1) * (nx - 1)};
    }
    while (t + PF <= n1) {
#pragma unroll
        for (int u = 0; u < PF; ++u) step(in[u], std::true_type{});
    }
    while (t < n0) {
#pragma unroll
        for (int u = 0; u < PF; ++u)
            if (t < n0) step(in[u], std::false_type{});
    }
    for (; t < steps; ++t) {
        if (rstart + t == ny) {  // virtual row ny: Vx row ny = row ny-1, Vy zero
            double* const h = hand + (t & 1) * PTP_HAND;
            h[lane + 1] = o.vx;
            h[PTP_VROW + lane + 1] = 0.0;
            mats[slot * (PTP_MATS * SF_WAVE) + 5 * SF_WAVE + lane] = rho1_m;
        }
        slot = slot + 1 == PTPShape<K>::RING ? 0 : slot + 1;
        ptp_barrier();
    }
}

// Wave w >= 1: stage A = PTPShape::stage(w) and, with TWO, the next one, B; with LAST the later one
// is stored.
template <int K, bool TWO, bool LAST, class PP>
__device__ __forceinline__ void ptp_later(const PP& p, const PTPConst& kc, const PTPEdge& e, const double* mats,
                                          const double* hand_in, double* hand_out, int wave, int c, int r0, int r1,
                                          int rstart, int steps)
{
    typedef PTPShape<K> S;
    constexpr int RING = S::RING, OUT = S::OUT;
    const int lane = threadIdx.x & 63;
    const int nx = p.nx, ny = p.ny;
    const bool out_lane = lane >= K - 1 && lane < K - 1 + OUT;
    const int sa = S::stage(wave), lag = S::lag(wave);
    const PTPRange ra = ptp_range<K>(sa, r0, r1, ny), rb = ptp_range<K>(sa + 1, r0, r1, ny);
    // every output lane's column is inside the grid by more than the boundary columns
    const bool inner = !e.any;
    PTPWin wa{}, wb{};
    PTPMat mb{};                          // the materials of stage B's row
    double pn_c = 0.0, dvx_c = 0.0, dvy_c = 0.0;  // P, dV handed over for stage A's next row
    PTRow oa{};                           // stage A's last row
    double rho_0 = 0.0, rho_m1 = 0.0;     // rho1 of stage A's row and the row above
    PTRow ob{};                           // stage B's last row
    // material slot of stage A's row at step t: row index t - lag
    int slot = (RING - lag % RING) % RING;
    int t = 0;
    // Lanes that store P, dVy and Vy; dVx and Vx; and the columns beside the boundary ones.
    const bool st_p = out_lane && c < nx - 1, st_x = out_lane && c < nx - 2;
    const bool st_l = out_lane && c == 0, st_r = out_lane && c == nx - 2;
    const unsigned cb = 8 * (unsigned)c;
    // Row pointers of the next stored row (none of rows 0, 1 and ny-1).
    struct Rows {
        double *p, *dvx, *vx, *dvy, *vy;
    } q{};
    auto store = [&](const PTRow& out, int ro, auto mid_tag) {
        if constexpr (decltype(mid_tag)::value) {
            if (ro < r0) return;  // the pipeline fills
            if (inner) {
                if (out_lane) {
                    ptp_at(q.p, cb) = out.pn;
                    ptp_at(q.dvx, cb) = out.dvx;
                    ptp_at(q.vx, cb) = out.vx;
                    ptp_at(q.dvy, cb) = out.dvy;
                    ptp_at(q.vy, cb) = out.vy;
                }
            } else {
                if (st_p) {
                    ptp_at(q.p, cb) = out.pn;
                    ptp_at(q.dvy, cb) = out.dvy;
                    ptp_at(q.vy, cb) = out.vy;
                }
                if (st_x) {
                    ptp_at(q.dvx, cb) = out.dvx;
                    ptp_at(q.vx, cb) = out.vx;
                }
                if (st_l) {  // bc_x_zero!, bc_x_noflux!
                    q.vx[-1] = 0.0;
                    q.vy[-1] = out.vy;
                }
                if (st_r) {
                    q.vx[nx - 2] = 0.0;
                    q.vy[nx - 1] = out.vy;
                }
            }
            q.p += nx - 1;
            q.dvx += nx - 2;
            q.vx += nx;
            q.dvy += nx - 1;
            q.vy += nx + 1;
        } else {
            pt2_store(p, out, c, ro, r0, out_lane);
        }
    };
    auto aim = [&](int ro) {  // the row pointers at row ro
        const int64_t r = ro;
        q = Rows{p.p_b + r * (nx - 1), p.dvx_o + (r - 1) * (nx - 2), p.vx_b + r * nx + 1, p.dvy_o + (r - 1) * (nx - 1),
                 p.vy_b + r * (nx + 1) + 1};
    };
    // One step.  MID: no stage runs a boundary row.  Rows outside a stage's range (while the pipeline
    // fills and drains) are then computed like the others, from whatever the buffers hold: no row
    // of the range depends on them, and none of them is stored.
    auto step = [&](auto mid_tag) {
        constexpr bool MID = decltype(mid_tag)::value;
        const int r = rstart + t - lag;
        const int slot1 = slot + 1 == RING ? 0 : slot + 1;
        const double* const hi = hand_in + ((t + 1) & 1) * PTP_HAND + lane;
        const double* const ms = mats + slot * (PTP_MATS * SF_WAVE) + lane;
        const double vx1 = hi[0], vx1p = hi[1], vy1 = hi[PTP_VROW], vy1p = hi[PTP_VROW + 1];
        PTPMat ma;
        ma.m2 = ms[0];
        ma.mub = ms[SF_WAVE];
        ma.taup = ms[2 * SF_WAVE];
        ma.tauvx = ms[3 * SF_WAVE];
        ma.tauvy = ms[4 * SF_WAVE];
        ma.rho1 = rho_0;
        ma.dxi = ms[6 * SF_WAVE];
        const double rho_1 = mats[slot1 * (PTP_MATS * SF_WAVE) + 5 * SF_WAVE + lane];
        ma.dyi = rho_1 - rho_m1;
        const double pn_n = hi[2 * PTP_VROW], dvx_n = hi[2 * PTP_VROW + SF_WAVE], dvy_n = hi[2 * PTP_VROW + 2 * SF_WAVE];
        const double pn_b = oa.pn, dvx_b = oa.dvx, dvy_b = oa.dvy;
        bool have = MID;  // the wave hands over (or stores) a row
        if (MID || (r >= ra.lo && r <= ra.hi)) {
            if (!MID && r == 0) {  // Vx row 0 = row 1, Vy row 0 zero
                wa.vx = vx1;
                wa.vxp = vx1p;
                wa.vy = wa.vyp = 0.0;
            }
            oa = ptp_row(kc, wa, vx1, vx1p, vy1, vy1p, ma, pn_c, dvx_c, dvy_c);
            if (!TWO) have = true;
            if (TWO || !LAST) ptp_bc(e, !MID && r == ny - 1, oa.vx, oa.vy);
        } else {
            wa.vx = vx1;
            wa.vxp = vx1p;
            wa.vy = vy1;
            wa.vyp = vy1p;
            if (r == ny) oa.vy = 0.0;  // virtual row ny: Vx row ny = row ny-1, Vy zero
        }
        if constexpr (TWO) {
            const int ro = r - 1;
            const double ux = lane_up(oa.vx, 1), uy = lane_up(oa.vy, 1);
            if (MID || (ro >= rb.lo && ro <= rb.hi)) {
                if (!MID && ro == 0) {
                    wb.vx = ux;
                    wb.vxp = oa.vx;
                    wb.vy = wb.vyp = 0.0;
                }
                ob = ptp_row(kc, wb, ux, oa.vx, uy, oa.vy, mb, pn_b, dvx_b, dvy_b);
                have = true;
                if (!LAST) ptp_bc(e, !MID && ro == ny - 1, ob.vx, ob.vy);
            } else {
                wb.vx = ux;
                wb.vxp = oa.vx;
                wb.vy = uy;
                wb.vyp = oa.vy;
                if (ro == ny) ob.vy = 0.0;
            }
            if constexpr (LAST) {
                if (have) store(ob, ro, mid_tag);
            } else {
                if (have || ro == ny) ptp_put(hand_out + (t & 1) * PTP_HAND, lane, ob);
            }
        } else {
            static_assert(TWO || LAST, "only the last wave may have one stage");
            if (have) store(oa, r, mid_tag);
        }
        mb = ma;
        pn_c = pn_n;
        dvx_c = dvx_n;
        dvy_c = dvy_n;
        rho_m1 = rho_0;
        rho_0 = rho_1;
        slot = slot1;
        ++t;
        ptp_barrier();
    };
    // Boundary rows: stage A at row 0 up to the later stage at row 0 (LAST: 1, whose store writes row
    // 0 too), and stage A at row ny-1 and all later steps.
    constexpr int B = TWO ? 1 : 0;
    const int ta = lag - rstart;                  // the step at which stage A runs row 0
    const int tb = min(ta + ny - 1, steps);       // and row ny-1
    for (int part = 0; part < 2; ++part) {
        const int te = part == 0 && rstart == 0 ? min(ta, tb) : tb;
        const int tf = part == 1 ? steps : (rstart == 0 ? min(ta + 1 + B + (LAST ? 1 : 0), steps) : te);
        if constexpr (LAST) aim(max(rstart + t - lag - B, r0));
        while (t + 1 < te) {  // two steps per trip: values carried on alternate between two registers
            step(std::true_type{});
            step(std::true_type{});
        }
        if (t < te) step(std::true_type{});
        while (t < tf) step(std::false_type{});
    }
}

// The parameters behind a pointer that the compiler takes for a new one: each role's loop then loads
// the ones it uses (scalar loads) instead of holding those of all roles, which spilled SGPRs.
typedef const PTParams __attribute__((address_space(4))) PTParamsC;
__device__ __forceinline__ PTParamsC& ptp_fresh(PTParamsC& p)
{
    PTParamsC* q = &p;
    asm volatile("" : "+s"(q));
    return *q;
}

// K PT iterations over the tile (strip, segid) of seg rows by the PTPShape<K>::WAVES waves of a workgroup:
// state k from (vx_a, vy_a, p_a, dvx, dvy), state k+K to (vx_b, vy_b, p_b, dvx_o, dvy_o); lds holds
// PTPShape<K>::LDS doubles.  Every wave of the workgroup calls this (one barrier per step).
template <int K>
__device__ __forceinline__ void ptp_tile(PTParamsC& p, int seg, int strip, int segid, double* lds)
{
    typedef PTPShape<K> S;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nx = p.nx, ny = p.ny;
    const int c0 = strip * S::OUT - (K - 1);
    const int c = c0 + lane;
    const int r0 = segid * seg;
    const int r1 = min(r0 + seg, ny);
    const int rstart = max(r0 - K, 0);
    const int steps = r1 - rstart + S::LAG;
    PTPEdge e;
    e.any = c0 < 0 || c0 + SF_WAVE + 1 >= nx;
    e.vx_zero = (c + 1 == 0) || (c + 1 == nx - 1);
    e.vy_left = c + 1 == 0;
    e.vy_right = c + 1 == nx;
    PTPConst kc;
    kc.rdx = p.rdx;
    kc.rdy = p.rdy;
    kc.rdx8 = 0.125 * p.rdx;
    kc.rdy2 = 0.5 * p.rdy;
    kc.g = p.g;
    kc.dt = *p.dt;
    kc.dampx = p.dampx;
    kc.dampy = p.dampy;
    double* const mats = lds;
    double* const hand = lds + S::RING * PTP_MATS * SF_WAVE;
    // The waves meet at every step's barrier, and the first (loads, divisions) and the last (stores)
    // have the most instructions to issue besides their arithmetic: they go first.
    if (wave == 0) {
        __builtin_amdgcn_s_setprio(3);
        ptp_first<K>(ptp_fresh(p), kc, e, mats, hand, c, r0, r1, rstart, steps);
    } else {
        const double* const hi = hand + (wave - 1) * 2 * PTP_HAND;
        double* const ho = hand + wave * 2 * PTP_HAND;
        if (wave < S::WAVES - 1) {
            ptp_later<K, true, false>(ptp_fresh(p), kc, e, mats, hi, ho, wave, c, r0, r1, rstart, steps);
        } else {
            __builtin_amdgcn_s_setprio(2);
            ptp_later<K, S::LAST_TWO, true>(ptp_fresh(p), kc, e, mats, hi, ho, wave, c, r0, r1, rstart, steps);
        }
    }
}

}  // namespace sf
