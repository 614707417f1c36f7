// The reference's barotropic_dynamics (Function/vel_ssh.f90:379-679) as one
// fused kernel launch per leap-frog substep, behind the reference's own
// boundary: 2*nstep substeps (nstep state-advancing, nstep look-ahead),
// the state after substep nstep returned as the call's result (:638-648),
// the averages ubrtr_i, vbrtr_i, ssh4gradx, ssh4grady accumulated over all
// 2*nstep substeps (:549-550, :567-568), the caller's RHS, water flux,
// viscosity and Rayleigh coefficient per cell, and any metrics.  The
// depths at entry are hh_init(ssh_e, sshp_e) as the reference holds them
// between calls (depth.f90:2-105, vel_ssh.f90:668-675); nothing of them is
// stored: level-n depths are formed from the surface height and the
// filtered U/V depths are carried between substeps as hh_shift filters
// them (depth.f90:174-220).
//
// Arithmetic: the reference's expressions operation by operation, in its
// evaluation order, without fused multiply-add (the library is compiled
// with -ffp-contract=off): the results are the reference's bit for bit.
//
// Work decomposition as in the fused step (bt_fused.hip): one 64-lane wave
// owns a strip of 60 output columns (lanes 0-1 and 62-63 are halo) and
// marches down a chunk of rows with a rolling register window three rows
// deep; x-neighbours come from the adjacent lanes by DPP row shifts.  An
// intermediate that the reference evaluates at a neighbouring point is
// taken from the neighbour's lane (or the previous row) only where the
// reference's expression there is the same, operand for operand, up to the
// order of an addition of two terms (fx_m(m) = fx_p(m-1), fy_m(n) =
// fy_p(n-1)); everything else is evaluated as written.
//
// Eligible calls: full_free_surface = 1, no periodicity, and land on the
// two halo cells of every side (the reference's loop bounds then coincide
// with its masks).  Other calls take the stage-by-stage path.
// Two kernels: the march of k_dropin, and one point per lane on tiles
// (k_dropin_tile) for small grids and for the biharmonic term uv_diff4
// (ksw4 > 0, vel_ssh.f90:187-317), which it forms in the same launch.
// Metrics: per cell (any grid), or per row when every metric and the
// Coriolis parameter are uniform along x (Cartesian and longitude-latitude
// grids): then they are read from row tables instead of 8 + 1 arrays; or one
// number (uniform metrics), whose quotients the march shares (bt_exactdiv.h).
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "bt_dropin.h"
#include "bt_fused_body.h"
#include "bt_literal.h"

namespace ibt {

struct DropinParams {
    int nx, ny, strips, chunk, nchunks, total, per_xcd;
    const uint8_t *mb;
    const double *H, *rd, *mu, *wf, *rx, *ry;
    // dx, dy, dxt, dyt, dxh, dyh, dxb, dyb and rlh_s: per cell, or (ROWMET)
    // per row, row n at [n - 1]; rows only: dy/dx, dx/dy, dxb/dyb, dyb/dxb
    const double *met[13];
    const double *u, *v, *s, *up, *vp, *sp;  // state entering the substep
    double *uo, *vo, *so, *upo, *vpo, *spo;  // state after it (uo null: not written)
    double *cu, *cv, *cs, *cup, *cvp, *csp;  // copy of the entering state (cu null: none)
    double *hupc, *hvpc;                     // filtered U/V depths carried in place (substeps > 1 read)
    bool carry_out;                          // write the filtered U/V depths for the next substep
    double *acc[4];                          // ubrtr_i, vbrtr_i, ssh4gradx, ssh4grady, in place
    const double *mu4;                       // the biharmonic viscosity (ksw4 > 0)
    double g, rho0, ts, tau, ffs;
    // divisors that every point shares (bt_exactdiv.h): rho0, tau, dfloat(nstep),
    // 4 nstep and, on uniform metrics, d and d * d; the limit of ExpCheck
    Den q_rho0, q_tau, q_dn, q_d4n, q_d, q_dd;
    int exp_lim;
};

// how the metrics are read: per cell, per row, or one number for all
enum { MET_CELL = 0, MET_ROW = 1, MET_ONE = 2 };

// What iteration n consumes (outside the array the mask is 0 and the rest
// whatever the clamped loads give: every use is selected by a mask, or
// multiplied by a depth that is 0 there; zeroing the row metrics by lane would
// hold them in vector registers): row n+2 of the
// surface height, depth at rest, masks, dx, dy; row n+1 of the level-n and
// filtered velocities and height, Rayleigh coefficient, viscosity, water
// flux, dxt, dyh, dxh, dyt; row n of the Coriolis parameter, the caller's
// RHS, dxb, dyb, the carried depths and the accumulators.
struct DIn {
    double s2, H2, dx2, dy2;
    int mb2;
    double u1, v1, up1, vp1, sp1, rd1, mu1, wf1, dxt1, dyh1, dxh1, dyt1;
    double f0, rx0, ry0, dxb0, dyb0, hupc0, hvpc0, a0, a1, a2, a3;
};

// What one substep produces for row n.
struct DOut {
    double s, u, v, sp, up, vp;  // state after the Robert-Asselin shift
    double hu, hv;               // hh_shift-filtered U/V depths
    double a0, a1, a2, a3;       // accumulators
};

// One substep marching down the rows of one strip.  Suffixes: m1 = row
// n-1, 0 = row n, p1 = row n+1, p2 = row n+2.  FIRST: the call's first
// substep (filtered depths from hh_init, accumulators start at zero).
template <bool FIRST, bool ONE>
struct DStage {
    const DropinParams &p;
    const bool inx, inx1;

    double u_0 = 0, u_p1 = 0, v_0 = 0, v_p1 = 0, s_0 = 0, s_p1 = 0, s_p2 = 0, H_p1 = 0, H_p2 = 0;
    double up_0 = 0, up_p1 = 0, vp_0 = 0, vp_p1 = 0, sp_0 = 0, sp_p1 = 0, rd_0 = 0, rd_p1 = 0;
    double mu_m1 = 0, mu_0 = 0, mu_p1 = 0;
    int mb_m1 = 0, mb_0 = 0, mb_p1 = 0, mb_p2 = 0;
    double dx_p1 = 0, dx_p2 = 0, dy_p1 = 0, dy_p2 = 0;
    double dxt_0 = 0, dxt_p1 = 0, dyh_0 = 0, dyh_p1 = 0, dxh_0 = 0, dxh_p1 = 0, dyt_0 = 0, dyt_p1 = 0;
    double dxb_m1 = 0;
    double hq_0 = 0, hq_p1 = 0, hq_p2 = 0;  // level-n T depth
    double w_0 = 0, w_p1 = 0, w_p2 = 0;     // hq*dx*dy*lu (depth.f90 area weights)
    double wp_0 = 0, wp_p1 = 0;             // the same for the filtered level (hh_init)
    double wn_0 = 0, wn_p1 = 0;             // the same for the new level (hh_update)
    double hu_0 = 0, hu_p1 = 0, hup_0 = 0, hup_p1 = 0, hv_0 = 0, hv_p1 = 0, hun_0 = 0, hun_p1 = 0;
    double hh_m1 = 0, hh_0 = 0;
    double sn_0 = 0, sn_p1 = 0;
    double P_0 = 0, Px_0 = 0;      // dy^2*mu*hq*str_t and dx^2*mu*hq*str_t on T points
    double sts_m1 = 0;             // str_s of row n-1
    double Cc_m1 = 0, Fc_m1 = 0;   // row n-1 vorticity and Coriolis terms of the zonal equation
    double A_0 = 0;                // u*dyh*hu on U points
    double Bv_0 = 0;               // v*dxh*hv on V points
    double fv_0 = 0;               // v*hv*dxh on V points (continuity)
    double b_0 = 0, c_0 = 0, h_0 = 0;  // vp/dxh (V), up/dxt and u*dxt (U)
    double fyU_m1 = 0, fyV_m1 = 0;     // fy_p of row n-1 (zonal and meridional equations)
    int slow = 0;                      // ONE: rows for which the depths take IEEE divisions

    __device__ DStage(const DropinParams &pp, int m)
        : p(pp), inx(m >= 3 && m <= pp.nx - 2), inx1(m >= 2 && m <= pp.nx - 1)
    {
    }

    // hh_init / hh_update's average onto a U or V point of two T area weights,
    // and onto an H point of four (Function/depth.f90:29-66): (w_a + w_b) / slu /
    // metric_1 / metric_2, slu the number of wet T cells; here what follows the
    // first quotient, `mean`
    __device__ __forceinline__ double avg(double mean, double m1, double m2) const
    {
        if constexpr (!ONE) return mean / m1 / m2;
        double a[1] = {mean};
        quots2(a, p.q_d, slow > 0);
        return a[0];
    }
    // a[k] / m[k], metrics (ONE: all of them d)
    template <int N>
    __device__ __forceinline__ void by_metric(double (&a)[N], const double (&m)[N]) const
    {
        if constexpr (ONE) {
            by(a, p.q_d);
        } else {
#pragma unroll
            for (int k = 0; k < N; ++k) a[k] = a[k] / m[k];
        }
    }
    // a[k] / d, after a look at the numerators; with metrics per row or cell by
    // IEEE divisions: there the quotients' operands spill (2048 x 1536, us per
    // substep: rows 187 -> 221, cells 235 -> 633)
    template <int N>
    __device__ __forceinline__ void by(double (&a)[N], const Den &d) const
    {
        ExpCheck ck;
        if constexpr (ONE) {
#pragma unroll
            for (int k = 0; k < N; ++k) ck.add(a[k]);
            quots(a, d, ck.any(p.exp_lim));
        } else {
#pragma unroll
            for (int k = 0; k < N; ++k) a[k] = a[k] / d.b;
        }
    }

    __device__ __forceinline__ void row(int n, const DIn &q, bool produce, DOut &o)
    {
        const double G = p.g, tau = p.tau;
        const int k1 = n + 1;
        s_p2 = q.s2;
        H_p2 = q.H2;
        mb_p2 = q.mb2;
        dx_p2 = q.dx2;
        dy_p2 = q.dy2;
        u_p1 = q.u1;
        v_p1 = q.v1;
        up_p1 = q.up1;
        vp_p1 = q.vp1;
        sp_p1 = q.sp1;
        rd_p1 = q.rd1;
        mu_p1 = q.mu1;
        dxt_p1 = q.dxt1;
        dyh_p1 = q.dyh1;
        dxh_p1 = q.dxh1;
        dyt_p1 = q.dyt1;
        const double dxb_0 = q.dxb0, dyb_0 = q.dyb0;

        const int lu_0 = mb_0 & MB_LU ? 1 : 0, lu_p1 = mb_p1 & MB_LU ? 1 : 0, lu_p2 = mb_p2 & MB_LU ? 1 : 0;
        const double lf_p1 = lu_p1, lf_p2 = lu_p2;
        const int lus_0 = lu_0 + xr(lu_0), lus_p1 = lu_p1 + xr(lu_p1);
        const double in_u = inv_cells(lus_p1), in_v0 = inv_cells(lu_0 + lu_p1);
        const bool iny1 = (k1 >= 3 && k1 <= p.ny - 2);

        // ---- depths at level n (hh_init at the first substep, hh_update's
        // results of the previous substep afterwards: both are these
        // averages of hq = H + ssh, depth.f90:21-66, 122-150)
        hq_p2 = H_p2 + s_p2;
        w_p2 = hq_p2 * dx_p2 * dy_p2 * lf_p2;
        if constexpr (FIRST) wp_p1 = (H_p1 + sp_p1) * dx_p1 * dy_p1 * lf_p1;  // hh_init's filtered level
        if constexpr (ONE) {
            ExpCheck ck;
            ck.add(w_p2);
            if (FIRST) ck.add(wp_p1);
            slow = ck.any(p.exp_lim) ? 4 : slow - 1;
        }
        {
            const double w1r = xr(w_p1);
            hu_p1 = (mb_p1 & MB_LLU) ? avg((w_p1 + w1r) * in_u, dxt_p1, dyh_p1) : 0.0;
            hv_p1 = (mb_p1 & MB_LLV) ? avg((w_p1 + w_p2) * inv_cells(lu_p1 + lu_p2), dxh_p1, dyt_p1) : 0.0;
            const double w0r = xr(w_0), mean = mean_cells(w_0 + w0r + w_p1 + w1r, lus_0 + lus_p1);
            hh_0 = (mb_0 & MB_LUH) ? avg(mean, dxb_0, dyb_0) : 0.0;
        }
        double hvp_0 = 0.0;
        if constexpr (FIRST) {
            // filtered-level depths of hh_init (depth.f90:22, :32-34, :41-43)
            const double wp1r = xr(wp_p1);
            hup_p1 = (mb_p1 & MB_LLU) ? avg((wp_p1 + wp1r) * in_u, dxt_p1, dyh_p1) : 0.0;
            hvp_0 = (mb_0 & MB_LLV) ? avg((wp_0 + wp_p1) * in_v0, dxh_0, dyt_0) : 0.0;
        }

        // ---- T point of row n+1: continuity (vel_ssh.f90:487-499)
        const double fu_p1 = u_p1 * hu_p1 * dyh_p1;
        const double fv_p1 = v_p1 * hv_p1 * dxh_p1;
        {
            const bool tw = (mb_p1 & MB_LU) && inx && iny1;
            double wf[1] = {q.wf1}, div[1] = {fu_p1 - xl(fu_p1) + fv_p1 - fv_0};
            by(wf, p.q_rho0);
            if constexpr (ONE)
                by(div, p.q_dd);
            else
                div[0] = div[0] / (dx_p1 * dy_p1);
            const double sn = sp_p1 + 2.0 * tau * (wf[0] * p.ffs - div[0]);
            sn_p1 = tw ? sn : 0.0;
        }
        // new-level depths (hh_update, depth.f90:122-150)
        const double hqn_p1 = H_p1 + sn_p1;
        wn_p1 = hqn_p1 * dx_p1 * dy_p1 * lf_p1;
        if constexpr (ONE) {
            ExpCheck ck;
            ck.add(wn_p1);
            if (ck.any(p.exp_lim)) slow = 4;
        }
        const double wn1r = xr(wn_p1);
        hun_p1 = (mb_p1 & MB_LLU) ? avg((wn_p1 + wn1r) * in_u, dxt_p1, dyh_p1) : 0.0;
        const double hvn_0 = (mb_0 & MB_LLV) ? avg((wn_0 + wn_p1) * in_v0, dxh_0, dyt_0) : 0.0;

        // tension of the filtered level on T points of row n+1 (mixing.f90:129-132)
        // and the two products uv_diff2 takes of it (vel_ssh.f90:146-148, 162-164)
        double P_p1, Px_p1;
        double ab[2] = {up_p1, vp_p1};
        by_metric(ab, {dyh_p1, dxh_p1});
        const double e_0 = ONE ? b_0 : vp_0 / dyt_0, c_p1 = ONE ? ab[0] : up_p1 / dxt_p1;
        {
            const bool tw = (mb_p1 & MB_LU) && inx && iny1;
            const double a_p1 = ab[0];
            const double b_p1 = ab[1];
            // d / d is 1 on uniform metrics
            const double yx = ONE ? 1.0 : dy_p1 / dx_p1, xy = ONE ? 1.0 : dx_p1 / dy_p1;
            const double st = yx * (a_p1 - xl(a_p1)) - xy * (b_p1 - b_0);
            const double stt_p1 = tw ? st : 0.0;
            P_p1 = dy_p1 * dy_p1 * mu_p1 * hq_p1 * stt_p1;
            Px_p1 = dx_p1 * dx_p1 * mu_p1 * hq_p1 * stt_p1;
            b_0 = b_p1;  // consumed above as row n; row n+1 from here on
        }
        // flux-form advection factors on U and V points of row n+1 (vel_ssh.f90:63-70, 88-95)
        const double A_p1 = u_p1 * dyh_p1 * hu_p1;
        const double Bv_p1 = v_p1 * dxh_p1 * hv_p1;

        // ---- H point of row n: shear of the filtered level (mixing.f90:141-144)
        // and the metric vorticity (vel_ssh.f90:35-37)
        double sts_0, vo_0;
        {
            const bool hw = (mb_0 & MB_LUU) && inx && (n >= 3 && n <= p.ny - 2);
            const double bxy = ONE ? 1.0 : dxb_0 / dyb_0, byx = ONE ? 1.0 : dyb_0 / dxb_0;
            const double ss = bxy * (c_p1 - c_0) + byx * (xr(e_0) - e_0);
            const double h_p1 = u_p1 * dxt_p1;
            const double g_0 = v_0 * dyt_0;
            const double vo = (xr(g_0) - g_0) - (h_p1 - h_0) - ((xr(v_0) - v_0) * dyb_0 - (u_p1 - u_0) * dxb_0);
            sts_0 = hw ? ss : 0.0;
            vo_0 = hw ? vo : 0.0;
            c_0 = c_p1;
            h_0 = h_p1;
        }
        const double v0r = xr(v_0);
        // fy_p of the zonal equation on U(m, n) (vel_ssh.f90:69-70), every row:
        // row n's is fy_m of row n+1
        const double fyU_0 = (Bv_0 + xr(Bv_0)) / 2.0 * (u_p1 + u_0) / 2.0 * bitf<double>(mb_0, MB_LUU);
        // fy_p of the meridional equation on V(m, n) (:88-89)
        const double fyV_0 = (Bv_0 + Bv_p1) / 2.0 * (v_0 + v_p1) / 2.0;
        // vorticity and Coriolis terms on H(m, n) (:76-77, vel_ssh.f90:545-546)
        const double vh = vo_0 * hh_0;
        const double Cc_0 = vh * (v0r + v_0);
        const double fhdd = q.f0 * hh_0 * dxb_0 * dyb_0;
        const double Fc_0 = fhdd * (v0r + v_0);

        if (produce) {
            const bool iny = (n >= 3 && n <= p.ny - 2);
            const double hupc = FIRST ? hup_0 : q.hupc0;
            const double hvpc = FIRST ? hvp_0 : q.hvpc0;
            const double muh_p = (mu_0 + xr(mu_0) + mu_p1 + xr(mu_p1)) / 4.0;

            // zonal momentum (vel_ssh.f90:534-551) with uv_trans (:59-81) and uv_diff2 (:146-159)
            const double fx_p = (A_0 + xr(A_0)) / 2.0 * (u_0 + xr(u_0)) / 2.0;
            const double fx_m = xl(fx_p);
            const double radv = -(fx_p - fx_m + fyU_0 - fyU_m1) + (Cc_0 + Cc_m1) / 4.0;
            const double muh_m = (mu_0 + xr(mu_0) + mu_m1 + xr(mu_m1)) / 4.0;
            const double muhv_m = (mu_0 + xl(mu_0) + mu_p1 + xl(mu_p1)) / 4.0;
            const double dybl = xl(dyb_0), hhl = xl(hh_0), stsl = xl(sts_0), P0r = xr(P_0);
            double rdfx, rdfy, bp, bp0, bq, bq0;
            if constexpr (ONE) {
                double df[4] = {P0r - P_0,
                                dxb_0 * dxb_0 * muh_p * hh_0 * sts_0 - dxb_m1 * dxb_m1 * muh_m * hh_m1 * sts_m1,
                                Px_p1 - Px_0,
                                dyb_0 * dyb_0 * muh_p * hh_0 * sts_0 - dybl * dybl * muhv_m * hhl * stsl};
                double b[4] = {hun_0 * dxt_0 * dyh_0 / 2.0, hupc * dxt_0 * dyh_0 / 2.0, hvn_0 * dyt_0 * dxh_0 / 2.0,
                               hvpc * dyt_0 * dxh_0 / 2.0};
                by(df, p.q_d);
                by(b, p.q_tau);
                rdfx = df[0] + df[1];
                rdfy = -df[2] + df[3];
                bp = b[0];
                bp0 = b[1];
                bq = b[2];
                bq0 = b[3];
            } else {
                rdfx = (P0r - P_0) / dyh_0 +
                       (dxb_0 * dxb_0 * muh_p * hh_0 * sts_0 - dxb_m1 * dxb_m1 * muh_m * hh_m1 * sts_m1) / dxt_0;
                rdfy = -(Px_p1 - Px_0) / dxh_0 +
                       (dyb_0 * dyb_0 * muh_p * hh_0 * sts_0 - dybl * dybl * muhv_m * hhl * stsl) / dyt_0;
                bp = hun_0 * dxt_0 * dyh_0 / 2.0 / tau;
                bp0 = hupc * dxt_0 * dyh_0 / 2.0 / tau;
                bq = hvn_0 * dyt_0 * dxh_0 / 2.0 / tau;
                bq0 = hvpc * dyt_0 * dxh_0 / 2.0 / tau;
            }
            const double slx = -G * (xr(s_0) - s_0) * dyh_0 * hu_0;
            const double slxn = -G * (xr(sn_0) - sn_0) * dyh_0 * hun_0;
            const double grx = q.rx0 + slx + rdfx + radv - (rd_0 + xr(rd_0)) / 2.0 * up_0 * dxt_0 * dyh_0 * hu_0 +
                               (Fc_0 + Fc_m1) / 4.0;
            double un = (up_0 * bp0 + grx) / bp;

            // meridional momentum (vel_ssh.f90:554-569) with uv_trans (:84-105) and uv_diff2 (:162-175)
            const double fxV_p = (A_0 + A_p1) / 2.0 * (v0r + v_0) / 2.0;
            const double fxV_m = xl(fxV_p);
            const double D = vh * (u_p1 + u_0);
            const double rady = -(fxV_p - fxV_m + fyV_0 - fyV_m1) - (D + xl(D)) / 4.0;
            const double sly = -G * (s_p1 - s_0) * dxh_0 * hv_0;
            const double slyn = -G * (sn_p1 - sn_0) * dxh_0 * hvn_0;
            const double Gc = fhdd * (u_p1 + u_0);
            const double gry = q.ry0 + sly + rdfy + rady - (rd_0 + rd_p1) / 2.0 * vp_0 * dxh_0 * dyt_0 * hv_0 -
                               (Gc + xl(Gc)) / 4.0;
            double vn = (vp_0 * bq0 + gry) / bq;

            const bool uw = (mb_0 & MB_LCU) && inx && iny;
            const bool vw = (mb_0 & MB_LCV) && inx && iny;
            un = uw ? un : 0.0;
            vn = vw ? vn : 0.0;

            // averages over the call's substeps (vel_ssh.f90:549-550, 567-568)
            const double a0 = FIRST ? 0.0 : q.a0, a1 = FIRST ? 0.0 : q.a1;
            const double a2 = FIRST ? 0.0 : q.a2, a3 = FIRST ? 0.0 : q.a3;
            if constexpr (ONE) {
                double t[4] = {u_0 * hu_0 + un * hun_0, v_0 * hv_0 + vn * hvn_0, slx + slxn, sly + slyn};
                by(t, p.q_d4n);
                o.a0 = uw ? a0 + t[0] : a0;
                o.a1 = vw ? a1 + t[1] : a1;
                o.a2 = uw ? a2 + t[2] : a2;
                o.a3 = vw ? a3 + t[3] : a3;
            } else {
                o.a0 = uw ? a0 + (u_0 * hu_0 + un * hun_0) / p.q_d4n.b : a0;
                o.a2 = uw ? a2 + (slx + slxn) / p.q_d4n.b : a2;
                o.a1 = vw ? a1 + (v_0 * hv_0 + vn * hvn_0) / p.q_d4n.b : a1;
                o.a3 = vw ? a3 + (sly + slyn) / p.q_d4n.b : a3;
            }

            // time-level shift with the Robert-Asselin filter (vel_ssh.f90:588-612)
            // and hh_shift of the U/V depths (depth.f90:195-203)
            const double ts = p.ts;
            if constexpr (ONE) {
                double e[5] = {ts * (sn_0 - 2.0 * s_0 + sp_0) / 2.0, ts * (un - 2.0 * u_0 + up_0) / 2.0,
                               ts * (vn - 2.0 * v_0 + vp_0) / 2.0, ts * (hun_0 - 2.0 * hu_0 + hupc) / 2.0,
                               ts * (hvn_0 - 2.0 * hv_0 + hvpc) / 2.0};
                by(e, p.q_dn);
                const bool sh = inx1 && n >= 2 && n <= p.ny - 1;
                const bool bs = sh && (mb_0 & MB_LU), bu = sh && (mb_0 & MB_LCU), bv = sh && (mb_0 & MB_LCV);
                o.s = bs ? sn_0 : s_0;
                o.u = bu ? un : u_0;
                o.v = bv ? vn : v_0;
                o.sp = bs ? s_0 + e[0] : sp_0;
                o.up = bu ? u_0 + e[1] : up_0;
                o.vp = bv ? v_0 + e[2] : vp_0;
                o.hu = sh && (mb_0 & MB_LLU) ? hu_0 + e[3] : hupc;
                o.hv = sh && (mb_0 & MB_LLV) ? hv_0 + e[4] : hvpc;
            } else {
                double s_new = s_0, u_new = u_0, v_new = v_0;
                double sp_new = sp_0, up_new = up_0, vp_new = vp_0;
                double hu_new = hupc, hv_new = hvpc;
                const double dn = p.q_dn.b;
                if (inx1 && n >= 2 && n <= p.ny - 1) {
                    if (mb_0 & MB_LU) {
                        sp_new = s_0 + ts * (sn_0 - 2.0 * s_0 + sp_0) / 2.0 / dn;
                        s_new = sn_0;
                    }
                    if (mb_0 & MB_LCU) {
                        up_new = u_0 + ts * (un - 2.0 * u_0 + up_0) / 2.0 / dn;
                        u_new = un;
                    }
                    if (mb_0 & MB_LCV) {
                        vp_new = v_0 + ts * (vn - 2.0 * v_0 + vp_0) / 2.0 / dn;
                        v_new = vn;
                    }
                    if (mb_0 & MB_LLU) hu_new = hu_0 + ts * (hun_0 - 2.0 * hu_0 + hupc) / 2.0 / dn;
                    if (mb_0 & MB_LLV) hv_new = hv_0 + ts * (hvn_0 - 2.0 * hv_0 + hvpc) / 2.0 / dn;
                }
                o.s = s_new;
                o.u = u_new;
                o.v = v_new;
                o.sp = sp_new;
                o.up = up_new;
                o.vp = vp_new;
                o.hu = hu_new;
                o.hv = hv_new;
            }
        }

        // ---- advance the window one row
        u_0 = u_p1;
        v_0 = v_p1;
        s_0 = s_p1;
        s_p1 = s_p2;
        H_p1 = H_p2;
        up_0 = up_p1;
        vp_0 = vp_p1;
        sp_0 = sp_p1;
        rd_0 = rd_p1;
        mu_m1 = mu_0;
        mu_0 = mu_p1;
        mb_m1 = mb_0;
        mb_0 = mb_p1;
        mb_p1 = mb_p2;
        dx_p1 = dx_p2;
        dy_p1 = dy_p2;
        dxt_0 = dxt_p1;
        dyh_0 = dyh_p1;
        dxh_0 = dxh_p1;
        dyt_0 = dyt_p1;
        dxb_m1 = dxb_0;
        hq_0 = hq_p1;
        hq_p1 = hq_p2;
        w_0 = w_p1;
        w_p1 = w_p2;
        wp_0 = wp_p1;
        wn_0 = wn_p1;
        hu_0 = hu_p1;
        hup_0 = hup_p1;
        hv_0 = hv_p1;
        hun_0 = hun_p1;
        hh_m1 = hh_0;
        sn_0 = sn_p1;
        P_0 = P_p1;
        Px_0 = Px_p1;
        sts_m1 = sts_0;
        Cc_m1 = Cc_0;
        Fc_m1 = Fc_0;
        A_0 = A_p1;
        Bv_0 = Bv_p1;
        fv_0 = fv_p1;
        fyU_m1 = fyU_0;
        fyV_m1 = fyV_0;
    }
};

// Loads of one iteration, issued one iteration ahead of their use.  As the fused step's Loader: a row's address by the scalar unit, a lane's
// constant column added to it.
template <bool FIRST, int MET>
struct DLoader {
    const DropinParams &p;
    const uint32_t col;  // the lane's column, clamped, from 0
    const bool colok;
    struct Pre {
        double s, H, dx, dy, u, v, up, vp, sp, rd, mu, wf, dxt, dyh, dxh, dyt, f, rx, ry, dxb, dyb, hupc, hvpc;
        double a[4];
        int mb;
    } q;

    __device__ DLoader(const DropinParams &pp, int m)
        : p(pp), col(min(max(m, 1), pp.nx) - 1), colok(m >= 1 && m <= pp.nx)
    {
    }
    __device__ __forceinline__ bool rowok(int row) const { return colok && row >= 1 && row <= p.ny; }
    // the lane's element of the row whose index row_of gave
    template <class T>
    __device__ __forceinline__ T at(const T *base, size_t row) const
    {
        if constexpr (MET == MET_CELL) return base[row];
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base + row) + (uint32_t)(col * sizeof(T)));
    }
    // metric k (0..7: dx dy dxt dyt dxh dyh dxb dyb; 8: rlh_s) at (this column,
    // row), whose cells start at element i
    __device__ __forceinline__ double met(int k, int row, size_t i) const
    {
        if (MET == MET_ONE && k < 8) return p.q_d.b;
        if constexpr (MET != MET_CELL)
            return scalar_load(p.met[k] + min(max(row, 1), p.ny) - 1);
        else
            return at(p.met[k], i);
    }
    // first element of a row, or (MET_CELL) the lane's own element of it: there
    // nine more arrays' scalar addresses spill (235 us a substep -> 547)
    __device__ __forceinline__ size_t row_of(int r) const
    {
        return (size_t)(min(max(r, 1), p.ny) - 1) * (size_t)p.nx + (MET == MET_CELL ? col : 0u);
    }
    __device__ __forceinline__ void issue(int n)
    {
        const size_t i2 = row_of(n + 2), i1 = row_of(n + 1), i0 = row_of(n);
        q.s = at(p.s, i2);
        q.H = at(p.H, i2);
        q.mb = at(p.mb, i2);
        q.dx = met(0, n + 2, i2);
        q.dy = met(1, n + 2, i2);
        q.u = at(p.u, i1);
        q.v = at(p.v, i1);
        q.up = at(p.up, i1);
        q.vp = at(p.vp, i1);
        q.sp = at(p.sp, i1);
        q.rd = at(p.rd, i1);
        q.mu = at(p.mu, i1);
        q.wf = at(p.wf, i1);
        q.dxt = met(2, n + 1, i1);
        q.dyt = met(3, n + 1, i1);
        q.dxh = met(4, n + 1, i1);
        q.dyh = met(5, n + 1, i1);
        q.dxb = met(6, n, i0);
        q.dyb = met(7, n, i0);
        q.f = met(8, n, i0);
        q.rx = at(p.rx, i0);
        q.ry = at(p.ry, i0);
        if constexpr (!FIRST) {
            q.hupc = at((const double *)p.hupc, i0);
            q.hvpc = at((const double *)p.hvpc, i0);
            for (int k = 0; k < 4; ++k) q.a[k] = at((const double *)p.acc[k], i0);
        }
    }
    __device__ __forceinline__ void take(int n, DIn &in) const
    {
        in.s2 = q.s;
        in.H2 = q.H;
        in.mb2 = rowok(n + 2) ? q.mb : 0;
        in.dx2 = q.dx;
        in.dy2 = q.dy;
        in.u1 = q.u;
        in.v1 = q.v;
        in.up1 = q.up;
        in.vp1 = q.vp;
        in.sp1 = q.sp;
        in.rd1 = q.rd;
        in.mu1 = q.mu;
        in.wf1 = q.wf;
        in.dxt1 = q.dxt;
        in.dyh1 = q.dyh;
        in.dxh1 = q.dxh;
        in.dyt1 = q.dyt;
        in.f0 = q.f;
        in.rx0 = q.rx;
        in.ry0 = q.ry;
        in.dxb0 = q.dxb;
        in.dyb0 = q.dyb;
        if constexpr (!FIRST) {
            in.hupc0 = q.hupc;
            in.hvpc0 = q.hvpc;
            in.a0 = q.a[0];
            in.a1 = q.a[1];
            in.a2 = q.a[2];
            in.a3 = q.a[3];
        } else {
            in.hupc0 = in.hvpc0 = in.a0 = in.a1 = in.a2 = in.a3 = 0.0;
        }
    }
};

// Two waves per SIMD.  Measured on MI355X, us per substep before (metrics per row
// or cell, 44 IEEE divisions a point) / now: one metric (MET_ONE: two IEEE
// divisions, the others by d, tau, rho0 and the numbers of substeps from their
// reciprocals) 700 x 600 37.6 / 29.4, 1300 x 1000 81 / 71, 2048 x 1536 187 / 177,
// where its 224 bytes a cell take 144; per row (depth means by products, scalar row
// addresses) 38.0 / 36.5, 81 / 78.6, 186 / 183; per cell unchanged.
template <bool FIRST, int MET>
__global__ void __launch_bounds__(WAVE, 2) k_dropin(DropinParams p)
{
    const int w = blockIdx.x;
    const int t = (w % NXCD) * p.per_xcd + (w / NXCD);
    if (t >= p.total) return;
    const int chunk_id = t / p.strips, strip = t - chunk_id * p.strips;
    const int lane = threadIdx.x;
    const int m = strip * SW + lane - 1;
    const bool colok = (m >= 1 && m <= p.nx);
    const bool writer = colok && lane >= 2 && lane <= SW + 1;
    const int r0 = chunk_id * p.chunk + 1;
    const int r1 = min(r0 + p.chunk, p.ny + 1);

    DStage<FIRST, MET == MET_ONE> st(p, m);
    DLoader<FIRST, MET> ld(p, m);
    DIn in;
    DOut o;
    ld.issue(r0 - 3);
    for (int n = r0 - 3; n < r1; ++n) {
        ld.take(n, in);
        if (n + 1 < r1) ld.issue(n + 1);
        const bool produce = n >= r0;
        if (produce && p.cu && writer) {
            // the state entering this substep (the call's result when this is
            // substep nstep + 1, vel_ssh.f90:638-648), row n of the window
            const size_t io = (size_t)(n - 1) * p.nx + (m - 1);
            st_out<true, double>(p.cu, io, st.u_0);
            st_out<true, double>(p.cv, io, st.v_0);
            st_out<true, double>(p.cs, io, st.s_0);
            st_out<true, double>(p.cup, io, st.up_0);
            st_out<true, double>(p.cvp, io, st.vp_0);
            st_out<true, double>(p.csp, io, st.sp_0);
        }
        st.row(n, in, produce, o);
        if (produce && writer) {
            const size_t io = (size_t)(n - 1) * p.nx + (m - 1);
            if (p.uo) {
                st_out<true, double>(p.so, io, o.s);
                st_out<true, double>(p.uo, io, o.u);
                st_out<true, double>(p.vo, io, o.v);
                st_out<true, double>(p.spo, io, o.sp);
                st_out<true, double>(p.upo, io, o.up);
                st_out<true, double>(p.vpo, io, o.vp);
            }
            if (p.carry_out) {
                p.hupc[io] = o.hu;
                p.hvpc[io] = o.hv;
            }
            p.acc[0][io] = o.a0;
            p.acc[1][io] = o.a1;
            p.acc[2][io] = o.a2;
            p.acc[3][io] = o.a3;
        }
    }
}

// Small grids: one substep per launch on tiles of 64 x nr points, one point
// per lane and one row per wave (the scheme of the fast modes' fused_tile).
// A march gives a 289 x 163 grid 400 waves of 5 dependent rows, and the
// biharmonic term two more launches; here a substep is four phases (six with
// the biharmonic term, whose terms are formed in the same launch) with the
// row neighbours' values exchanged through LDS, the column neighbours' by
// lane shifts.  A substep reaches two points at most in every direction, so a
// tile writes lanes 2..61 of rows 2..nr-3.  The expressions are DStage's and
// the stage-by-stage path's (uv_diff4), operand for operand: the same bits.
// FIRST of DStage is the launch argument here (it is uniform).
// Measured on MI355X, us per substep on a longitude-latitude grid, march /
// tiles: 285 x 159 14.5 / 7.7, 512 x 384 24.3 / 19.1 (take_march has the sizes
// where the march is the faster); with the biharmonic term (its march took two
// more launches) 285 x 159 42 / 10.3, 2048 x 1536 408 / 369, and with metrics
// per cell 657 / 434.  Bound by FP64 issue (about 30 IEEE divisions a point, 50
// with the term) and, below 300 x 200, by the launch and the phases' latency.
constexpr int DT_MAX_ROWS = 12;
constexpr int DT_RIM = 4;  // rows of a tile that it does not write
constexpr int DT_ARRAYS = 18;
constexpr size_t dropin_tile_lds(int nr) { return (size_t)DT_ARRAYS * nr * WAVE * sizeof(double); }

template <bool ROWMET, bool D4>
__global__ void __launch_bounds__(WAVE * DT_MAX_ROWS) k_dropin_tile(DropinParams p, int first)
{
    extern __shared__ __attribute__((aligned(16))) double dt_shared[];
    const int t = (blockIdx.x % NXCD) * p.per_xcd + (blockIdx.x / NXCD);
    if (t >= p.total) return;  // the whole block
    const int ty = t / p.strips, tx = t - ty * p.strips;
    const int lane = threadIdx.x % WAVE, nr = blockDim.x / WAVE;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const int m = tx * SW + lane - 1, n = ty * (nr - DT_RIM) + w - 1;
    auto at = [&](int a, int r) -> double & { return dt_shared[(a * nr + r) * WAVE + lane]; };
    const int rn = min(w + 1, nr - 1), rs = max(w - 1, 0);  // (the rim rows' neighbours reach no output)

    const RowAddr ra{p.nx, p.ny, min(max(m, 1), p.nx)};
    const bool colok = m >= 1 && m <= p.nx;
    const size_t i0 = ra.at(n), i1 = ra.at(n + 1), is = ra.at(n - 1);
    const double u = p.u[i0], v = p.v[i0], s = p.s[i0], up = p.up[i0], vp = p.vp[i0], sp = p.sp[i0];
    const double H = p.H[i0], rd = p.rd[i0], rd1 = p.rd[i1], mu = p.mu[i0], mu1 = p.mu[i1], mus = p.mu[is];
    const double wf = p.wf[i0], rx = p.rx[i0], ry = p.ry[i0];
    double mu4 = 0.0, mu41 = 0.0, mu4s = 0.0;
    if constexpr (D4) {
        mu4 = p.mu4[i0];
        mu41 = p.mu4[i1];
        mu4s = p.mu4[is];
    }
    int mb = p.mb[i0], mb1 = p.mb[i1];
    auto met = [&](int k, int row, size_t i) -> double {
        if constexpr (ROWMET)
            return p.met[k][min(max(row, 1), p.ny) - 1];
        else
            return p.met[k][i];
    };
    const double dx = met(0, n, i0), dy = met(1, n, i0), dxt = met(2, n, i0), dyt = met(3, n, i0);
    const double dxh = met(4, n, i0), dyh = met(5, n, i0), dxb = met(6, n, i0), dyb = met(7, n, i0);
    const double f = met(8, n, i0), dxbs = met(6, n - 1, is);
    if (!(colok && n >= 1 && n <= p.ny)) mb = 0;
    if (!(colok && n + 1 >= 1 && n + 1 <= p.ny)) mb1 = 0;
    const bool writer = colok && n >= 1 && n <= p.ny && lane >= 2 && lane <= SW + 1 && w >= 2 && w <= nr - 3;
    const size_t io = i0;  // a writer's point is in the array
    double hupc = 0.0, hvpc = 0.0, a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    if (!first && writer) {
        hupc = p.hupc[io];
        hvpc = p.hvpc[io];
        a0 = p.acc[0][io];
        a1 = p.acc[1][io];
        a2 = p.acc[2][io];
        a3 = p.acc[3][io];
    }

    const bool in = m >= 3 && m <= p.nx - 2 && n >= 3 && n <= p.ny - 2;
    const double lu0 = bitf<double>(mb, MB_LU), lu1 = bitf<double>(mb1, MB_LU);
    const double lu0r = xr(lu0), lu1r = xr(lu1);
    const bool tw = (mb & MB_LU) && in, hw = (mb & MB_LUU) && in;
    const double G = p.g, tau = p.tau;

    // ---- phase 1: depths' area weights and the stresses' quotients
    const double hq = H + s;
    const double w0 = hq * dx * dy * lu0;
    const double wp0 = (H + sp) * dx * dy * lu0;
    const double qa = up / dyh, qb = vp / dxh, qc = up / dxt, qe = vp / dyt;
    const double hh_ = u * dxt, gg = v * dyt;
    at(0, w) = w0;
    at(1, w) = wp0;
    at(2, w) = qb;
    at(3, w) = qc;
    at(4, w) = hh_;
    at(5, w) = u;
    at(6, w) = s;
    at(7, w) = v;
    __syncthreads();
    // ---- phase 2: depths, fluxes, stresses, vorticity and Coriolis products
    auto avg = [](double wsum, double slu, double m1, double m2) { return wsum / slu / m1 / m2; };
    const double w1 = at(0, rn), w0r = xr(w0), w1r = xr(w1);
    double hu = avg(w0 + w0r, lu0 + lu0r, dxt, dyh), hv = avg(w0 + w1, lu0 + lu1, dxh, dyt);
    double hh = avg(w0 + w0r + w1 + w1r, lu0 + lu0r + lu1 + lu1r, dxb, dyb);
    hu = (mb & MB_LLU) ? hu : 0.0;
    hv = (mb & MB_LLV) ? hv : 0.0;
    hh = (mb & MB_LUH) ? hh : 0.0;
    if (first) {
        const double wp1 = at(1, rn), wp0r = xr(wp0);
        hupc = (mb & MB_LLU) ? avg(wp0 + wp0r, lu0 + lu0r, dxt, dyh) : 0.0;
        hvpc = (mb & MB_LLV) ? avg(wp0 + wp1, lu0 + lu1, dxh, dyt) : 0.0;
    }
    const double qbs = at(2, rs), qc1 = at(3, rn), hh1_ = at(4, rn), u1 = at(5, rn), s1 = at(6, rn), v1 = at(7, rn);
    const double vs = at(7, rs);
    const double fu = u * hu * dyh, fv = v * hv * dxh;
    const double A = u * dyh * hu, Bv = v * dxh * hv;
    double yx, xy, bxy, byx;
    if constexpr (ROWMET) {
        yx = met(9, n, i0);
        xy = met(10, n, i0);
        bxy = met(11, n, i0);
        byx = met(12, n, i0);
    } else {
        yx = dy / dx;
        xy = dx / dy;
        bxy = dxb / dyb;
        byx = dyb / dxb;
    }
    const double st = yx * (qa - xl(qa)) - xy * (qb - qbs);
    const double stt = tw ? st : 0.0;
    const double P = dy * dy * mu * hq * stt, Px = dx * dx * mu * hq * stt;
    const double ss = bxy * (qc1 - qc) + byx * (xr(qe) - qe);
    const double v0r = xr(v);
    const double vo_ = (xr(gg) - gg) - (hh1_ - hh_) - ((v0r - v) * dyb - (u1 - u) * dxb);
    const double sts = hw ? ss : 0.0, vo = hw ? vo_ : 0.0;
    const double fyU = (Bv + xr(Bv)) / 2.0 * (u1 + u) / 2.0 * bitf<double>(mb, MB_LUU);
    const double vh = vo * hh;
    const double Cc = vh * (v0r + v);
    const double fhdd = f * hh * dxb * dyb;
    const double Fc = fhdd * (v0r + v);
    double P4 = 0.0, Px4 = 0.0;
    at(8, w) = fv;
    at(9, w) = Bv;
    at(10, w) = A;
    at(11, w) = Px;
    at(12, w) = hh;
    at(13, w) = sts;
    at(14, w) = fyU;
    at(15, w) = Cc;
    at(16, w) = Fc;
    if constexpr (D4) {
        P4 = dy * dy * mu4 * hq * stt;
        Px4 = dx * dx * mu4 * hq * stt;
        at(17, w) = Px4;
    }
    __syncthreads();
    // ---- phase 3: continuity and the new depths; uv_diff4's first pass
    const double fvs = at(8, rs), Bvs = at(9, rs), Bv1 = at(9, rn), A1 = at(10, rn), Px1 = at(11, rn);
    const double hhs = at(12, rs), stss = at(13, rs), fyUs = at(14, rs), Ccs = at(15, rs), Fcs = at(16, rs);
    const double sn_ = sp + 2.0 * tau * (wf / p.rho0 * p.ffs - (fu - xl(fu) + fv - fvs) / (dx * dy));
    const double sn = tw ? sn_ : 0.0;
    const double wn0 = (H + sn) * dx * dy * lu0;
    at(0, w) = wn0;
    at(1, w) = sn;
    const double dybl = xl(dyb), hhl = xl(hh), stsl = xl(sts);
    double qa4 = 0.0, qb4 = 0.0, qc4 = 0.0, qe4 = 0.0, mu4p = 0.0, mu4m = 0.0, mu4v = 0.0;
    if constexpr (D4) {
        const double mu4r = xr(mu4), mu41r = xr(mu41);
        mu4p = (mu4 + mu4r + mu41 + mu41r) / 4.0;
        mu4m = (mu4 + mu4r + mu4s + xr(mu4s)) / 4.0;
        mu4v = (mu4 + xl(mu4) + mu41 + xl(mu41)) / 4.0;
        const double pu = (xr(P4) - P4) / dyh;
        const double qu = (dxb * dxb * mu4p * hh * sts - dxbs * dxbs * mu4m * hhs * stss) / dxt;
        const double pv = (at(17, rn) - Px4) / dxh;
        const double qv = (dyb * dyb * mu4p * hh * sts - dybl * dybl * mu4v * hhl * stsl) / dyt;
        const double fu4 = pu + qu, fv4 = -pv + qv;
        const double vx = -fu4 / hu / dxt / dyh, vy = -fv4 / hv / dxh / dyt;
        const double fx = ((mb & MB_LCU) && in) ? vx : 0.0, fy = ((mb & MB_LCV) && in) ? vy : 0.0;
        qa4 = fx / dyh;
        qb4 = fy / dxh;
        qc4 = fx / dxt;
        qe4 = fy / dyt;
        at(2, w) = qb4;
        at(3, w) = qc4;
    }
    __syncthreads();
    const double wn1 = at(0, rn), sn1 = at(1, rn);
    double px = 0.0, qx = 0.0, py = 0.0, qy = 0.0;
    if constexpr (D4) {
        // uv_diff4's second pass: the stress of (fx, fy) and its two terms
        const double tt = yx * (qa4 - xl(qa4)) - xy * (qb4 - at(2, rs));
        const double sh = bxy * (at(3, rn) - qc4) + byx * (xr(qe4) - qe4);
        const double stt4 = tw ? tt : 0.0, sts4 = hw ? sh : 0.0;
        const double R4 = dy * dy * mu4 * hq * stt4, Rx4 = dx * dx * mu4 * hq * stt4;
        at(4, w) = Rx4;
        at(5, w) = sts4;
        __syncthreads();
        const double sts4l = xl(sts4);
        px = (xr(R4) - R4) / dyh;
        qx = (dxb * dxb * mu4p * hh * sts4 - dxbs * dxbs * mu4m * hhs * at(5, rs)) / dxt;
        py = (at(4, rn) - Rx4) / dxh;
        qy = (dyb * dyb * mu4p * hh * sts4 - dybl * dybl * mu4v * hhl * sts4l) / dyt;
    }
    // ---- last phase: momentum, averages, time-level shift (DStage::row)
    double hun = avg(wn0 + xr(wn0), lu0 + lu0r, dxt, dyh), hvn = avg(wn0 + wn1, lu0 + lu1, dxh, dyt);
    hun = (mb & MB_LLU) ? hun : 0.0;
    hvn = (mb & MB_LLV) ? hvn : 0.0;
    const double mur = xr(mu), mu1r = xr(mu1);
    const double muh_p = (mu + mur + mu1 + mu1r) / 4.0;
    const double fx_p = (A + xr(A)) / 2.0 * (u + xr(u)) / 2.0;
    const double fx_m = xl(fx_p);
    const double radv = -(fx_p - fx_m + fyU - fyUs) + (Cc + Ccs) / 4.0;
    const double muh_m = (mu + mur + mus + xr(mus)) / 4.0;
    double rdfx = (xr(P) - P) / dyh + (dxb * dxb * muh_p * hh * sts - dxbs * dxbs * muh_m * hhs * stss) / dxt;
    if constexpr (D4) rdfx = rdfx + px + qx;
    const double bp = hun * dxt * dyh / 2.0 / tau;
    const double bp0 = hupc * dxt * dyh / 2.0 / tau;
    const double slx = -G * (xr(s) - s) * dyh * hu;
    const double slxn = -G * (xr(sn) - sn) * dyh * hun;
    const double grx = rx + slx + rdfx + radv - (rd + xr(rd)) / 2.0 * up * dxt * dyh * hu + (Fc + Fcs) / 4.0;
    double un = (up * bp0 + grx) / bp;

    const double fxV_p = (A + A1) / 2.0 * (v0r + v) / 2.0;
    const double fxV_m = xl(fxV_p);
    const double fyV = (Bv + Bv1) / 2.0 * (v + v1) / 2.0, fyVs = (Bvs + Bv) / 2.0 * (vs + v) / 2.0;
    const double D = vh * (u1 + u);
    const double rady = -(fxV_p - fxV_m + fyV - fyVs) - (D + xl(D)) / 4.0;
    const double muhv_m = (mu + xl(mu) + mu1 + xl(mu1)) / 4.0;
    double rdfy = -(Px1 - Px) / dxh + (dyb * dyb * muh_p * hh * sts - dybl * dybl * muhv_m * hhl * stsl) / dyt;
    if constexpr (D4) rdfy = rdfy - py + qy;
    const double bq = hvn * dyt * dxh / 2.0 / tau;
    const double bq0 = hvpc * dyt * dxh / 2.0 / tau;
    const double sly = -G * (s1 - s) * dxh * hv;
    const double slyn = -G * (sn1 - sn) * dxh * hvn;
    const double Gc = fhdd * (u1 + u);
    const double gry = ry + sly + rdfy + rady - (rd + rd1) / 2.0 * vp * dxh * dyt * hv - (Gc + xl(Gc)) / 4.0;
    double vn = (vp * bq0 + gry) / bq;
    const bool uw = (mb & MB_LCU) && in, vw = (mb & MB_LCV) && in;
    un = uw ? un : 0.0;
    vn = vw ? vn : 0.0;
    if (!writer) return;
    if (p.cu) {
        // the state entering this substep: the call's result when this is
        // substep nstep + 1 (vel_ssh.f90:638-648)
        p.cu[io] = u;
        p.cv[io] = v;
        p.cs[io] = s;
        p.cup[io] = up;
        p.cvp[io] = vp;
        p.csp[io] = sp;
    }
    p.acc[0][io] = uw ? a0 + (u * hu + un * hun) / p.q_d4n.b : a0;
    p.acc[2][io] = uw ? a2 + (slx + slxn) / p.q_d4n.b : a2;
    p.acc[1][io] = vw ? a1 + (v * hv + vn * hvn) / p.q_d4n.b : a1;
    p.acc[3][io] = vw ? a3 + (sly + slyn) / p.q_d4n.b : a3;
    if (!p.uo) return;
    const double ts = p.ts;
    const bool sh_ = m >= 2 && m <= p.nx - 1 && n >= 2 && n <= p.ny - 1;
    const double spn = s + ts * (sn - 2.0 * s + sp) / 2.0 / p.q_dn.b;
    const double upn = u + ts * (un - 2.0 * u + up) / 2.0 / p.q_dn.b;
    const double vpn = v + ts * (vn - 2.0 * v + vp) / 2.0 / p.q_dn.b;
    const double hupn = hu + ts * (hun - 2.0 * hu + hupc) / 2.0 / p.q_dn.b;
    const double hvpn = hv + ts * (hvn - 2.0 * hv + hvpc) / 2.0 / p.q_dn.b;
    const bool bs = sh_ && (mb & MB_LU), bu = sh_ && (mb & MB_LCU), bv = sh_ && (mb & MB_LCV);
    p.so[io] = bs ? sn : s;
    p.spo[io] = bs ? spn : sp;
    p.uo[io] = bu ? un : u;
    p.upo[io] = bu ? upn : up;
    p.vo[io] = bv ? vn : v;
    p.vpo[io] = bv ? vpn : vp;
    p.hupc[io] = sh_ && (mb & MB_LLU) ? hupn : hupc;
    p.hvpc[io] = sh_ && (mb & MB_LLV) ? hvpn : hvpc;
}

// ------------------------------------------------------------------ host

struct DropinAlloc {
    double *S[2][6] = {};  // ping-pong state of the substeps: u, up, v, vp, ssh, sshp
    double *hupc = nullptr, *hvpc = nullptr;
    double *rowmet = nullptr;  // 13 x ny: the metrics, rlh_s and four quotients per row (uniform along x)
    uint8_t *mb = nullptr;
    int eligible = -1;  // grid part of the eligibility: -1 not checked, 0 no, 1 yes
    std::string why;
    bool rowmet_ok = false;
    int met = MET_CELL;  // how the march reads the metrics
    int chunk = 0;
    long long slots = 0;
    int tile_nr[2] = {};  // rows per tile without and with the biharmonic term (0: the march)
};

namespace {

// doubles per plane of the substeps' buffers, rounded up to 256 bytes
size_t scratch_plane(size_t n) { return (n + 31) / 32 * 32; }

#define DHC(expr)                                                                              \
    do {                                                                                       \
        hipError_t e_ = (expr);                                                                \
        if (e_ != hipSuccess) {                                                                \
            set_error(std::string(#expr) + ": " + hipGetErrorString(e_));                      \
            return INMSOM_BT_EDEVICE;                                                          \
        }                                                                                      \
    } while (0)

__global__ void k_dropin_masks(size_t n, const float *lu, const float *luu, const float *luh, const float *lcu,
                               const float *lcv, const float *llu, const float *llv, uint8_t *mb)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint8_t b = 0;
    if (lu[i] > 0.5f) b |= MB_LU;
    if (lcu[i] > 0.5f) b |= MB_LCU;
    if (lcv[i] > 0.5f) b |= MB_LCV;
    if (luu[i] > 0.5f) b |= MB_LUU;
    if (luh[i] > 0.5f) b |= MB_LUH;
    if (llu[i] > 0.5f) b |= MB_LLU;
    if (llv[i] > 0.5f) b |= MB_LLV;
    mb[i] = b;
}

template <bool FIRST>
const void *march_kernel(int met)
{
    return met == MET_ONE   ? (const void *)k_dropin<FIRST, MET_ONE>
           : met == MET_ROW ? (const void *)k_dropin<FIRST, MET_ROW>
                            : (const void *)k_dropin<FIRST, MET_CELL>;
}

const void *tile_kernel(bool rowmet, bool d4)
{
    return rowmet ? (d4 ? (const void *)k_dropin_tile<true, true> : (const void *)k_dropin_tile<true, false>)
                  : (d4 ? (const void *)k_dropin_tile<false, true> : (const void *)k_dropin_tile<false, false>);
}

// Whether a call without the biharmonic term takes the march, by the rounds in
// which the CUs, one block each, work through the t tiles of 12 rows (with the
// term: the tiles always).  A tile's time goes in such steps, the march's with the
// cells.  Measured on MI355X (256 CUs), us per substep, march / the better tiles,
// with t: metrics per row 340 x 260 (198) 17.3 / 11.3, 380 x 300 (266) 21.8 / 18.3,
// 512 x 384 (441) 24.6 / 20.0, 540 x 420 (530) 29.2 / 29.8, 600 x 440 (616) 30.3 /
// 28.6, 640 x 512 (715) 32.0 / 30.7, 620 x 580 (803) 35.7 / 37.3; per cell 340 x 260
// 17.5 / 12.1, 380 x 300 21.9 / 19.7, 540 x 420 30.5 / 34.0, 600 x 440 34.1 / 32.8,
// 640 x 512 37.6 / 35.2, 620 x 580 39.9 / 42.8; one metric, whose quotients only
// the march shares, 340 x 260 13.6 / 11.3, 380 x 300 16.3 / 18.1, 512 x 384 18.7 /
// 20.5, 640 x 512 26.7 / 30.7.
bool take_march(int met, long long t, long long cus)
{
    if (met == MET_ONE) return t > cus;
    return t > 3 * cus || (t > 2 * cus && 3 * t < 7 * cus);
}

// Whether this grid's calls run on tiles, and their rows, 8 or 12: the fewer us
// by the rounds r of each, 9.0 r + 1.3 with 12 rows and 5.2 r + 3.1 with 8 (with
// the biharmonic term 1.3 times as long; us with 12 / 8 rows without and with it:
// 285 x 159, r = 1 and 1, 10.6 / 8.7, 13.8 / 11.2; 340 x 260, 1 and 2, 11.3 / 13.5,
// 15.0 / 17.9; 400 x 360, 2 and 3, 19.0 / 18.7, 25.7 / 25.0; 512 x 384, 2 and 4,
// 20.0 / 23.8, 27.2 / 31.3; 1021 x 763 with it 83 / 93).
int choose_tiles(inmsom_bt_ctx *c, DropinAlloc *a, int cus)
{
    const long long strips = (c->nx + SW - 1) / SW;
    auto tiles = [&](int nr) { return strips * ((c->ny + nr - DT_RIM - 1) / (nr - DT_RIM)); };
    auto rounds = [&](int nr) { return (double)((tiles(nr) + cus - 1) / cus); };
    const int nr = 9.0 * rounds(12) + 1.3 < 5.2 * rounds(8) + 3.1 ? 12 : 8;
    for (int d4 = 0; d4 < 2; ++d4) {
        a->tile_nr[d4] = d4 || !take_march(a->met, tiles(12), cus) ? nr : 0;
        DHC(hipFuncSetAttribute(tile_kernel(a->rowmet_ok, d4), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)dropin_tile_lds(DT_MAX_ROWS)));
    }
    return INMSOM_BT_OK;
}

// The grid part of the eligibility and the row tables, checked once per
// context (the static grid does not change).
int check_grid(inmsom_bt_ctx *c, DropinAlloc *a)
{
    if (a->eligible >= 0) return INMSOM_BT_OK;
    a->eligible = 0;
    if (c->g.ffs != 1) {
        a->why = "full_free_surface != 1";
        return INMSOM_BT_OK;
    }
    if (c->g.px || c->g.py) {
        a->why = "periodic grid";
        return INMSOM_BT_OK;
    }
    const int nx = c->nx, ny = c->ny;
    if (nx < 5 || ny < 5) {
        a->why = "grid smaller than 5 x 5";
        return INMSOM_BT_OK;
    }
    const size_t n = c->n;
    std::vector<float> lu(n);
    DHC(hipMemcpy(lu.data(), c->mask[0], n * 4, hipMemcpyDeviceToHost));
    for (int r = 1; r <= ny; ++r)
        for (int m = 1; m <= nx; ++m) {
            const bool halo = m <= 2 || m >= nx - 1 || r <= 2 || r >= ny - 1;
            if (halo && lu[(size_t)(r - 1) * nx + (m - 1)] > 0.5f) {
                a->why = "ocean on the two halo cells of a side (the loop bounds then differ from the masks)";
                return INMSOM_BT_OK;
            }
        }
    // metrics and rlh_s uniform along x on columns 2..nx-1: row tables.  With
    // land on the halo the outputs never depend on columns 1 and nx (the
    // reference's own grid set-up leaves its metrics zero there and rlh_s
    // unscaled, Service/basin_parameters.f90:250-300).
    std::vector<double> f(n), tab((size_t)13 * ny);
    bool rows = true;
    for (int k = 0; k < 9 && rows; ++k) {
        DHC(hipMemcpy(f.data(), k < 8 ? c->metric[k] : c->rlh_s, n * 8, hipMemcpyDeviceToHost));
        for (int r = 0; r < ny && rows; ++r) {
            const double *row = &f[(size_t)r * nx];
            for (int m = 2; m < nx - 1; ++m)
                if (std::memcmp(&row[m], &row[1], sizeof(double)) != 0) {
                    rows = false;
                    break;
                }
            tab[(size_t)k * ny + r] = row[1];
        }
    }
    a->rowmet_ok = rows;
    for (int r = 0; r < ny && rows; ++r) {
        const double dx = tab[r], dy = tab[ny + r], dxb = tab[(size_t)6 * ny + r], dyb = tab[(size_t)7 * ny + r];
        tab[(size_t)9 * ny + r] = dy / dx;
        tab[(size_t)10 * ny + r] = dx / dy;
        tab[(size_t)11 * ny + r] = dxb / dyb;
        tab[(size_t)12 * ny + r] = dyb / dxb;
    }
    if (rows) {
        DHC(hipMalloc(&a->rowmet, tab.size() * 8));
        DHC(hipMemcpy(a->rowmet, tab.data(), tab.size() * 8, hipMemcpyHostToDevice));
    }
    DHC(hipMalloc(&a->mb, n));
    hipLaunchKernelGGL(k_dropin_masks, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, n, c->mask[0],
                       c->mask[1], c->mask[2], c->mask[3], c->mask[4], c->mask[5], c->mask[6], a->mb);
    DHC(hipGetLastError());
    // launch shape: rows per wave filling whole rounds of the device's wave slots
    int dev = 0, cus = 0, per_cu = 0;
    DHC(hipGetDevice(&dev));
    DHC(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    a->met = !rows ? MET_CELL
             : c->uniform_metrics && c->metric0 > DEN_MIN && c->metric0 < DEN_MAX ? MET_ONE
                                                                                 : MET_ROW;
    DHC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, march_kernel<false>(a->met), WAVE, 0));
    a->slots = (long long)cus * (per_cu > 0 ? per_cu : 1);
    const int strips = (nx + SW - 1) / SW;
    a->chunk = fit_chunk(ny, strips, a->slots, 3, 2);
    if (const int rc = choose_tiles(c, a, cus)) return rc;
    DHC(hipStreamSynchronize(c->stream));
    a->eligible = 1;
    return INMSOM_BT_OK;
}

// the substeps' two state sets and carried depths (14 planes of n doubles)
// in library-owned memory, allocated at the first call that needs them
int ensure_buffers(inmsom_bt_ctx *c, DropinAlloc *a)
{
    const size_t n = c->n;
    for (int b = 0; b < 2; ++b)
        for (int k = 0; k < 6; ++k)
            if (!a->S[b][k]) DHC(hipMalloc(&a->S[b][k], n * 8));
    if (!a->hvpc) DHC(hipMalloc(&a->hvpc, n * 8));
    if (!a->hupc) DHC(hipMalloc(&a->hupc, n * 8));
    return INMSOM_BT_OK;
}

template <bool FIRST>
void launch_dropin(inmsom_bt_ctx *c, const DropinParams &p, int met)
{
    dim3 grid((unsigned)(p.per_xcd * NXCD)), blk(WAVE);
    void *args[] = {const_cast<DropinParams *>(&p)};
    (void)hipLaunchKernel(march_kernel<FIRST>(met), grid, blk, args, 0, c->stream);
}

}  // namespace

static DropinAlloc *dalloc(inmsom_bt_ctx *c)
{
    if (!c->da) c->da = new DropinAlloc();
    return c->da;
}

bool dropin_eligible(inmsom_bt_ctx *c, int ksw4, std::string *why)
{
    DropinAlloc *a = dalloc(c);
    if (check_grid(c, a) != INMSOM_BT_OK) {
        if (why) *why = std::string("device error while checking the grid: ") + inmsom_bt_last_error();
        return false;
    }
    if (!a->eligible) {
        if (why) *why = a->why;
        return false;
    }
    (void)ksw4;  // the biharmonic term runs on the tiles
    return true;
}

int dropin_setup(inmsom_bt_ctx *c) { return check_grid(c, dalloc(c)); }

size_t dropin_scratch_doubles(const inmsom_bt_ctx *c) { return 14 * scratch_plane(c->n); }

int dropin_call(inmsom_bt_ctx *c, double tau, int nstep, double *const st[6], double *const acc[4],
                const double *rhsx, const double *rhsy, const double *wflux, const double *mu, const double *rdis,
                double *scratch, int ksw4, const double *mu4)
{
    DropinAlloc *a = dalloc(c);
    int rc = check_grid(c, a);
    if (rc) return rc;
    if (!a->eligible) {
        set_error("the fused barotropic_dynamics does not cover this grid: " + a->why);
        return INMSOM_BT_ESTATE;
    }
    // the substeps' state sets and carried depths: 14 planes
    double *S[2][6], *hupc, *hvpc;
    if (scratch) {
        const size_t plane = scratch_plane(c->n);
        for (int b = 0; b < 2; ++b)
            for (int k = 0; k < 6; ++k) S[b][k] = scratch + (size_t)(6 * b + k) * plane;
        hupc = scratch + 12 * plane;
        hvpc = scratch + 13 * plane;
    } else {
        if ((rc = ensure_buffers(c, a))) return rc;
        for (int b = 0; b < 2; ++b)
            for (int k = 0; k < 6; ++k) S[b][k] = a->S[b][k];
        hupc = a->hupc;
        hvpc = a->hvpc;
    }
    const int tile_nr = a->tile_nr[ksw4 > 0];
    DropinParams p{};
    p.nx = c->nx;
    p.ny = c->ny;
    p.strips = (c->nx + SW - 1) / SW;
    p.chunk = a->chunk;
    p.nchunks = (c->ny + a->chunk - 1) / a->chunk;
    p.total = p.strips * p.nchunks;
    p.per_xcd = (p.total + NXCD - 1) / NXCD;
    p.mb = a->mb;
    p.H = c->hr;
    p.rd = rdis;
    p.mu = mu;
    p.wf = wflux;
    p.rx = rhsx;
    p.ry = rhsy;
    for (int k = 0; k < 13; ++k)
        p.met[k] = a->rowmet_ok ? a->rowmet + (size_t)k * c->ny : k < 8 ? c->metric[k] : k == 8 ? c->rlh_s : nullptr;
    p.hupc = hupc;
    p.hvpc = hvpc;
    for (int k = 0; k < 4; ++k) p.acc[k] = acc[k];
    p.g = c->g.g;
    p.rho0 = c->g.rho0;
    p.ts = c->g.ts;
    p.tau = tau / (double)nstep;  // tau_inner, vel_ssh.f90:465
    p.ffs = (double)c->g.ffs;
    const double dn = (double)nstep, d4n = (double)(4 * nstep);
    p.q_rho0 = make_den(p.rho0);
    p.q_tau = make_den(p.tau);
    p.q_dn = make_den(dn);
    p.q_d4n = make_den(d4n);
    p.exp_lim = ExpCheck::LIMIT;
    for (const double d : {p.rho0, p.tau, dn, d4n})
        if (!(d > DEN_MIN && d < DEN_MAX)) p.exp_lim = -1;  // IEEE divisions throughout
    if (a->met == MET_ONE) {
        p.q_d = make_den(c->metric0);
        p.q_dd = make_den(c->metric0 * c->metric0);
    }
    if (ksw4 > 0) {
        if (!mu4) {
            set_error("mu4 is required when ksw4 > 0");
            return INMSOM_BT_EINVAL;
        }
    }
    if (tile_nr) {
        p.mu4 = mu4;
        p.chunk = tile_nr - DT_RIM;
        p.nchunks = (c->ny + p.chunk - 1) / p.chunk;
        p.total = p.strips * p.nchunks;
        p.per_xcd = (p.total + NXCD - 1) / NXCD;
    }
    const int last = 2 * nstep;
    for (int k = 1; k <= last; ++k) {
        // substep k reads the caller's state (k = 1) or the buffer substep
        // k - 1 wrote, and writes S[k % 2] (nothing after the last substep)
        const double *const *in = k == 1 ? (const double *const *)st : (const double *const *)S[(k - 1) % 2];
        p.u = in[0];
        p.up = in[1];
        p.v = in[2];
        p.vp = in[3];
        p.s = in[4];
        p.sp = in[5];
        double *const *out = S[k % 2];
        const bool wr = k < last;
        p.uo = wr ? out[0] : nullptr;
        p.upo = wr ? out[1] : nullptr;
        p.vo = wr ? out[2] : nullptr;
        p.vpo = wr ? out[3] : nullptr;
        p.so = wr ? out[4] : nullptr;
        p.spo = wr ? out[5] : nullptr;
        // substep nstep + 1 enters with the state after substep nstep: the
        // call's result (vel_ssh.f90:638-648)
        const bool snap = k == nstep + 1;
        p.cu = snap ? st[0] : nullptr;
        p.cup = snap ? st[1] : nullptr;
        p.cv = snap ? st[2] : nullptr;
        p.cvp = snap ? st[3] : nullptr;
        p.cs = snap ? st[4] : nullptr;
        p.csp = snap ? st[5] : nullptr;
        p.carry_out = k < last;
        if (tile_nr) {
            int first = k == 1;
            void *args[] = {&p, &first};
            (void)hipLaunchKernel(tile_kernel(a->rowmet_ok, ksw4 > 0), dim3((unsigned)(p.per_xcd * NXCD)),
                                  dim3((unsigned)(WAVE * tile_nr)), args, dropin_tile_lds(tile_nr), c->stream);
        } else if (k == 1)
            launch_dropin<true>(c, p, a->met);
        else
            launch_dropin<false>(c, p, a->met);
    }
    DHC(hipGetLastError());
    return INMSOM_BT_OK;
}

// Scratch of the entry point that allocates nothing
// (inmsom_bt_barotropic_dynamics_noalloc): the substeps' two state sets and
// carried depths, 14 planes of nx*ny doubles, in a fixed array every GPU the
// library runs on holds until the process ends.  Calls on one GPU share it:
// calls that overlap on one GPU race.  Nothing in it needs to start at
// zero (every plane is written before it is read within a call).
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)384 << 20;
static __device__ __align__(256) double scratch[NOALLOC_SCRATCH_BYTES / sizeof(double)];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
double *g_scratch[MAX_DEVICES] = {};
}  // namespace

int noalloc_scratch_setup(int device)
{
    if (device < 0 || device >= MAX_DEVICES) {
        set_error("device index beyond the scratch table");
        return INMSOM_BT_EINVAL;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[device]) return INMSOM_BT_OK;
    void *ptr = nullptr;  // the array's address on the current device (each GPU has its own copy)
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        set_error(std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        return INMSOM_BT_EDEVICE;
    }
    g_scratch[device] = static_cast<double *>(ptr);
    return INMSOM_BT_OK;
}

double *noalloc_scratch(int device, size_t *doubles)
{
    *doubles = NOALLOC_SCRATCH_BYTES / sizeof(double);
    if (device < 0 || device >= MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return g_scratch[device];
}

void dropin_release(inmsom_bt_ctx *c)
{
    DropinAlloc *a = c->da;
    if (!a) return;
    for (auto &b : a->S)
        for (double *q : b)
            if (q) (void)hipFree(q);
    for (void *q : {(void *)a->hupc, (void *)a->hvpc, (void *)a->rowmet, (void *)a->mb})
        if (q) (void)hipFree(q);
    delete a;
    c->da = nullptr;
}

void dropin_shape(const inmsom_bt_ctx *c, int *rows_per_wave, bool *row_metrics)
{
    *rows_per_wave = c->da ? c->da->chunk : 0;
    *row_metrics = c->da ? c->da->rowmet_ok : false;
}

}  // namespace ibt
