// Device body of the fused barotropic step, shared by the single-basin
// kernel (bt_fused.hip) and the batched-ensemble kernel (bt_ensemble.hip).
// The algorithm and its modes are described at the top of bt_fused.hip.
#pragma once

#include <type_traits>

#include "bt_exactdiv.h"
#include "bt_internal.h"

namespace ibt {

constexpr int WAVE = 64;
constexpr int SW = 60;   // output columns per wave, one substep per launch
constexpr int SW2 = 58;  // output columns per wave, two substeps per launch
constexpr int NXCD = 8;
// cells (summed over an ensemble's members) from which the fused step's fast
// modes run substep pairs as a two-wave pipeline by default, and below which
// they run them on tiles (fused_tile).  Measured on MI355X, us per substep,
// tiles / pipeline: 512 x 384 FP64 7.9 / 8.2, FP32 6.4 / 8.4; 640 x 512 FP64
// 11.4 / 10.8, FP32 9.1 / 9.8; 768 x 640 FP64 15.3 / 13.5, FP32 12.2 / 10.1;
// 1021 x 763 FP64 22.3 / 17.0, FP32 17.5 / 13.0.
constexpr long long TWO_SUBSTEP_CELLS = 300000;

struct FusedParams {
    int nx, ny, strips, chunk, nchunks, total, per_xcd;
    const uint8_t *mb;
    const void *H, *rd;     // stencil type
    const void *u, *v, *s;  // level n, stencil type
    const double *up, *vp, *sp;
    void *uo, *vo, *so;
    double *upo, *vpo, *spo;
    const double *row_f, *row_sx, *row_sy, *row_wf;  // per row, index n-1
    double g, rho0, ts, tau, cb, eb, nu, ffs, d;
    // sub-cycling: substep `sub` of `nsub` (tau = tau_inner = outer tau / nsub)
    int sub, nsub;
    double dn;             // dfloat(nstep)
    double inv_d, g_d, nu_d, ffs_rho0;  // 1 / d, g / d, nu / d, ffs / rho0
    Den q_d, q_dd, q_tau, q_dn, q_rho0;    // FP64_EXACT: divisors d, d * d, tau, dn, rho0
    int exp_lim;                           // and the limit of ExpCheck
    void *frx, *fry;       // forcing frozen over the substeps of one call (stencil type), written
    const void *frx_in, *fry_in;  // the same, read (a separate buffer when a launch forms new forcing)
    // filtered U/V depths carried between substeps (FP64_EXACT only): read, and
    // written for the next launch (the other buffer: a pair's work items read
    // them on the rows around their own)
    const double *hup_in, *hvp_in;
    double *hup_c, *hvp_c;
};

// the constants' quotients of the fast modes and FP64_EXACT's divisors, once on
// the host, and the divisors that go with a call's time step
constexpr double DEN_MIN = 0x1p-60, DEN_MAX = 0x1p60;  // divisors' range (ExpCheck)
inline void step_constants(FusedParams &p)
{
    p.inv_d = 1.0 / p.d;
    p.g_d = p.g / p.d;
    p.nu_d = p.nu / p.d;
    p.ffs_rho0 = p.ffs / p.rho0;
    p.q_d = make_den(p.d);
    p.q_dd = make_den(p.d * p.d);
    p.q_rho0 = make_den(p.rho0);
    const bool ok = p.d > DEN_MIN && p.d < DEN_MAX && p.rho0 > DEN_MIN && p.rho0 < DEN_MAX;
    p.exp_lim = ok ? ExpCheck::LIMIT : -1;  // -1: IEEE divisions throughout
}
__host__ __device__ inline void time_constants(FusedParams &p)
{
    p.q_tau = make_den(p.tau);
    p.q_dn = make_den(p.dn);
    const bool ok = p.tau > DEN_MIN && p.tau < DEN_MAX && p.dn > DEN_MIN && p.dn < DEN_MAX;
    p.exp_lim = ok ? p.exp_lim : -1;
}

// A wave-uniform value of a table that no kernel writes, by the scalar unit:
// into scalar registers (the compiler cannot tell by itself that the kernel's
// stores leave the table alone).
template <class T>
__device__ __forceinline__ T scalar_load(const T *p)
{
    typedef const T __attribute__((address_space(4))) * ConstPtr;
    return *(ConstPtr)(uintptr_t)p;
}

// Lane shifts by DPP (no LDS traffic).  wave_shl:1 gives lane L the value
// of lane L+1 (column m+1), wave_shr:1 the value of lane L-1 (column m-1);
// the lanes at the wave's ends receive 0 and only ever feed halo lanes.
__device__ __forceinline__ int dpp_from_right(int x)
{
    return __builtin_amdgcn_update_dpp(0, x, 0x130, 0xF, 0xF, true);
}
__device__ __forceinline__ int dpp_from_left(int x)
{
    return __builtin_amdgcn_update_dpp(0, x, 0x138, 0xF, 0xF, true);
}
__device__ __forceinline__ double xr(double x)  // value of column m+1
{
    return __hiloint2double(dpp_from_right(__double2hiint(x)), dpp_from_right(__double2loint(x)));
}
__device__ __forceinline__ double xl(double x)  // value of column m-1
{
    return __hiloint2double(dpp_from_left(__double2hiint(x)), dpp_from_left(__double2loint(x)));
}
__device__ __forceinline__ float xr(float x) { return __int_as_float(dpp_from_right(__float_as_int(x))); }
__device__ __forceinline__ int xr(int x) { return dpp_from_right(x); }
__device__ __forceinline__ float xl(float x) { return __int_as_float(dpp_from_left(__float_as_int(x))); }

// Stores of the step's outputs.  Measured on MI355X at 2048 x 1536 (us per
// launch, FP64 / FP32 / 64-member FP32 ensemble): all cached 100.0 / 71.5 /
// 577; non-temporal level-n and filtered-level stores in FP64, filtered-level
// stores in FP32 (FP64 arrays), frozen forcing cached: 94.4 / 66.5 / 572.
// Non-temporal FP32 level-n stores (69.0 / 612 FP32 / ensemble) and
// non-temporal loads of the filtered level (74.3 / 603) are slower.
template <bool NT, class T>
__device__ __forceinline__ void st_out(void *base, size_t i, T v)
{
    T *q = static_cast<T *>(base) + i;
    if constexpr (NT)
        __builtin_nontemporal_store(v, q);
    else
        *q = v;
}

template <class R>
__device__ __forceinline__ R bitf(int mb, int bit)
{
    return (mb & bit) ? R(1) : R(0);
}

// Loads are branch-free: the address is clamped into the array and the
// value is zeroed afterwards when the cell lies outside it.  Straight-line
// loads let the compiler wait for exactly the older (prefetched) loads.
struct RowAddr {
    int nx, ny, mc;  // mc = column clamped to 1..nx
    __device__ __forceinline__ size_t at(int row) const
    {
        const int rc = min(max(row, 1), ny);
        return (size_t)(rc - 1) * nx + (mc - 1);
    }
};

// Rows per wave when the caller does not choose one, for a grid of `rows`
// rows cut into `strips` strips on a chip that holds `slots` waves of the
// kernel at once.  An item marches its chunk plus `warm` warm-up rows, and
// the launch takes as many rounds as it has items per slot, so the time
// goes as rounds x (chunk + warm): pick the number of rounds k (1..8) that
// minimises it, with the chunk that fits k rounds exactly.  Measured on
// MI355X at 2048 x 1536 (1024 SIMDs): one item more than a round costs up to
// 40 % (two substeps per launch in FP32: 28 rows, 1980 items in 2048 slots,
// 54 us per substep; 27 rows, 2088 items, 77 us).  Items keep at least `lo`
// rows (512 x 384, one substep per launch: 2 rows 8.7 us, 1 row 10.5 us).
inline int fit_chunk(int rows, int strips, long long slots, int warm, int lo)
{
    int best = rows;
    long long best_cost = -1;
    for (int k = 1; k <= 8; ++k) {
        const long long per = (long long)k * slots / strips;  // chunks per strip that fit k rounds
        if (per < 1) continue;
        int chunk = (int)((rows + per - 1) / per);
        if (chunk < lo) chunk = lo;
        const long long items = (long long)strips * ((rows + chunk - 1) / chunk);
        const long long rounds = (items + slots - 1) / slots;
        const long long cost = rounds * (chunk + warm);
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            best = chunk;
        }
    }
    return best;
}

// The older rule, kept for the ensemble's persistent launch: the measured
// best for large grids (FP64 32, FP32 20 rows), fewer when the work items
// (strips x row chunks) would not give the chip about 4 per CU.
inline int auto_chunk(bool fp32, long long strip_rows)
{
    const long long big = fp32 ? 20 : 32;
    const long long c = strip_rows / 1024;
    return (int)(c < 4 ? 4 : c > big ? big : c);
}

// What one substep consumes at iteration n of its march (the mask bits zeroed
// outside the array): surface height, depth at rest and mask bits of row
// n+2; level-n velocity, filtered level and Rayleigh coefficient of row
// n+1; the frozen forcing and carried U/V depths of row n; the row tables.
template <typename R>
struct StageIn {
    R s2, H2;
    int mb2;
    R u1, v1, rd1;
    double up1, vp1, sp1;
    R fx0, fy0;
    double hupc0, hvpc0;
    R f0, sx0, sy0, wf1;
};

// What one substep produces for output row n: the new level-n fields and
// filtered level after the Robert-Asselin shift, the forcing it used
// (formed at the call's first substep, frozen afterwards) and, in
// FP64_EXACT, the hh_shift-filtered U/V depths for the next substep.
template <typename R>
struct StageOut {
    R s, u, v;
    double sp, up, vp;
    R rhs_u, rhs_v;
    double hu, hv;
};

// 1 / n of a depth average over n = 1, 2 or 4 cells, whose product is the
// quotient (n = 0: not a number, as 0 / 0)
__device__ __forceinline__ double inv_cells(int n)
{
    return n == 4 ? 0.25 : n == 2 ? 0.5 : n == 0 ? __builtin_inf() : 1.0;
}
// sum / n for n of 4 cells; the division by 3 only in a wave that has one
__device__ __forceinline__ double mean_cells(double sum, int n)
{
    double mean = sum * inv_cells(n);
    if (__any(n == 3)) mean = n == 3 ? sum / 3.0 : mean;
    return mean;
}

// One leap-frog substep of FP64_EXACT marching down the rows of one strip: the
// rolling register window (suffix m1 = row n-1, 0 = row n, p1 = n+1, p2 = n+2)
// of input rows and of T-, U-, V- and H-point terms.  row(n) takes the inputs
// of iteration n and, when asked, computes the outputs of row n.  FORM: the
// call's first substep, which forms the wind + drag forcing; the later
// substeps take it frozen (StageIn::fx0, fy0).
//
// The results are the reference's expressions operation by operation.  Bound
// by its FP64 operations, of which IEEE divisions were two thirds, so:
//  - terms that neighbours use (the cell volumes w of the depth averages, the
//    fluxes, the stress terms, a velocity's quotient by d) are formed once and
//    shifted; a sum of two is the same in either order;
//  - d / d is 1, and a quotient by 1, 2 or 4 a product, exactly;
//  - the quotients by d, d * d, tau, dn and rho0 take quots (bt_exactdiv.h),
//    groups of them after one look at their numerators' exponents;
//  - the quotient by 3 of a depth average of three cells is formed where a
//    lane of the wave has one;
//  - un and vn, by a depth, stay IEEE divisions.
// Measured on MI355X, us per substep before / after: 1021 x 763 43.5 / 34.6,
// 2048 x 1536 154 / 118, where its traffic (about 160 bytes a cell: 103 us at
// the copy rate of 4.9 TB/s) bounds it instead.
template <bool FORM>
struct ExactStage {
    const FusedParams &p;
    const bool inx, inx1;

    double u_0 = 0, u_p1 = 0, v_0 = 0, v_p1 = 0;
    double s_0 = 0, s_p1 = 0, s_p2 = 0, H_p1 = 0, H_p2 = 0;
    double up_0 = 0, up_p1 = 0, vp_0 = 0, vp_p1 = 0, sp_0 = 0, sp_p1 = 0;
    double rd_0 = 0, rd_p1 = 0;
    int mb_0 = 0, mb_p1 = 0, mb_p2 = 0;
    // cell volumes ((q * d) * d) * lu of the levels n, n-1 and n+1, and w + its
    // right neighbour's
    double w_p1 = 0, w_p2 = 0, su_0 = 0, su_p1 = 0, wp_0 = 0, wn_0 = 0;
    int lus_0 = 0, lus_p1 = 0, lu_p1 = 0, lu_p2 = 0;  // lu, lu + its right neighbour's
    double hq_p1 = 0, hq_p2 = 0;
    double hu_0 = 0, hu_p1 = 0, hup_0 = 0, hv_0 = 0, hv_p1 = 0;
    double sn_0 = 0, hun_0 = 0;
    double qu_0 = 0, qv_0 = 0;            // up / d, vp / d
    double V_0 = 0, Q_0 = 0;              // v hv d, v d d hv
    double A_0 = 0, B_0 = 0;              // u d hu, v d hv
    double T_0 = 0, S_m1 = 0;             // d d mu hq stt, d d muh hh sts
    double fy_m1 = 0, gy_m1 = 0;          // momentum fluxes through the row's south faces
    double C_m1 = 0, E_m1 = 0;            // vorticity and Coriolis terms of the H point south
    double bf_0 = 0;
    int slow = 0;                         // rows for which the depths take IEEE divisions

    __device__ ExactStage(const FusedParams &pp, int m)
        : p(pp), inx(m >= 3 && m <= pp.nx - 2), inx1(m >= 2 && m <= pp.nx - 1)
    {
    }

    __device__ __forceinline__ void row(int n, const StageIn<double> &q, bool produce, StageOut<double> &o)
    {
        const double d = p.d, tau = p.tau, nu = p.nu;
        const int k1 = n + 1;
        s_p2 = q.s2;
        H_p2 = q.H2;
        mb_p2 = q.mb2;
        u_p1 = q.u1;
        v_p1 = q.v1;
        up_p1 = q.up1;
        vp_p1 = q.vp1;
        sp_p1 = q.sp1;
        rd_p1 = q.rd1;
        const double f_0 = q.f0;
        const bool iny1 = (k1 >= 3 && k1 <= p.ny - 2);
        const bool tw = (mb_p1 & MB_LU) && inx && iny1;

        // ---- depths (hh_init / hh_update, Function/depth.f90)
        lu_p2 = mb_p2 & MB_LU ? 1 : 0;
        lus_p1 = lu_p1 + xr(lu_p1);
        const int lu_0 = mb_0 & MB_LU ? 1 : 0;
        const double lf_p1 = lu_p1, lf_p2 = lu_p2;
        hq_p2 = H_p2 + s_p2;
        w_p2 = ((hq_p2 * d) * d) * lf_p2;
        su_p1 = w_p1 + xr(w_p1);
        const double wp_p1 = (((H_p1 + sp_p1) * d) * d) * lf_p1;
        double hup_p1 = 0.0, hvp_0 = 0.0, hh_0;
        {
            ExpCheck ck;
            ck.add(w_p2);
            if (FORM) ck.add(wp_p1);
            slow = ck.any(p.exp_lim) ? 4 : slow - 1;
            const int nh = lus_0 + lus_p1;
            const double mean4 = mean_cells((su_0 + w_p1) + xr(w_p1), nh);
            double a[3] = {su_p1 * inv_cells(lus_p1), (w_p1 + w_p2) * inv_cells(lu_p1 + lu_p2), mean4};
            quots2(a, p.q_d, slow > 0);
            hu_p1 = (mb_p1 & MB_LLU) ? a[0] : 0.0;
            hv_p1 = (mb_p1 & MB_LLV) ? a[1] : 0.0;
            hh_0 = (mb_0 & MB_LUH) ? a[2] : 0.0;
            if constexpr (FORM) {
                double b[2] = {(wp_p1 + xr(wp_p1)) * inv_cells(lus_p1), (wp_0 + wp_p1) * inv_cells(lu_0 + lu_p1)};
                quots2(b, p.q_d, slow > 0);
                hup_p1 = (mb_p1 & MB_LLU) ? b[0] : 0.0;
                hvp_0 = (mb_0 & MB_LLV) ? b[1] : 0.0;
            }
        }

        // ---- T-point stage of row n+1: continuity, new depths, tension, drag
        const double U_p1 = u_p1 * hu_p1 * d, V_p1 = v_p1 * hv_p1 * d;
        const double div = U_p1 - xl(U_p1) + V_p1 - V_0;
        double qc[1] = {div}, qw[1] = {q.wf1}, quv[2] = {up_p1, vp_p1};
        {
            ExpCheck ck;
            ck.add(div);
            ck.add(q.wf1);
            ck.add(up_p1);
            ck.add(vp_p1);
            const bool ieee = ck.any(p.exp_lim);
            quots(qc, p.q_dd, ieee);
            quots(qw, p.q_rho0, ieee);
            quots(quv, p.q_d, ieee);
        }
        const double sn = sp_p1 + 2.0 * tau * (qw[0] * p.ffs - qc[0]);
        const double sn_p1 = tw ? sn : 0.0;
        const double wn_p1 = (((H_p1 + sn_p1) * d) * d) * lf_p1;
        double hun_p1, hvn_0;
        {
            ExpCheck ck;
            ck.add(wn_p1);
            if (ck.any(p.exp_lim)) slow = 4;
            double a[2] = {(wn_p1 + xr(wn_p1)) * inv_cells(lus_p1), (wn_0 + wn_p1) * inv_cells(lu_0 + lu_p1)};
            quots2(a, p.q_d, slow > 0);
            hun_p1 = (mb_p1 & MB_LLU) ? a[0] : 0.0;
            hvn_0 = (mb_0 & MB_LLV) ? a[1] : 0.0;
        }
        const double qu_p1 = quv[0], qv_p1 = quv[1];
        const double qu1l = xl(qu_p1), qv0r = xr(qv_0);  // lane shifts, outside any branch
        const double stt_p1 = tw ? (qu_p1 - qu1l) - (qv_p1 - qv_0) : 0.0;
        double bf_p1 = 0.0, Q_p1 = 0.0;
        if constexpr (FORM) {
            const double P_p1 = u_p1 * d * d * hu_p1;
            Q_p1 = v_p1 * d * d * hv_p1;
            double a[2] = {(P_p1 + xl(P_p1)) / 2.0, (Q_p1 + Q_0) / 2.0};
            ExpCheck ck;
            ck.add(a[0]);
            ck.add(a[1]);
            quots2(a, p.q_d, ck.any(p.exp_lim));
            const double ut = a[0] / hq_p1, vt = a[1] / hq_p1;
            const double bf = p.cb * sqrt(ut * ut + vt * vt + p.eb);
            bf_p1 = tw ? bf : 0.0;
        }

        // ---- H-point stage of row n: shear, metric vorticity, Coriolis
        const double v0r = xr(v_0);
        const bool hw = (mb_0 & MB_LUU) && inx && (n >= 3 && n <= p.ny - 2);
        const double sts_0 = hw ? (qu_p1 - qu_0) + (qv0r - qv_0) : 0.0;
        const double vo = (v0r * d - v_0 * d) - (u_p1 * d - u_0 * d) - ((v0r - v_0) * d - (u_p1 - u_0) * d);
        const double vh = (hw ? vo : 0.0) * hh_0;
        const double fh = f_0 * hh_0 * d * d;
        const double C_0 = vh * (v0r + v_0), D_0 = vh * (u_p1 + u_0);
        const double E_0 = fh * (v0r + v_0), F_0 = fh * (u_p1 + u_0);
        // viscosity: mu at T points, its mean at the H point
        const double mu_0 = lu_0 * nu, mu_p1 = lf_p1 * nu;
        const double muh = (mu_0 + xr(mu_0) + mu_p1 + xr(mu_p1)) / 4.0;
        const double T_p1 = d * d * mu_p1 * hq_p1 * stt_p1, S_0 = d * d * muh * hh_0 * sts_0;
        // momentum fluxes (uv_trans, vel_ssh.f90:59-105)
        const double A_p1 = u_p1 * d * hu_p1, B_p1 = v_p1 * d * hv_p1;
        const double B0r = xr(B_0), luu0 = mb_0 & MB_LUU ? 1.0 : 0.0;
        const double fy_0 = (B_0 + B0r) / 2.0 * (u_p1 + u_0) / 2.0 * luu0;
        const double gy_0 = (B_0 + B_p1) / 2.0 * (v_0 + v_p1) / 2.0;

        // ---- outputs of row n
        if (produce) {
            const bool iny = (n >= 3 && n <= p.ny - 2);
            const double bf0r = xr(bf_0), s0r = xr(s_0), rd0r = xr(rd_0);
            // the RHS of Control/dyncall.f90:114-126 is formed once per call
            // (first substep) and frozen over the call's substeps
            double rhs_u = q.fx0, rhs_v = q.fy0;
            if constexpr (FORM) {
                rhs_u = 0.0 + (q.sx0 + (-(bf_0 + bf0r) / 2.0 * up_0)) * d * d;
                rhs_v = 0.0 + (q.sy0 + (-(bf_0 + bf_p1) / 2.0 * vp_0)) * d * d;
            }
            o.rhs_u = rhs_u;
            o.rhs_v = rhs_v;
            // level n-1 U/V depths: hh_init values at the first substep,
            // the hh_shift-filtered carry afterwards (depth.f90:195-203)
            const double hupc = FORM ? hup_0 : q.hupc0, hvpc = FORM ? hvp_0 : q.hvpc0;
            const double T0r = xr(T_0), S0l = xl(S_0), F0l = xl(F_0), D0l = xl(D_0);
            double a[4] = {T0r - T_0, S_0 - S_m1, T_p1 - T_0, S_0 - S0l};
            double b[4] = {hun_0 * d * d / 2.0, hupc * d * d / 2.0, hvn_0 * d * d / 2.0, hvpc * d * d / 2.0};
            {
                ExpCheck ck;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    ck.add(a[k]);
                    ck.add(b[k]);
                }
                const bool ieee = ck.any(p.exp_lim);
                quots(a, p.q_d, ieee);
                quots(b, p.q_tau, ieee);
            }
            // zonal momentum (vel_ssh.f90:536-551) with uv_trans (:59-81) and uv_diff2 (:146-159)
            double un, vn;
            {
                const double fx_p = (A_0 + xr(A_0)) / 2.0 * (u_0 + xr(u_0)) / 2.0, fx_m = xl(fx_p);
                const double radv = -(fx_p - fx_m + fy_0 - fy_m1) + (C_0 + C_m1) / 4.0;
                const double rdfx = a[0] + a[1];
                const double slx = -p.g * (s0r - s_0) * d * hu_0;
                const double grx =
                    rhs_u + slx + rdfx + radv - (rd_0 + rd0r) / 2.0 * up_0 * d * d * hu_0 + (E_0 + E_m1) / 4.0;
                un = (up_0 * b[1] + grx) / b[0];
            }
            // meridional momentum (vel_ssh.f90:554-569) with uv_trans (:84-105) and uv_diff2 (:162-175)
            {
                const double gx_p = (A_0 + A_p1) / 2.0 * (v0r + v_0) / 2.0, gx_m = xl(gx_p);
                const double rady = -(gx_p - gx_m + gy_0 - gy_m1) - (D_0 + D0l) / 4.0;
                const double rdfy = -a[2] + a[3];
                const double sly = -p.g * (s_p1 - s_0) * d * hv_0;
                const double gry =
                    rhs_v + sly + rdfy + rady - (rd_0 + rd_p1) / 2.0 * vp_0 * d * d * hv_0 - (F_0 + F0l) / 4.0;
                vn = (vp_0 * b[3] + gry) / b[2];
            }
            un = ((mb_0 & MB_LCU) && inx && iny) ? un : 0.0;
            vn = ((mb_0 & MB_LCV) && inx && iny) ? vn : 0.0;

            // time-level shift with the Robert-Asselin filter (vel_ssh.f90:588-612),
            // and hh_shift of the U/V depths for the next substep (depth.f90:195-203)
            const double ts = p.ts;
            double e[5] = {ts * (sn_0 - 2.0 * s_0 + sp_0) / 2.0, ts * (un - 2.0 * u_0 + up_0) / 2.0,
                           ts * (vn - 2.0 * v_0 + vp_0) / 2.0, ts * (hun_0 - 2.0 * hu_0 + hupc) / 2.0,
                           ts * (hvn_0 - 2.0 * hv_0 + hvpc) / 2.0};
            {
                ExpCheck ck;
#pragma unroll
                for (int k = 0; k < 5; ++k) ck.add(e[k]);
                quots(e, p.q_dn, ck.any(p.exp_lim));
            }
            const bool sh = inx1 && n >= 2 && n <= p.ny - 1;
            const bool su = sh && (mb_0 & MB_LU), uu = sh && (mb_0 & MB_LCU), vv = sh && (mb_0 & MB_LCV);
            o.s = su ? sn_0 : s_0;
            o.u = uu ? un : u_0;
            o.v = vv ? vn : v_0;
            o.sp = su ? s_0 + e[0] : sp_0;
            o.up = uu ? u_0 + e[1] : up_0;
            o.vp = vv ? v_0 + e[2] : vp_0;
            o.hu = sh && (mb_0 & MB_LLU) ? hu_0 + e[3] : hupc;
            o.hv = sh && (mb_0 & MB_LLV) ? hv_0 + e[4] : hvpc;
        }

        // ---- advance the window one row
        u_0 = u_p1; v_0 = v_p1;
        s_0 = s_p1; s_p1 = s_p2;
        H_p1 = H_p2;
        up_0 = up_p1; vp_0 = vp_p1; sp_0 = sp_p1; rd_0 = rd_p1;
        mb_0 = mb_p1; mb_p1 = mb_p2;
        lu_p1 = lu_p2; lus_0 = lus_p1;
        w_p1 = w_p2; su_0 = su_p1; wp_0 = wp_p1; wn_0 = wn_p1;
        hq_p1 = hq_p2;
        hu_0 = hu_p1; hup_0 = hup_p1; hv_0 = hv_p1;
        sn_0 = sn_p1; hun_0 = hun_p1;
        qu_0 = qu_p1; qv_0 = qv_p1;
        V_0 = V_p1; Q_0 = Q_p1; A_0 = A_p1; B_0 = B_p1;
        T_0 = T_p1; S_m1 = S_0; fy_m1 = fy_0; gy_m1 = gy_0; C_m1 = C_0; E_m1 = E_0;
        bf_0 = bf_p1;
    }
};

// Explicit multiply-adds of the fast modes: the library is compiled without
// contraction, so the march, the pair march, the pipeline and the tiles give
// the same bits whatever the compiler does around them.
__device__ __forceinline__ double fmad(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fmad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// a / b for a layer depth b (about 1 .. 10^4, far from the limits of the
// format, so nothing is scaled or fixed up: an infinite numerator or a depth
// of zero gives NaN): the hardware's reciprocal (FP32: 1 ulp; FP64: about
// 2^-26, two Newton steps) and one correction of the quotient by its exact
// remainder.  The IEEE quotient in both formats on each of 2^30 random pairs,
// depths 1 .. 2^14 and numerators 2^-30 .. 2^15.
__device__ __forceinline__ float depth_div(float a, float b)
{
    const float r = __builtin_amdgcn_rcpf(b);
    const float q = a * r;
    return fmad(fmad(-b, q, a), r, q);
}
__device__ __forceinline__ double depth_div(double a, double b)
{
    double r = __builtin_amdgcn_rcp(b);
    r = fmad(fmad(-b, r, 1.0), r, r);
    r = fmad(fmad(-b, r, 1.0), r, r);
    const double q = a * r;
    return fmad(fmad(-b, q, a), r, q);
}

// Scalars of the fast modes' formulas.
template <typename R>
struct FastConst {
    R id, two_tau, gid, nuid, ffr, cb, eb, two_tau_id;
    double cts;
    __device__ FastConst(const FusedParams &p)
        : id(R(p.inv_d)), two_tau(R(2.0 * p.tau)), gid(R(p.g_d)), nuid(R(p.nu_d)), ffr(R(p.ffs_rho0)), cb(R(p.cb)),
          eb(R(p.eb)), two_tau_id(R(2.0 * p.tau * p.inv_d)), cts(0.5 * p.ts / p.dn)
    {
    }
};

// The fast modes' formulas (FP64, FP32) on a uniform grid, point by point.
// The reference's algebra with the metric factored out, every flux and
// product formed once where its two neighbours share it: the fluxes u hu and
// v hv, the advective fluxes, the viscous products nu hq str_t and nu hh
// str_s (the mean viscosity of four wet cells is nu), the Coriolis products.
namespace fast {
// 1 / (number of wet T cells) of a U or V point: both wet (`both`) or one
template <typename R>
__device__ __forceinline__ R depth2(R wsum, bool any, bool both)
{
    return any ? (both ? R(0.5) * wsum : wsum) : R(0);
}
// the same on an H point with cnt wet T cells of 4
template <typename R>
__device__ __forceinline__ R depth4(R wsum, int cnt)
{
    const R rs = cnt == 4 ? R(0.25) : cnt == 3 ? R(1.0 / 3.0) : cnt == 2 ? R(0.5) : R(1);
    return cnt > 0 ? rs * wsum : R(0);
}
// continuity (Function/vel_ssh.f90:487-499): the increment of the surface
template <typename R>
__device__ __forceinline__ double surface(const FastConst<R> &c, double sp, R wf, R fu, R ful, R fv, R fvs)
{
    const R div = (fu - ful) + (fv - fvs);
    return sp + double(fmad(-c.two_tau_id, div, c.two_tau * (wf * c.ffr)));
}
// bottom drag rate (Function/fluxes.f90:226-250)
template <typename R>
__device__ __forceinline__ R drag(const FastConst<R> &c, R hq, R fu, R ful, R fv, R fvs)
{
    const R rh = depth_div(R(0.5), hq);
    const R ut = (fu + ful) * rh, vt = (fv + fvs) * rh;
    return c.cb * sqrt(fmad(ut, ut, fmad(vt, vt, c.eb)));
}
// new velocity of a U (V) point (Function/vel_ssh.f90:531-573): rhs the
// frozen forcing, ds the surface difference, h, hp, hn the depth at levels
// n, n-1, n+1, adv the sum of the four advective fluxes (times -4), dif the
// viscous differences, rds the two Rayleigh coefficients, cor the signed sum
// of the two Coriolis products, up the filtered velocity.  up hp is by far the
// larger of the two terms of the numerator: the multiply-add keeps it exact
// and rounds the small one (rounded by itself first, it moved the FP64 mode's
// states 4 to 6 % further from extended-precision ones).
template <typename R>
__device__ __forceinline__ R momentum(const FastConst<R> &c, R rhs, R ds, R h, R hp, R hn, R adv, R dif, R rds,
                                      R cor, R up)
{
    R F = fmad(c.id, fmad(R(-0.25), adv, dif), rhs);
    F = fmad(-c.gid * ds, h, F);
    F = fmad(R(-0.5) * rds * up, h, F);
    F = fmad(R(0.25), cor, F);
    return depth_div(fmad(up, hp, c.two_tau * F), hn);
}
// Robert-Asselin filter (Function/vel_ssh.f90:588-612), in FP64
__device__ __forceinline__ double filter(double cts, double now, double next, double prev)
{
    return fmad(cts, fmad(-2.0, now, next) + prev, now);
}
}  // namespace fast

// One leap-frog substep marching down the rows of one strip in the fast
// modes.  Cells outside the array enter with mask 0, and every use of a
// neighbour is selected by a mask, so their values do not matter (they need
// not be zeroed).  Lane shifts stand outside the selections: inside an arm
// they would read lanes that the arm's branch has switched off.
template <typename R, bool FORM>
struct FastStage {
    const FusedParams &p;
    const FastConst<R> c;
    const bool inx, inx1;

    R u_0 = 0, v_0 = 0, s_0 = 0, s_p1 = 0, H_p1 = 0, rd_0 = 0;
    double up_0 = 0, vp_0 = 0, sp_0 = 0;
    int mb_0 = 0, mb_p1 = 0;
    int lus_0 = 0;                         // wet T cells of (m, n), (m+1, n)
    bool lv_0 = false;                     // (m, n) and (m, n+1) both wet
    R w_p1 = 0, a_0 = 0;                   // wet depth of row n+1; sum over m, m+1 of row n
    R wp_0 = 0, wn_0 = 0;                  // wet depth of the filtered and the new level
    R hu_0 = 0, hup_0 = 0, hv_0 = 0, hun_0 = 0;
    R fu_0 = 0, fv_0 = 0;                  // u hu, v hv
    R fyU_m1 = 0, fyV_m1 = 0;              // advective fluxes through the south faces
    R Q_m1 = 0, Fc_m1 = 0, P_0 = 0, bf_0 = 0;
    double sn_0 = 0;

    __device__ FastStage(const FusedParams &pp, int m)
        : p(pp), c(pp), inx(m >= 3 && m <= pp.nx - 2), inx1(m >= 2 && m <= pp.nx - 1)
    {
    }

    __device__ __forceinline__ void row(int n, const StageIn<R> &q, bool produce, StageOut<R> &o)
    {
        const int k1 = n + 1;
        const bool tw = (mb_p1 & MB_LU) && inx && (k1 >= 3 && k1 <= p.ny - 2);
        const bool hw = (mb_0 & MB_LUU) && inx && (n >= 3 && n <= p.ny - 2);
        const int l1 = mb_p1 & MB_LU;
        const int lus_p1 = l1 + dpp_from_right(l1);
        const bool lu1 = l1 != 0, lv_p1 = (mb_p1 & q.mb2 & MB_LU) != 0;
        const bool llu1 = mb_p1 & MB_LLU, lu2 = lus_p1 == 2;
        const bool llv0 = mb_0 & MB_LLV, lcv0 = mb_0 & MB_LCV;
        const R up1 = R(q.up1), vp1 = R(q.vp1), up0 = R(up_0), vp0 = R(vp_0);

        // ---- depths (hh_init / hh_update, Function/depth.f90)
        const R w_p2 = (q.mb2 & MB_LU) ? q.H2 + q.s2 : R(0);
        const R a_p1 = w_p1 + xr(w_p1);
        const R hu_p1 = fast::depth2(a_p1, llu1, lu2);
        const R hv_p1 = fast::depth2(w_p1 + w_p2, bool(mb_p1 & MB_LLV), lv_p1);
        const R hh_0 = fast::depth4(a_0 + a_p1, (mb_0 & MB_LUH) ? lus_0 + lus_p1 : 0);
        const R wp_p1 = lu1 ? H_p1 + R(q.sp1) : R(0);
        const R hup_p1 = fast::depth2(wp_p1 + xr(wp_p1), llu1, lu2);

        // ---- T point of row n+1: continuity, new depths, tension, drag
        const R fu_p1 = q.u1 * hu_p1, fv_p1 = q.v1 * hv_p1;
        const R ful = xl(fu_p1);
        const double sn_p1 = tw ? fast::surface(c, q.sp1, q.wf1, fu_p1, ful, fv_p1, fv_0) : 0.0;
        const R wn_p1 = lu1 ? H_p1 + R(sn_p1) : R(0);
        const R hun_p1 = fast::depth2(wn_p1 + xr(wn_p1), llu1, lu2);
        const R tens = (up1 - xl(up1)) - (vp1 - vp0);
        const R P_p1 = tw ? c.nuid * w_p1 * tens : R(0);
        R bf_p1 = R(0);
        if constexpr (FORM) bf_p1 = tw ? fast::drag(c, w_p1, fu_p1, ful, fv_p1, fv_0) : R(0);

        // ---- H point of row n: shear, Coriolis (the metric vorticity is
        // identically zero for uniform metrics, Function/vel_ssh.f90:35-37)
        const R shear = (up1 - up0) + (xr(vp0) - vp0);
        const R Q_0 = hw ? c.nuid * hh_0 * shear : R(0);
        const R vsum = xr(v_0) + v_0, usum = q.u1 + u_0;
        const R cor = q.f0 * hh_0;
        const R Fc_0 = cor * vsum;
        const R fvs = fv_0 + xr(fv_0);
        const R fyU_0 = (mb_0 & MB_LUU) ? fvs * usum : R(0);
        const R fyV_0 = (fv_0 + fv_p1) * (v_0 + q.v1);

        // ---- outputs of row n
        if (produce) {
            R rhs_u = q.fx0, rhs_v = q.fy0;
            if constexpr (FORM) {
                // the RHS of Control/dyncall.f90:114-126, frozen over the call's substeps
                rhs_u = fmad(R(-0.5) * (bf_0 + xr(bf_0)), up0, q.sx0);
                rhs_v = fmad(R(-0.5) * (bf_0 + bf_p1), vp0, q.sy0);
            }
            o.rhs_u = rhs_u;
            o.rhs_v = rhs_v;
            const R hvp_0 = fast::depth2(wp_0 + wp_p1, llv0, lv_0);
            const R hvn_0 = fast::depth2(wn_0 + wn_p1, llv0, lv_0);
            const R fx = (fu_0 + xr(fu_0)) * (u_0 + xr(u_0));
            const R gx = (fu_0 + fu_p1) * vsum;
            const R Gc = cor * usum;
            R un = fast::momentum(c, rhs_u, xr(s_0) - s_0, hu_0, hup_0, hun_0, (fx - xl(fx)) + (fyU_0 - fyU_m1),
                                  (xr(P_0) - P_0) + (Q_0 - Q_m1), rd_0 + xr(rd_0), Fc_0 + Fc_m1, up0);
            R vn = fast::momentum(c, rhs_v, s_p1 - s_0, hv_0, hvp_0, hvn_0, (gx - xl(gx)) + (fyV_0 - fyV_m1),
                                  (P_0 - P_p1) + (Q_0 - xl(Q_0)), rd_0 + q.rd1, -(Gc + xl(Gc)), vp0);
            const bool iny = (n >= 3 && n <= p.ny - 2);
            un = ((mb_0 & MB_LCU) && inx && iny) ? un : R(0);
            vn = (lcv0 && inx && iny) ? vn : R(0);

            // time-level shift with the Robert-Asselin filter
            const bool sh = inx1 && n >= 2 && n <= p.ny - 1;
            const bool su = (mb_0 & MB_LCU) && sh, sv = lcv0 && sh, ss = (mb_0 & MB_LU) && sh;
            o.s = ss ? R(sn_0) : s_0;
            o.u = su ? un : u_0;
            o.v = sv ? vn : v_0;
            o.sp = ss ? fast::filter(c.cts, double(s_0), sn_0, sp_0) : sp_0;
            o.up = su ? fast::filter(c.cts, double(u_0), double(un), up_0) : up_0;
            o.vp = sv ? fast::filter(c.cts, double(v_0), double(vn), vp_0) : vp_0;
        }

        // ---- advance the window one row
        u_0 = q.u1; v_0 = q.v1;
        s_0 = s_p1; s_p1 = q.s2;
        H_p1 = q.H2;
        up_0 = q.up1; vp_0 = q.vp1; sp_0 = q.sp1; rd_0 = q.rd1;
        mb_0 = mb_p1; mb_p1 = q.mb2;
        lus_0 = lus_p1; lv_0 = lv_p1;
        w_p1 = w_p2; a_0 = a_p1;
        wp_0 = wp_p1; wn_0 = wn_p1;
        hu_0 = hu_p1; hup_0 = hup_p1; hv_0 = hv_p1; hun_0 = hun_p1;
        fu_0 = fu_p1; fv_0 = fv_p1;
        fyU_m1 = fyU_0; fyV_m1 = fyV_0;
        Q_m1 = Q_0; Fc_m1 = Fc_0; P_0 = P_p1; bf_0 = bf_p1;
        sn_0 = sn_p1;
    }
};

// the march of a mode
template <typename R, bool EXACT, bool FORM>
using MarchStage = std::conditional_t<EXACT, ExactStage<FORM>, FastStage<R, FORM>>;

// Loads of one iteration n of a strip (issued one iteration ahead of their
// use: measured on MI355X at 2048 x 1536, two iterations ahead runs 5 %
// slower in FP32 and halves FP64's occupancy).
// A row is the same for the whole wave, so its address is formed by the scalar
// unit and a lane adds its constant column (the loads of an iteration took 47
// vector operations for their addresses, now none; 2048 x 1536, us per substep:
// FP32 35.2 -> 33.4, FP64 48.0 -> 47.7, FP64_EXACT 122 -> 118).  Rows and columns
// outside the array are clamped into it and their mask bits zeroed: the stages
// select by them, and no value outside the array reaches an output.
template <typename R, bool EXACT, bool FROZEN>
struct Loader {
    const FusedParams &p;
    const uint32_t col;  // the lane's column, clamped, from 0
    const bool colok;
    struct Pre {
        R s, H, u, v, rd, fx, fy;
        double up, vp, sp, hupc, hvpc, f, sx, sy, wf;
        int mb;
    } q;

    __device__ Loader(const FusedParams &pp, int m)
        : p(pp), col(min(max(m, 1), pp.nx) - 1), colok(m >= 1 && m <= pp.nx)
    {
    }
    __device__ __forceinline__ double tab(const double *t, int row) const
    {
        return scalar_load(t + (min(max(row, 1), p.ny) - 1));
    }
    // the lane's element of the row that starts at element `row` of the array
    template <class T>
    __device__ __forceinline__ T at(const T *base, size_t row) const
    {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base + row) + (uint32_t)(col * sizeof(T)));
    }
    __device__ __forceinline__ void issue(int n)  // the loads iteration n consumes
    {
        const R *S = static_cast<const R *>(p.s), *Hh = static_cast<const R *>(p.H);
        const R *U = static_cast<const R *>(p.u), *V = static_cast<const R *>(p.v);
        const R *RD = static_cast<const R *>(p.rd);
        const R *FX = static_cast<const R *>(p.frx_in), *FY = static_cast<const R *>(p.fry_in);
        auto row = [&](int r) { return (size_t)(min(max(r, 1), p.ny) - 1) * (size_t)p.nx; };
        const size_t r2 = row(n + 2), r1 = row(n + 1), r0 = row(n);
        q.s = at(S, r2);
        q.H = at(Hh, r2);
        q.mb = at(p.mb, r2);
        q.u = at(U, r1);
        q.v = at(V, r1);
        q.up = at(p.up, r1);
        q.vp = at(p.vp, r1);
        q.sp = at(p.sp, r1);
        q.rd = at(RD, r1);
        // per-cell frozen forcing and carried depths of the output row n
        if constexpr (FROZEN) {
            q.fx = at(FX, r0);
            q.fy = at(FY, r0);
        } else {
            q.fx = q.fy = R(0);
        }
        if constexpr (EXACT && FROZEN) {
            q.hupc = at(p.hup_in, r0);
            q.hvpc = at(p.hvp_in, r0);
        } else {
            q.hupc = q.hvpc = 0.0;
        }
        q.f = tab(p.row_f, n);
        q.sx = tab(p.row_sx, n);
        q.sy = tab(p.row_sy, n);
        q.wf = tab(p.row_wf, n + 1);
    }
    // the prefetched values of iteration n
    __device__ __forceinline__ void take(int n, StageIn<R> &in) const
    {
        in.s2 = q.s;
        in.H2 = q.H;
        in.mb2 = colok && n + 2 >= 1 && n + 2 <= p.ny ? q.mb : 0;
        in.u1 = q.u;
        in.v1 = q.v;
        in.up1 = q.up;
        in.vp1 = q.vp;
        in.sp1 = q.sp;
        in.rd1 = q.rd;
        in.fx0 = q.fx;
        in.fy0 = q.fy;
        in.hupc0 = q.hupc;
        in.hvpc0 = q.hvpc;
        in.f0 = R(q.f);
        in.sx0 = R(q.sx);
        in.sy0 = R(q.sy);
        in.wf1 = R(q.wf);
    }
};

// Store policy (measured, see st_out): level-n outputs non-temporal in the
// FP64 modes, the FP64 filtered level non-temporal in every mode.
template <typename R>
__device__ __forceinline__ void store_state(const FusedParams &p, size_t i, const StageOut<R> &o)
{
    constexpr bool NTS = sizeof(R) == 8;
    st_out<NTS, R>(p.so, i, o.s);
    st_out<NTS, R>(p.uo, i, o.u);
    st_out<NTS, R>(p.vo, i, o.v);
    st_out<true, double>(p.spo, i, o.sp);
    st_out<true, double>(p.upo, i, o.up);
    st_out<true, double>(p.vpo, i, o.vp);
}

// One work item: `chunk` output rows of one 60-column strip of one basin,
// substep p.sub (FORM: p.sub == 1).  Called by every lane of a wave with
// wave-uniform arguments.
template <typename R, bool EXACT, bool FORM>
__device__ __forceinline__ void fused_chunk(const FusedParams &p, int chunk_id, int strip)
{
    const int lane = threadIdx.x;
    const int m = strip * SW + lane - 1;
    const bool colok = (m >= 1 && m <= p.nx);
    const bool writer = colok && lane >= 2 && lane <= SW + 1;
    const int r0 = chunk_id * p.chunk + 1;
    const int r1 = min(r0 + p.chunk, p.ny + 1);

    MarchStage<R, EXACT, FORM> st(p, m);
    Loader<R, EXACT, !FORM> ld(p, m);
    StageIn<R> in;
    StageOut<R> o;
    ld.issue(r0 - 3);
    for (int n = r0 - 3; n < r1; ++n) {
        ld.take(n, in);
        if (n + 1 < r1) ld.issue(n + 1);
        st.row(n, in, n >= r0, o);
        if (n >= r0 && writer && n <= p.ny) {
            const size_t io = (size_t)(n - 1) * p.nx + (m - 1);
            // the forcing formed by the first substep, for the later ones
            if (FORM && p.nsub > 1) {
                st_out<false, R>(p.frx, io, o.rhs_u);
                st_out<false, R>(p.fry, io, o.rhs_v);
            }
            if constexpr (EXACT) {
                if (p.nsub > 1 && p.sub < p.nsub) {
                    st_out<sizeof(R) == 8, double>(p.hup_c, io, o.hu);
                    st_out<sizeof(R) == 8, double>(p.hvp_c, io, o.hv);
                }
            }
            store_state<R>(p, io, o);
        }
    }
}

// Two substeps, p.sub and p.sub + 1, in one march (AFORM: p.sub == 1):
// stage A reads the arrays; stage B runs two rows behind A on A's outputs
// and on the static rows A loaded two iterations earlier (depth at rest,
// mask bits, Rayleigh coefficient), which never leave the registers
// (re-reading them from cache instead was measured 5 % slower).  A strip
// is 58 output columns (B's output at lane L needs
// A's lanes L-1..L+2, which need the loads of L-2..L+4); A starts two rows
// above the chunk so that B's window sees A's rows from r0-2 on.  The
// results are those of two launches of fused_chunk.
template <typename R, bool EXACT, bool AFORM>
__device__ __forceinline__ void fused_chunk2(const FusedParams &p, int chunk_id, int strip)
{
    const int lane = threadIdx.x;
    const int m = strip * SW2 + lane - 1;
    const bool colok = (m >= 1 && m <= p.nx);
    const bool writer = colok && lane >= 2 && lane <= SW2 + 1;
    const int r0 = chunk_id * p.chunk + 1;
    const int r1 = min(r0 + p.chunk, p.ny + 1);
    const int subB = p.sub + 1;

    MarchStage<R, EXACT, AFORM> A(p, m);
    MarchStage<R, EXACT, false> B(p, m);
    Loader<R, EXACT, !AFORM> ld(p, m);
    StageIn<R> ia, ib;
    StageOut<R> oa, ob;
    // delay lines from A's iteration to B's (B's iteration n - 2 runs in
    // A's iteration n): the static rows A loaded, A's forcing / carried
    // depths, and A's outputs of row n - 1 (B's level-n input one row ahead)
    R H_d1 = 0, H_d2 = 0, rd_d1 = 0, rd_d2 = 0;
    int mb_d1 = 0, mb_d2 = 0;
    R fx_d1 = 0, fx_d2 = 0, fy_d1 = 0, fy_d2 = 0;
    double hu_d1 = 0, hu_d2 = 0, hv_d1 = 0, hv_d2 = 0;
    R u_prev = 0, v_prev = 0;
    double up_prev = 0, vp_prev = 0, sp_prev = 0;
    ld.issue(r0 - 5);
    for (int n = r0 - 5; n < r1 + 2; ++n) {
        const int nb = n - 2;
        const bool runB = nb >= r0 - 3;
        ld.take(n, ia);
        if (n + 1 < r1 + 2) ld.issue(n + 1);
        const bool keepA = n >= r0 - 2;
        A.row(n, ia, keepA, oa);
        if (runB) {
            ib.s2 = oa.s;
            ib.H2 = H_d2;
            ib.mb2 = mb_d2;
            ib.u1 = u_prev;
            ib.v1 = v_prev;
            ib.up1 = up_prev;
            ib.vp1 = vp_prev;
            ib.sp1 = sp_prev;
            ib.rd1 = rd_d2;
            ib.fx0 = fx_d2;
            ib.fy0 = fy_d2;
            ib.hupc0 = hu_d2;
            ib.hvpc0 = hv_d2;
            ib.f0 = R(ld.tab(p.row_f, nb));
            ib.sx0 = R(ld.tab(p.row_sx, nb));
            ib.sy0 = R(ld.tab(p.row_sy, nb));
            ib.wf1 = R(ld.tab(p.row_wf, nb + 1));
            const bool produce = nb >= r0;
            B.row(nb, ib, produce, ob);
            if (produce && writer && nb <= p.ny) {
                const size_t io = (size_t)(nb - 1) * p.nx + (m - 1);
                if (AFORM && p.nsub > subB) {
                    st_out<false, R>(p.frx, io, ob.rhs_u);
                    st_out<false, R>(p.fry, io, ob.rhs_v);
                }
                if constexpr (EXACT) {
                    if (subB < p.nsub) {
                        st_out<sizeof(R) == 8, double>(p.hup_c, io, ob.hu);
                        st_out<sizeof(R) == 8, double>(p.hvp_c, io, ob.hv);
                    }
                }
                store_state<R>(p, io, ob);
            }
        }
        // shift the delay lines
        H_d2 = H_d1; H_d1 = ia.H2;
        mb_d2 = mb_d1; mb_d1 = ia.mb2;
        rd_d2 = rd_d1; rd_d1 = ia.rd1;
        fx_d2 = fx_d1; fx_d1 = oa.rhs_u;
        fy_d2 = fy_d1; fy_d1 = oa.rhs_v;
        if constexpr (EXACT) {
            hu_d2 = hu_d1; hu_d1 = oa.hu;
            hv_d2 = hv_d1; hv_d1 = oa.hv;
        }
        u_prev = oa.u;
        v_prev = oa.v;
        up_prev = oa.up;
        vp_prev = oa.vp;
        sp_prev = oa.sp;
    }
}

// ------------------------------------------------------------------
// K substeps per launch as a pipeline of K waves (one workgroup of 64 K
// threads per work item): wave w runs substep sub + w on row n - 3 w at
// iteration n, on what wave w - 1 produced in the three iterations before
// (its rows n - 3 w + 2, + 1 and + 0), handed over through a ring of
// PIPE_SLOTS rows in LDS with one workgroup barrier per iteration.  Each
// wave holds one substep's window (registers of one stage), the
// intermediate levels never leave the chip, and wave 0 alone reads the
// arrays; the last wave writes them.  The results are those of K launches
// of fused_chunk bit for bit (the same Stage and Loader code).

constexpr int PIPE_SLOTS = 4;
// Rows per unrolled group of the pipeline's march (the window's registers
// rotate by renaming instead of moves).  Measured on MI355X at 2048 x 1536,
// us per substep with 1 / 2 / 4 rows: FP64 61.7 / 58.5 / 57.1, FP32
// 50.1 / 49.0 / 51.3 (the 64-member FP32 ensemble 820 / 801 / 830 us per
// outer step).
template <typename R>
__host__ __device__ constexpr int pipe_unroll()
{
    return sizeof(R) == 8 ? 4 : 2;
}
// output columns per strip with K stages: stage w's results are valid on
// lanes w + 1 .. 61 - 2 w (a stage's result at lane j needs its inputs at
// j - 1 .. j + 2); the last stage writes lanes K .. 63 - 2 K
__host__ __device__ constexpr int pipe_width(int K) { return WAVE - 3 * K; }
// iterations of a work item beyond its rows: the first stage starts
// 2 K + 1 rows above the chunk, the last ends 3 (K - 1) rows later
__host__ __device__ constexpr int pipe_extra(int K) { return 5 * K - 2; }

// What stage w hands to stage w + 1 for one row (each lane its column).
template <typename R>
struct PipeSlot {
    R s[WAVE], u[WAVE], v[WAVE], fx[WAVE], fy[WAVE], H[WAVE], rd[WAVE];
    double sp[WAVE], up[WAVE], vp[WAVE];
    uint8_t mb[WAVE];
};

template <typename R, int K, bool LOAD, bool FORM>
__device__ __forceinline__ void fused_pipe_stage(const FusedParams &p, int chunk_id, int strip, int w,
                                                 bool save_forcing, PipeSlot<R> (*ring)[PIPE_SLOTS])
{
    constexpr int SWK = pipe_width(K);
    const int lane = threadIdx.x % WAVE;
    const int m = strip * SWK + lane - (K - 1);
    const bool colok = (m >= 1 && m <= p.nx);
    const bool writer = colok && lane >= K && lane <= WAVE - 1 - 2 * K;
    const int r0 = chunk_id * p.chunk + 1;
    const int r1 = min(r0 + p.chunk, p.ny + 1);
    constexpr int U = pipe_unroll<R>();
    const int n0 = r0 - 2 * K - 1;  // first iteration
    // iterations n0..n1, a whole number of unrolled groups of U (the rows
    // past the chunk that this adds are computed, not stored)
    const int n1 = n0 + (r1 + 3 * (K - 1) - n0 + U - 1) / U * U - 1;
    const int valid_from = n0 + 3 + 2 * w;  // first row of valid results
    const bool last = (w == K - 1);

    FastStage<R, FORM> st(p, m);
    Loader<R, false, !FORM> ld(p, m);
    StageIn<R> in;
    StageOut<R> o;
    // the row's own static fields for the next stage (inputs arrive two rows,
    // and the Rayleigh coefficient one row, ahead)
    R H_d1 = 0, H_d2 = 0, rd_d1 = 0;
    int mb_d1 = 0, mb_d2 = 0;
    if constexpr (LOAD) ld.issue(n0);
    for (int nb = n0; nb <= n1; nb += U)
#pragma unroll
    for (int n = nb; n < nb + U; ++n) {
        const int r = n - 3 * w;
        if constexpr (LOAD) {
            ld.take(r, in);
            if (r + 1 <= n1) ld.issue(r + 1);
        } else {
            const PipeSlot<R> &a = ring[w - 1][(n - 1) & (PIPE_SLOTS - 1)];  // row r + 2
            const PipeSlot<R> &b = ring[w - 1][(n - 2) & (PIPE_SLOTS - 1)];  // row r + 1
            const PipeSlot<R> &c = ring[w - 1][(n - 3) & (PIPE_SLOTS - 1)];  // row r
            in.s2 = a.s[lane];
            in.H2 = a.H[lane];
            in.mb2 = a.mb[lane];
            in.u1 = b.u[lane];
            in.v1 = b.v[lane];
            in.up1 = b.up[lane];
            in.vp1 = b.vp[lane];
            in.sp1 = b.sp[lane];
            in.rd1 = b.rd[lane];
            in.fx0 = c.fx[lane];
            in.fy0 = c.fy[lane];
            in.hupc0 = in.hvpc0 = 0.0;
            in.f0 = R(ld.tab(p.row_f, r));
            in.sx0 = R(ld.tab(p.row_sx, r));
            in.sy0 = R(ld.tab(p.row_sy, r));
            in.wf1 = R(ld.tab(p.row_wf, r + 1));
        }
        const bool keep = last ? (r >= r0) : (r >= valid_from);
        st.row(r, in, keep, o);
        if (!last) {
            // row r for stage w + 1 (outside the array its mask is 0; what is
            // handed over before the results are valid reaches no output)
            PipeSlot<R> &q = ring[w][n & (PIPE_SLOTS - 1)];
            q.s[lane] = o.s;
            q.u[lane] = o.u;
            q.v[lane] = o.v;
            q.sp[lane] = o.sp;
            q.up[lane] = o.up;
            q.vp[lane] = o.vp;
            q.fx[lane] = o.rhs_u;
            q.fy[lane] = o.rhs_v;
            q.H[lane] = H_d2;
            q.rd[lane] = rd_d1;
            q.mb[lane] = (uint8_t)mb_d2;
        } else if (keep && writer && r < r1) {
            const size_t io = (size_t)(r - 1) * p.nx + (m - 1);
            // the forcing of a call that continues after this launch
            if (save_forcing) {
                st_out<false, R>(p.frx, io, o.rhs_u);
                st_out<false, R>(p.fry, io, o.rhs_v);
            }
            store_state<R>(p, io, o);
        }
        H_d2 = H_d1;
        H_d1 = in.H2;
        mb_d2 = mb_d1;
        mb_d1 = in.mb2;
        rd_d1 = in.rd1;
        __syncthreads();
    }
}

// One work item of the K-stage pipeline; every wave of the workgroup
// calls it.  form_mask bit w: stage w is the first substep of its call
// (forms the wind and drag forcing); save_forcing: the last stage's call
// continues after this launch.
template <typename R, int K>
__device__ __forceinline__ void fused_pipe(const FusedParams &p, int chunk_id, int strip, int form_mask,
                                           bool save_forcing, PipeSlot<R> (*ring)[PIPE_SLOTS])
{
    // the stage index as a scalar: each wave takes one branch, the same
    // number of barriers in every branch
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const bool form = (form_mask >> w) & 1;
    if (w == 0) {
        if (form)
            fused_pipe_stage<R, K, true, true>(p, chunk_id, strip, w, save_forcing, ring);
        else
            fused_pipe_stage<R, K, true, false>(p, chunk_id, strip, w, save_forcing, ring);
    } else {
        if (form)
            fused_pipe_stage<R, K, false, true>(p, chunk_id, strip, w, save_forcing, ring);
        else
            fused_pipe_stage<R, K, false, false>(p, chunk_id, strip, w, save_forcing, ring);
    }
}

// ------------------------------------------------------------------
// Small grids: TILE_K substeps per launch on tiles of 64 x nr points, one
// point per lane and one row per wave.  The march above gives a small grid
// too few waves, each of which then walks its rows one after the other
// (2 rows and 3 of warm-up at 256 x 256: 7 us a substep, most of it waiting);
// here every point is its own lane, a substep is four short phases with the
// row neighbours' values exchanged through LDS between them (the column
// neighbours come by lane shifts), and the intermediate level stays in
// registers.  A tile writes its columns TILE_K .. 63 - 2 TILE_K and rows
// TILE_K .. nr - 1 - 2 TILE_K (a substep reaches one point west and south, two
// east and north; the rim is computed by the tiles on both sides).  The
// formulas and their order are FastStage's: the same bits.  Measured on
// MI355X, us per substep, one launch of the march each / tiles: FP64 64 x 64
// 6.1 / 3.1, 256 x 256 6.6 / 3.8, 512 x 384 9.3 / 7.9; FP32 5.9 / 2.9,
// 6.4 / 3.4, 7.5 / 6.4.  What is left is the launch and the loads' latency
// (about 3 us of a launch) and, from 256 x 256 on, the issue of the rim's
// redundant points (38 % at 16 rows).
constexpr int TILE_K = 2;
constexpr int TILE_MAX_ROWS = 16;
constexpr int TILE_ARRAYS = 12;
constexpr int tile_out_rows(int nr) { return nr - 3 * TILE_K; }
template <typename R>
constexpr size_t tile_lds(int nr) { return (size_t)TILE_ARRAYS * nr * WAVE * sizeof(R); }

// Rows per tile (8, 12 or 16) for a grid or ensemble: `tiles(out_rows)` tiles
// on a chip of `cus` CUs, the fewest rows that the busiest CU works through.
// Measured (FP64, us per substep with 8 / 12 / 16 rows): 128 x 128 3.2 / 3.7 /
// 4.1, 256 x 256 5.5 / 3.8 / 4.3, 512 x 384 10.8 / 9.5 / 7.9.
template <typename F>
inline int tile_rows(long long cus, F tiles)
{
    int best = TILE_MAX_ROWS;
    long long best_cost = -1;
    for (int nr = TILE_MAX_ROWS; nr >= 8; nr -= 4) {
        const long long rounds = (tiles(tile_out_rows(nr)) + cus - 1) / cus;
        const long long cost = rounds * (nr + 4);  // 4: the phases' latency in rows' issue time
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            best = nr;
        }
    }
    return best;
}

// One tile: substeps p.sub .. p.sub + ksub - 1 (ksub <= TILE_K).  form_mask bit
// j: substep j of the launch is the first of its call; save_forcing: the last
// one's call goes on after this launch.  Every wave of the block calls it.
template <typename R>
__device__ __forceinline__ void fused_tile(const FusedParams &p, int ty, int tx, int ksub, int form_mask,
                                           bool save_forcing, R *lds)
{
    const int lane = threadIdx.x % WAVE, nr = blockDim.x / WAVE;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
    const int m = tx * pipe_width(TILE_K) + lane - (TILE_K - 1);
    const int n = ty * tile_out_rows(nr) + w - (TILE_K - 1);
    const FastConst<R> c(p);
    // array a of row r, this lane's column
    auto at = [&](int a, int r) -> R & { return lds[(a * nr + r) * WAVE + lane]; };
    const int wn = min(w + 1, nr - 1), ws = max(w - 1, 0);  // (the rim rows' neighbours reach no output)

    const RowAddr ra{p.nx, p.ny, min(max(m, 1), p.nx)};
    const bool colok = m >= 1 && m <= p.nx;
    const size_t i0 = ra.at(n), i1 = ra.at(n + 1);
    R u = static_cast<const R *>(p.u)[i0], v = static_cast<const R *>(p.v)[i0], s = static_cast<const R *>(p.s)[i0];
    double up = p.up[i0], vp = p.vp[i0], sp = p.sp[i0];
    const R H = static_cast<const R *>(p.H)[i0];
    const R rd = static_cast<const R *>(p.rd)[i0], rd1 = static_cast<const R *>(p.rd)[i1];
    int mb = p.mb[i0], mb1 = p.mb[i1];
    R rhs_u = R(0), rhs_v = R(0);
    if (!(form_mask & 1)) {
        rhs_u = static_cast<const R *>(p.frx_in)[i0];
        rhs_v = static_cast<const R *>(p.fry_in)[i0];
    }
    const int rc = min(max(n, 1), p.ny) - 1;
    const R f0 = R(p.row_f[rc]), sx = R(p.row_sx[rc]), sy = R(p.row_sy[rc]), wf = R(p.row_wf[rc]);
    if (!(colok && n >= 1 && n <= p.ny)) mb = 0;
    if (!(colok && n + 1 >= 1 && n + 1 <= p.ny)) mb1 = 0;

    const bool in = m >= 3 && m <= p.nx - 2 && n >= 3 && n <= p.ny - 2;
    const bool sh = m >= 2 && m <= p.nx - 1 && n >= 2 && n <= p.ny - 1;
    const int l0 = mb & MB_LU, l1 = mb1 & MB_LU;
    const int lus0 = l0 + dpp_from_right(l0), lus1 = l1 + dpp_from_right(l1);
    const bool lu = l0 != 0, lu2 = lus0 == 2, lv = (l0 & l1) != 0, llu = mb & MB_LLU, llv = mb & MB_LLV;
    const bool tw = lu && in, luu = mb & MB_LUU, hw = luu && in, lcu = mb & MB_LCU, lcv = mb & MB_LCV;
    const int cnt = (mb & MB_LUH) ? lus0 + lus1 : 0;
    const R rdu = rd + xr(rd), rdv = rd + rd1;

    for (int j = 0; j < ksub; ++j) {
        const bool form = (form_mask >> j) & 1;
        const R upr = R(up), vpr = R(vp);
        const R w0 = lu ? H + s : R(0);
        const R wp = lu ? H + R(sp) : R(0);
        at(0, w) = w0;
        at(1, w) = wp;
        at(2, w) = s;
        at(3, w) = u;
        at(4, w) = v;
        at(5, w) = upr;
        at(6, w) = vpr;
        __syncthreads();
        // depths, fluxes, shear and Coriolis products
        const R w1 = at(0, wn);
        const R a0 = w0 + xr(w0), a1 = w1 + xr(w1);
        const R hu = fast::depth2(a0, llu, lu2), hv = fast::depth2(w0 + w1, llv, lv);
        const R hh = fast::depth4(a0 + a1, cnt);
        const R hup = fast::depth2(wp + xr(wp), llu, lu2), hvp = fast::depth2(wp + at(1, wn), llv, lv);
        const R ds_v = at(2, wn) - s, u1 = at(3, wn), v1 = at(4, wn), vs = at(4, ws), up1 = at(5, wn), vps = at(6, ws);
        const R fu = u * hu, fv = v * hv;
        const R shear = (up1 - upr) + (xr(vpr) - vpr);
        const R Q = hw ? c.nuid * hh * shear : R(0);
        const R vsum = xr(v) + v, usum = u1 + u;
        const R cor = f0 * hh;
        const R Fc = cor * vsum, Gc = cor * usum;
        const R fvs = fv + xr(fv);
        const R fyU = luu ? fvs * usum : R(0);
        at(7, w) = fv;
        at(8, w) = fu;
        at(9, w) = Q;
        at(10, w) = Fc;
        at(11, w) = fyU;
        __syncthreads();
        // T point: continuity, new depth, tension, drag
        const R fv_s = at(7, ws), fv_n = at(7, wn), ful = xl(fu);
        const R Qs = at(9, ws), Fcs = at(10, ws), fyUs = at(11, ws);
        const R fu1 = at(8, wn);
        const double sn = tw ? fast::surface(c, sp, wf, fu, ful, fv, fv_s) : 0.0;
        const R wnew = lu ? H + R(sn) : R(0);
        const R tens = (upr - xl(upr)) - (vpr - vps);
        const R P = tw ? c.nuid * w0 * tens : R(0);
        R bf = R(0);
        if (form) bf = tw ? fast::drag(c, w0, fu, ful, fv, fv_s) : R(0);
        at(0, w) = wnew;
        at(1, w) = P;
        at(2, w) = bf;
        __syncthreads();
        // momentum and the time-level shift
        const R bf1 = at(2, wn), P1 = at(1, wn);
        if (form) {
            rhs_u = fmad(R(-0.5) * (bf + xr(bf)), upr, sx);
            rhs_v = fmad(R(-0.5) * (bf + bf1), vpr, sy);
        }
        const R hun = fast::depth2(wnew + xr(wnew), llu, lu2), hvn = fast::depth2(wnew + at(0, wn), llv, lv);
        const R fx = (fu + xr(fu)) * (u + xr(u));
        const R gx = (fu + fu1) * vsum;
        const R fyV = (fv + fv_n) * (v + v1), fyVs = (fv_s + fv) * (vs + v);
        R un = fast::momentum(c, rhs_u, xr(s) - s, hu, hup, hun, (fx - xl(fx)) + (fyU - fyUs), (xr(P) - P) + (Q - Qs),
                              rdu, Fc + Fcs, upr);
        R vn = fast::momentum(c, rhs_v, ds_v, hv, hvp, hvn, (gx - xl(gx)) + (fyV - fyVs), (P - P1) + (Q - xl(Q)), rdv,
                              -(Gc + xl(Gc)), vpr);
        un = (lcu && in) ? un : R(0);
        vn = (lcv && in) ? vn : R(0);
        const bool ss = lu && sh, su = lcu && sh, sv = lcv && sh;
        sp = ss ? fast::filter(c.cts, double(s), sn, sp) : sp;
        up = su ? fast::filter(c.cts, double(u), double(un), up) : up;
        vp = sv ? fast::filter(c.cts, double(v), double(vn), vp) : vp;
        s = ss ? R(sn) : s;
        u = su ? un : u;
        v = sv ? vn : v;
        if (j + 1 < ksub) __syncthreads();  // the last reads of the arrays the next substep writes
    }
    if (colok && n >= 1 && n <= p.ny && lane >= TILE_K && lane <= WAVE - 1 - 2 * TILE_K && w >= TILE_K &&
        w <= nr - 1 - 2 * TILE_K) {
        const size_t io = (size_t)(n - 1) * p.nx + (m - 1);
        if (save_forcing) {
            static_cast<R *>(p.frx)[io] = rhs_u;
            static_cast<R *>(p.fry)[io] = rhs_v;
        }
        // (cached: the grid is small and the next launch reads it)
        static_cast<R *>(p.so)[io] = s;
        static_cast<R *>(p.uo)[io] = u;
        static_cast<R *>(p.vo)[io] = v;
        p.spo[io] = sp;
        p.upo[io] = up;
        p.vpo[io] = vp;
    }
}

}  // namespace ibt
