// jk_kernels.hip -- gfx950 kernels of The Joker's likelihood + rejection path.
//
//  k_lnl<L, PHYS, MIXED>   fused per-sample marginal lnL: phase, Kepler solve,
//                          design column, moments, L x L Cholesky, lnL.  One
//                          lane per prior sample; the star's epoch arrays are
//                          wave-uniform and read through scalar loads.
//  k_lnl_split             the same for few rows, a row's epochs over many lanes.
//  k_lnl_cov               the same for a full covariance, rotated on the matrix
//                          cores; k_lnl_cov_lane for few epochs and many rows.
//  k_max_partial / final   NaN-propagating max (np.max).
//  k_reject_words / rows   numpy-PCG64 uniforms generated in registers for the
//                          rows that can pass, exp(ll - max) > u, one 64-bit
//                          mask word per lane (rows: four rows per lane).
//  k_reject_bsum/compact   order-preserving compaction of the mask words.
//  k_uniform               the raw uniforms (tests / callers).
//  k_linear_posterior      a = G^-1 rhs and G^-1 for accepted rows (16
//                          lanes per row).
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "jk_internal.h"

#define JK_PI_HALF 1.57079632679489661923
#define JK_PI_HI 3.141592653589793
#define JK_PI_LO 1.2246467991473532e-16
#define JK_PI_F_HI 3.1415927410125732f
#define JK_PI_F_LO -8.742277657347586e-08f
#define JK_LN2 0.69314718055994530942

__constant__ PcgJump c_jump;
// (A^t, D_t) for t = 0 .. 255: the jump of thread t of a 256-thread workgroup
// from its workgroup's first state.
__constant__ u128 c_tid_A[256];
__constant__ u128 c_tid_D[256];
// (A^64t, D_64t) for t = 0 .. 255: the same for lanes that own 64 rows each.
__constant__ u128 c_tid64_A[256];
__constant__ u128 c_tid64_D[256];

// (sin g_i, cos g_i) on the grid g_i = i * JK_TAB_H, i = 0 .. JK_TAB_N, over
// [0, pi].  JK_TAB_H is pi / 1024 rounded up to 42 significant bits, so i * H
// (i < 2^11) is exact in FP64.  Uploaded once per device by jk_init; the
// kernels that evaluate the likelihood stage it in LDS (26 KB with the FP32
// grid and the log table).  At this spacing cos d needs only the terms to d^4.
#define JK_TAB_N 1024
#define JK_TAB_H 0x1.921fb54443000p-9
#define JK_TAB_INV_H_F 325.9493f
__device__ double2 g_sincos_tab[JK_TAB_N + 1];
// The FP32 grid for the mixed-precision Kepler step: g_i = i * JK_TAB_H32
// (pi / 1024 rounded to FP32), (sin g_i, cos g_i) rounded once to FP32.
#define JK_TAB_H32 0x1.921fb6p-9f
__device__ float2 g_sincos_tab32[JK_TAB_N + 1];
// (R_i, -ln R_i) of jk_log_tab.
__device__ double2 g_log_tab[JK_LOG_TAB_N];
// LDS image: the FP64 table, the log table, then (kernels with mixed-precision
// rows only) the FP32 table packed two per double2 slot.
#define JK_TAB_LOG_OFF (JK_TAB_N + 1)
#define JK_TAB_LDS64 (JK_TAB_LOG_OFF + JK_LOG_TAB_N)
#define JK_TAB_LDS (JK_TAB_LDS64 + (JK_TAB_N + 2) / 2)

// Minimum waves per SIMD asked of the row kernels that evaluate many stars
// or scattered rows: 4 (at most 128 VGPRs) for L <= 3, where the allocator
// otherwise settled some variants at 129-132 VGPRs and 3 waves (at 128 none of
// them spills, but for two VGPRs of the capped pruned launch at L = 3 in mixed
// precision with jitter); none for larger L, which would spill.
#define JK_ROW_WAVES(L) ((L) <= 3 ? 4 : 1)
// The pruned launch with jitter asks for them at L = 4 too (171 VGPRs and 2
// waves in FP64 otherwise: 2^20 rows x 60 epochs 158 -> 96 us; mixed 106 -> 83,
// with three VGPRs spilled), and in mixed precision for 3 at L = 6, with one
// epoch at a time: 1024 and 2048 items of 2048 rows, 24 to 150 epochs, with and
// without survivors, 0.97 to 1.14 times as fast as a persistent grid was; two
// epochs at a time on 2 waves 0.87 to 1.04, on 3 waves 0.87 to 1.12.
#define JK_PRUNE_WAVES(L, PHYS, MIXED)                                                            \
    ((L) <= 3 || ((PHYS) && (L) == 4) ? 4 : ((PHYS) && (MIXED) && (L) == 6 ? 3 : 1))
#define JK_PRUNE_UNROLL(L, PHYS) ((PHYS) && (L) == 6 ? 1 : 2)

// F32: with the FP32 grid of the mixed-precision row.
template <bool F32>
__device__ __forceinline__ void jk_stage_tab(double2 *s_tab)
{
    float2 *t32 = reinterpret_cast<float2 *>(s_tab + JK_TAB_LDS64);
    for (int i = threadIdx.x; i <= JK_TAB_N; i += blockDim.x) {
        s_tab[i] = g_sincos_tab[i];
        if constexpr (F32) t32[i] = g_sincos_tab32[i];
    }
    for (int i = threadIdx.x; i < JK_LOG_TAB_N; i += blockDim.x)
        s_tab[JK_TAB_LOG_OFF + i] = g_log_tab[i];
    __syncthreads();
}

// sin and cos in FP64 of any finite FP64 angle x: Cody-Waite reduction to
// y in [-pi, pi], then the grid as in jk_sincos_tab on |y| (exact d = |y| - g_i
// by Sterbenz's lemma), then the sign of y.
__device__ __forceinline__ void jk_sincos_tab_f64(double x, const double2 *__restrict__ tab,
                                                  double &s, double &c)
{
    const double y = jk_reduce_2pi(x);
    const double ay = fabs(y);
    int idx = (int)(ay * (JK_TAB_N / JK_PI));
    idx = min(max(idx, 0), JK_TAB_N);
    const double2 t = tab[idx];
    const double d = fma(-(double)idx, JK_TAB_H, ay);
    const double d2 = d * d;
    const double sd = fma(d * d2, fma(d2, 1.0 / 120.0, -1.0 / 6.0), d);
    const double cd = fma(d2, fma(d2, 1.0 / 24.0, -0.5), 1.0);
    const double sa = fma(t.x, cd, t.y * sd);
    s = y < 0.0 ? -sa : sa;
    c = fma(t.y, cd, -(t.x * sd));
}

// sin and cos in FP64 of an FP32 angle Ef in [0, pi] (a little outside is
// fine): Ef = g_i + d with g_i the grid point below, |d| <= 1.01 H, then
//   sin Ef = sin g_i cos d + cos g_i sin d,  cos Ef = cos g_i cos d - sin g_i sin d
// with sin d to d^5 and cos d to d^4 (truncation below 2e-18).  d is exact:
// Ef has 24 significant bits and g_i 42 on a grid of the same scale, so their
// difference needs fewer than 53 (one fma: i H is exact, so the fused form
// gives the same bits as the product and the difference).
// The index is clamped into the table whatever Ef is.
__device__ __forceinline__ void jk_sincos_tab(float Ef, const double2 *__restrict__ tab,
                                              double &s, double &c)
{
    int idx = (int)(Ef * JK_TAB_INV_H_F);
    idx = min(max(idx, 0), JK_TAB_N);
    const double2 t = tab[idx];
    const double d = fma(-(double)idx, JK_TAB_H, (double)Ef);
    const double d2 = d * d;
    const double sd = fma(d * d2, fma(d2, 1.0 / 120.0, -1.0 / 6.0), d);
    const double cd = fma(d2, fma(d2, 1.0 / 24.0, -0.5), 1.0);
    s = fma(t.x, cd, t.y * sd);
    c = fma(t.y, cd, -(t.x * sd));
}

// sin and cos in FP32 of E in [0, pi] (a little outside is fine) from the FP32
// grid staged after the FP64 table: E = g_i + d, d = E - i H32 rounded once
// (fma), |d| <= 1.01 H; sin d to d^3 and cos d to d^2 (truncation below
// 4e-12, under FP32 rounding).  The index is clamped into the table.
__device__ __forceinline__ void jk_sincos_tab_f32(float E, const double2 *__restrict__ tab,
                                                  float &s, float &c)
{
    const float2 *__restrict__ t32 = reinterpret_cast<const float2 *>(tab + JK_TAB_LDS64);
    int idx = (int)(E * JK_TAB_INV_H_F);
    idx = min(max(idx, 0), JK_TAB_N);
    const float2 t = t32[idx];
    const float d = fmaf(-(float)idx, JK_TAB_H32, E);
    const float d2 = d * d;
    const float sd = fmaf(d * d2, -1.0f / 6.0f, d);
    const float cd = fmaf(d2, -0.5f, 1.0f);
    s = fmaf(t.x, cd, t.y * sd);
    c = fmaf(t.y, cd, -(t.x * sd));
}

// Kepler in FP64 on ax = |x| in [0, pi] (see jk_kepler_f64 in jk_device.h for
// the convergence argument); this variant evaluates sin/cos with the LDS
// table (jk_sincos_tab_f64).
__device__ __forceinline__ void jk_kepler_poly_f64(double x, double e,
                                                   const double2 *__restrict__ tab,
                                                   double &sinE, double &cosE)
{
    const double ax = fabs(x);
    double E = fmin(fma(0.85, e, ax), JK_PI);
    double s, c;
    jk_sincos_tab_f64(E, tab, s, c);
#pragma unroll 1
    for (int it = 0; it < JK_KEPLER_MAXITER; ++it) {
        const double fp = fma(-e, c, 1.0);
        const double f = fma(-e, s, E - ax);
        const double d = f / fp;
        E -= d;
        if (fabs(d) < JK_KEPLER_TOL) {
            const double s1 = fma(-d, c, s);
            c = fma(d, s, c);
            s = s1;
            break;
        }
        jk_sincos_tab_f64(E, tab, s, c);
    }
    sinE = x < 0.0 ? -s : s;
    cosE = c;
}

// ---------------------------------------------------------------------------
// Non-iterative Kepler solve.
// Starter: Markley (1995, "Kepler equation solver", Celest. Mech. Dyn.
// Astron. 63, 101), a Pade-based cubic accurate to 4.4e-4 rad for every e in
// [0, 1) and asymptotically exact as e -> 1, M -> 0.  It needs only that
// accuracy, so it runs in FP32 with the hardware sqrt / log2 / exp2 / rcp.
// Correction: with f(E) = E - e sin E - M expanded about the starter E1,
//   f(E1 + d) = f0 + f1 d + f2 d^2/2 + f3 d^3/6 + f4 d^4/24 + ...,
//   f0 = E1 - e sin E1 - M, f1 = 1 - e cos E1, f2 = e sin E1, f3 = e cos E1,
//   f4 = -f2,
// the root of the quartic is taken by series reversion in t = -f0 / f1:
//   d = t - b2 t^2 + (2 b2^2 - b3) t^3 + (-5 b2^3 + 5 b2 b3 - b4) t^4
// with b_k = f_k / (k! f1).  This is the fifth-order step of Markley's
// scheme computed with one reciprocal instead of three; from the starter's
// error it leaves an error below the conditioning of the problem
// (ulp(M) / (1 - e cos E)), the answer a converged Newton iteration gives.
// (sin E, cos E) at E = E1 + d come from rotating (sin E1, cos E1) by d with
// fourth-order series (|d| <= 4.4e-4, truncation < 2e-19).
// M is taken in [0, pi].  Per-sample constants: ome = 1 - e and
// a1 = 1.6 pi / ((1 + e) (pi^2 - 6)).
// ---------------------------------------------------------------------------
#define JK_MARKLEY_A0 7.6516382901912925f   // 3 pi^2 / (pi^2 - 6)
#define JK_MARKLEY_A1N 1.29898246041084f    // 1.6 pi / (pi^2 - 6)

__device__ __forceinline__ float jk_markley_starter(float M, float e, float ome, float a1)
{
    const float alpha = fmaf(a1, JK_PI_F_HI - M, JK_MARKLEY_A0);
    const float d = fmaf(alpha, e, 3.0f * ome);
    const float M2 = M * M;
    const float ad = alpha * d;
    const float q = fmaf(2.0f * ad, ome, -M2);
    const float r = M * fmaf(3.0f * ad, d - ome, M2);
    const float q2 = q * q;
    const float x = fabsf(r) + __builtin_amdgcn_sqrtf(fmaxf(fmaf(q2, q, r * r), 0.0f));
    const float w = __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(x) * 0.6666666667f);
    const float den = fmaf(w, w + q, q2);
    // (2 r w / den + M) / d with a single reciprocal
    return fmaf(2.0f * r, w, M * den) * __builtin_amdgcn_rcpf(den * d);
}

// 1/x in FP64 from the hardware reciprocal refined by Newton steps.
__device__ __forceinline__ double jk_rcp1(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    return fma(r, fma(-x, r, 1.0), r);
}

__device__ __forceinline__ double jk_rcp2(double x)
{
    const double r = jk_rcp1(x);
    return fma(r, fma(-x, r, 1.0), r);
}

// Returns false when the correction is outside the starter's error bound
// (|d| >= dmax), or always when dmax < 0 (e so close to 1 that its FP32 copy
// misleads the starter): the caller then re-evaluates the whole sample with
// the bracketed Newton iteration, outside the epoch loop, so that rare path
// adds no registers to the loop.
// With WV the epoch's variance v (sigma^2 + s^2) comes in and its reciprocal
// goes out in *w: both reciprocals come from one, R = 1 / ((1 - e cos E1) v),
// as r = R v and w = R (1 - e cos E1) (two roundings more than separate
// reciprocals, one hardware reciprocal fewer per epoch).
// sin E takes the sign of x by copysign: sin E1 and its rotation are >= 0 on
// [0, pi] up to rounding at the ends of the interval.
template <bool WV = false>
__device__ __forceinline__ bool jk_kepler_markley_f64(double x, double e, float ef, float omef,
                                                      float a1f, double dmax,
                                                      const double2 *__restrict__ tab,
                                                      double &sinE, double &cosE,
                                                      double v = 0.0, double *w = nullptr)
{
    const double ax = fabs(x);
    const float E1f = jk_markley_starter((float)ax, ef, omef, a1f);
    const double E1 = (double)E1f;
    double s1, c1;
    jk_sincos_tab(E1f, tab, s1, c1);
    const double f0 = fma(-e, s1, E1 - ax);
    // One Newton step makes r good to the square of the hardware estimate's
    // error, far below what d (<= 4.4e-4) needs.
    const double D1 = fma(-e, c1, 1.0);
    double r;
    if constexpr (WV) {
        const double R = jk_rcp1(D1 * v);
        r = R * v;
        *w = R * D1;
    } else {
        r = jk_rcp1(D1);
    }
    const double t = -f0 * r;
    const double b2 = (0.5 * e) * s1 * r;
    // e cos E1 r = r - 1 (r (1 - e cos E1) = 1 to a few ulp; the absolute
    // error of r - 1 moves d by t^3 5e-16, far below ulp(E)), over 6 in one fma
    const double b3 = fma(r, 1.0 / 6.0, -1.0 / 6.0);
    const double b22 = b2 * b2;
    const double c3 = fma(2.0, b22, -b3);
    const double c4 = b2 * fma(5.0, b3 - b22, 1.0 / 12.0);   // -b4 = b2 / 12
    const double d = t * fma(t, fma(t, fma(t, c4, c3), -b2), 1.0);
    const double d2 = d * d;
    const double cd = fma(d2, fma(d2, 1.0 / 24.0, -0.5), 1.0);
    const double sd = d * fma(d2, -1.0 / 6.0, 1.0);
    const double s = fma(s1, cd, c1 * sd);
    cosE = fma(c1, cd, -s1 * sd);
    sinE = copysign(s, x);
    return fabs(d) < dmax;
}

// FP32 Kepler for the mixed-precision row: the starter, its sin and cos, and
// one Newton step t = -f0 / f1 applied to (sin, cos) to first order.  In
// FP32 the higher orders of the FP64 correction buy nothing: emulated over
// the Beta prior and e up to 1 - 1e-6 (M down to 1e-9), the design-column
// error of this chain and of the fourth-order one are the same fraction
// (0.2) of the per-epoch error model of the bound, which FP32 rounding of
// sin E, cos E and 1 / (1 - e cos E) sets, not the truncation (t^2 ~ 2e-7).
__device__ __forceinline__ void jk_kepler_markley_f32(float x, float e, float ome, float a1,
                                                      const double2 *__restrict__ tab,
                                                      float &sinE, float &cosE)
{
    const float ax = fabsf(x);
    const float E1 = jk_markley_starter(ax, e, ome, a1);
    float s1, c1;
    jk_sincos_tab_f32(E1, tab, s1, c1);
    const float f0 = fmaf(-e, s1, E1 - ax);
    const float t = -f0 * __builtin_amdgcn_rcpf(fmaf(-e, c1, 1.0f));
    const float s = fmaf(c1, t, s1);
    cosE = fmaf(-s1, t, c1);
    // the sign of x flipped into s by bits (no FP64 compare of the phase)
    sinE = __uint_as_float(__float_as_uint(s) ^ (__float_as_uint(x) & 0x80000000u));
}

// ---------------------------------------------------------------------------
// Fused marginal-likelihood kernel.
// ---------------------------------------------------------------------------
// With BOUND (mixed precision only), *bnd receives a bound on
// |lnL(mixed) - lnL(FP64)| for the row.  First order in the design-column
// error dm_n (the only FP32 quantity that reaches the FP64 moments):
//   dlnL = a_K sum_n w_n r_n dm_n - sum_n w_n dm_n (G^-1 x_n)_0,
// with a_K the posterior mean of K and r_n the residuals at the optimum, so by
// Cauchy-Schwarz, with |dm_n| <= eps_n,
//   |dlnL| <= sqrt(sum_n w_n eps_n^2) (|a_K| sqrt(chi2_min) + sqrt((G^-1)_00)).
// eps_n = 2^-22 (1 + d_n)^2 (1 + d_n / 1000), d_n = 1 / (1 - e cos E_n), covers
// the FP32 solve and design column with a factor of two to spare (emulated
// over the Beta prior and e up to 1 - 1e-6).  eps_n grows with d_n, so
// sum_n w_n eps_n^2 <= eps(max_n d_n)^2 sum_n w_n: the epoch loop keeps only
// sum w and the largest d_n (two instructions per epoch).  The bound is
// doubled again for the terms of second order and given a relative floor of
// 1e-9.
#define JK_BOUND_EPS 2.384185791015625e-07   // 2^-22
// Error-bound value of a row whose lnL entry is only an upper bound on its
// lnL (a row pruned by k_lnl_prune_batch in mixed precision); 0 marks an FP64
// value, a positive bound a mixed-precision value.
#define JK_BOUND_UPPER (-1.0f)

// One prior row's orbit: what every epoch of it shares.
struct RowOrbit {
    double e, invP, nP, M0, M0t, s2, lam0, cw, ecw, swsq, dmax;
    // FP32 copies for the Kepler starter (e capped below 1 in FP32; 1 - e
    // rounded from its FP64 value, so it keeps its relative accuracy) and for
    // the mixed row's design value, which is combined in FP32.
    float ef, omef, a1f, cwf, swsqf, ecwf;
};

// Reads row r's columns and derives its orbit; false for an invalid row
// (its lnL is NaN).  Both precisions read the FP64 columns: the kernels are
// bound by arithmetic, not by the prior stream, and an FP32 copy of e would
// carry a relative error of up to 2^-24 / (1 - e) into sqrt(1 - e^2), the
// scale of the whole design column as e -> 1.
template <bool PHYS>
__device__ __forceinline__ bool jk_row_orbit(const StarDev &st, int64_t r,
                                             const double *__restrict__ P,
                                             const void *__restrict__ e_,
                                             const void *__restrict__ om_,
                                             const void *__restrict__ M0_,
                                             const void *__restrict__ s_,
                                             const double2 *__restrict__ tab, RowOrbit &o)
{
    const double *__restrict__ ecol = static_cast<const double *>(e_);
    const double *__restrict__ omcol = static_cast<const double *>(om_);
    const double *__restrict__ M0col = static_cast<const double *>(M0_);
    const double *__restrict__ scol = static_cast<const double *>(s_);

    const double Pv = P[r];
    const double ev = ecol[r];
    const double omv = omcol[r];
    const double M0v = M0col[r];
    const double sv = PHYS ? scol[r] : 0.0;

    bool valid = isfinite(Pv) && Pv != 0.0 && ev >= 0.0 && ev < 1.0 && isfinite(omv) &&
                 isfinite(M0v);
    if (PHYS) valid = valid && isfinite(sv);
    if (!valid) return false;

    if (st.k_prior_mode == JK_KPRIOR_FIXED_COMPANION_MASS)
        o.lam0 = jk_k_variance(&st, Pv, ev, true);
    else
        o.lam0 = st.lam0;

    o.e = ev;
    o.invP = jk_rcp2(Pv);
    o.nP = JK_TWO_PI * o.invP;
    o.M0 = M0v;
    o.M0t = M0v * JK_INV_TWO_PI;
    o.s2 = sv * sv;
    o.ef = fminf((float)ev, 0.99999994f);
    o.omef = fmaxf((float)(1.0 - ev), 5.9604645e-08f);
    o.a1f = JK_MARKLEY_A1N * __builtin_amdgcn_rcpf(1.0f + o.ef);
    double sw, cw;
    jk_sincos_tab_f64(omv, tab, sw, cw);
    o.swsq = sw * sqrt((1.0 - ev) * (1.0 + ev));
    o.cw = cw;
    o.ecw = ev * cw;
    o.cwf = (float)cw;
    o.swsqf = (float)o.swsq;
    o.ecwf = (float)o.ecw;
    // The FP32 starter sees e rounded to FP32; within 1e-7 of 1 that can put
    // it outside the correction's reach, so such samples take the fallback.
    o.dmax = ev > 0.9999999 ? -1.0 : 1e-3;
    return true;
}

// The design value of an epoch at dt and, with PHYS, its weight from the
// epoch's variance vk = sigma^2 + s^2.  MIXED: denb = 1 / (1 - e cos E) for
// the error bound.  FP64 (not SAFE): bad is set where the row needs the
// bracketed Newton iteration.  FINE: the design value's reciprocal to an ulp
// (two Newton steps on the hardware's) instead of a relative 2e-15.
template <bool PHYS, bool MIXED, bool SAFE, bool FINE = false>
__device__ __forceinline__ double jk_row_epoch(const RowOrbit &o, double dtk, double vk,
                                               const double2 *__restrict__ tab, double &w,
                                               float &denb, bool &bad)
{
    double x;
    if constexpr (MIXED) {
        // the FP32 Kepler step reads x rounded to FP32: the low part of
        // 2 pi (k * 2.4e-16 rad) is far below that rounding
        const double ph = fma(o.nP, dtk, -o.M0);
        x = fma(-rint(ph * JK_INV_TWO_PI), JK_TWO_PI_HI, ph);
    } else {
        // the phase in turns, dt / P - M0 / (2 pi), one rounding; its
        // fractional part is exact (Sterbenz) and scales to radians with
        // one more
        const double pt = fma(o.invP, dtk, -o.M0t);
        x = (pt - rint(pt)) * JK_TWO_PI;
    }
    double m;
    if constexpr (MIXED) {
        float sE, cE;
        jk_kepler_markley_f32((float)x, o.ef, o.omef, o.a1f, tab, sE, cE);
        const float den = __builtin_amdgcn_rcpf(fmaf(-o.ef, cE, 1.0f));
        // the design value combined in FP32 too (an FP32 instruction
        // issues in half the cycles of an FP64 one): its rounding stays
        // inside the per-epoch error model of the bound
        m = (double)fmaf(fmaf(o.cwf, cE - o.ef, -o.swsqf * sE), den, o.ecwf);
        denb = den;
        // the FP32 reciprocal (relative error below 2^-22, which the bound
        // covers)
        if constexpr (PHYS) w = (double)__builtin_amdgcn_rcpf((float)vk);
    } else {
        double sE, cE;
        if constexpr (SAFE) {
            jk_kepler_poly_f64(x, o.e, tab, sE, cE);
            if constexpr (PHYS) w = jk_rcp1(vk);
        } else if constexpr (PHYS) {
            // w = 1 / (sigma^2 + s^2) to a relative 2.5e-15 (one Newton step
            // on the hardware reciprocal, shared with the Kepler step's)
            bad |= !jk_kepler_markley_f64<true>(x, o.e, o.ef, o.omef, o.a1f, o.dmax, tab, sE, cE,
                                                vk, &w);
        } else {
            bad |= !jk_kepler_markley_f64(x, o.e, o.ef, o.omef, o.a1f, o.dmax, tab, sE, cE);
        }
        // m = [cos w (cos E - e) - sin w sqrt(1-e^2) sin E] / (1 - e cos E) + e cos w
        // (one Newton step on the hardware reciprocal: relative 2e-15).
        // cos f + e = (1-e^2) cos E / (1 - e cos E) saves one operation of
        // about 100 but moves the rows of e -> 1 by as much as their rounding
        // already does (up to 1e-8 of the lnL at 1 - e = 1e-6)
        const double f1 = fma(-o.e, cE, 1.0);
        const double den = FINE ? jk_rcp2(f1) : jk_rcp1(f1);
        m = fma(fma(o.cw, cE - o.e, -o.swsq * sE), den, o.ecw);
    }
    return m;
}

// The row's lnL from its sums over the epochs (PHYS: those of the trend
// columns too, and the product prod 2^pexp of the variances; otherwise they
// are star constants).  BOUND: with its error bound, from sum w and the
// largest 1 / (1 - e cos E).
template <int L, bool PHYS, bool BOUND>
__device__ __forceinline__ double jk_row_finish(const StarDev &st, double lam0,
                                                double Smm, double Smr, double Srr,
                                                const double *Smt, const double *Str,
                                                const double *Stt, double prod, int pexp,
                                                double Sw, float dmx,
                                                const double2 *__restrict__ tab, float *bnd)
{
    constexpr int LT = L > 1 ? L - 1 : 1;
    // Assemble G (lower triangle used), u, chi0, log-constant.
    double G[L * L], u[L];
    const double mu0 = st.mu0;
    const bool fcm = st.k_prior_mode == JK_KPRIOR_FIXED_COMPANION_MASS;
    G[0] = (fcm ? jk_rcp2(lam0) : st.lam_inv[0]) + Smm;
    u[0] = fma(-mu0, Smm, Smr);
    // log-constant: st.ln_c / ln_c_phys hold everything but the sample's
    // product prod(sigma_n^2 + s^2) = prod * 2^pexp and, for FixedCompanionMass,
    // ln lam0
    double chi0, lnc, scale = 1.0;
    if constexpr (PHYS) {
        chi0 = Srr;
        lnc = st.ln_c_phys + (double)pexp * JK_LN2;
        scale = prod;
    } else {
        chi0 = st.S_rr;
        lnc = st.ln_c;
    }
    if (fcm) scale *= lam0;
    chi0 = fma(mu0 * mu0, Smm, fma(-2.0 * mu0, Smr, chi0));
    if constexpr (L > 1) {
#pragma unroll
        for (int j = 1; j < L; ++j) {
            G[j * L] = Smt[j - 1];
            G[j] = Smt[j - 1];
            const double trj = PHYS ? Str[j - 1] : st.S_tr[j - 1];
            u[j] = fma(-mu0, Smt[j - 1], trj);
#pragma unroll
            for (int q = 1; q <= j; ++q) {
                const double tt =
                    PHYS ? Stt[(j - 1) * LT + (q - 1)] : st.S_tt[(j - 1) * JK_LMAX + (q - 1)];
                const double g = (q == j ? st.lam_inv[j] : 0.0) + tt;
                G[j * L + q] = g;
                G[q * L + j] = g;
            }
        }
    }
    if constexpr (BOUND) {
        double post[3];
        const double ll = jk_finish_lnl<L, true>(G, u, chi0, lnc, scale, tab + JK_TAB_LOG_OFF, post);
        const double aK = fabs(mu0 + post[1]);
        const double t1 = 1.0 + (double)dmx;
        const double ek = t1 * t1 * fma(1e-3, (double)dmx, 1.0);
        double b = 2.0 * JK_BOUND_EPS * ek * sqrt(Sw) *
                   fma(aK, sqrt(fmax(post[2], 0.0)), sqrt(fmax(post[0], 0.0)));
        // the weights' relative error e_w moves lnL by at most
        // e_w (chi2_min + L) / 2 (envelope theorem on chi2_min; the log-det
        // term is tr(G^-1 X^T W X) e_w <= L e_w); e_w < 2^-22 for the FP32
        // reciprocal of the physical jitter mode, 2.4e-15 otherwise
        b += (PHYS ? JK_BOUND_EPS : 2e-15) * (fmax(post[2], 0.0) + (double)L);
        b = fma(1e-9, 1.0 + fabs(ll), b) * 1.000001;
        *bnd = (isfinite(b) && isfinite(ll)) ? (float)b : INFINITY;
        return ll;
    } else {
        return jk_finish_lnl<L>(G, u, chi0, lnc, scale, tab + JK_TAB_LOG_OFF);
    }
}

// With ONE the first trend column is the constant 1 (StarDev::t0_one): its
// products fold away, with the same roundings (w * 1 = w exactly), and the
// bound's sum of the weights is that column's own moment.
// With REC the epoch loop reads the epochs' records (StarDev::ep: one base
// address, so few scalar registers and one or two scalar loads per epoch),
// else the separate arrays.  Same values either way; which is faster is the
// register allocator's doing: the FP64 rows (2^24 rows x 16 epochs 957 -> 927 us
// with the operations saved above; 2^20 x 37 at L = 5 134 -> 127 us, where scalars
// spilled into vector lanes went from 72 to 30) and the mixed
// rows of many stars (64 x 2^18 rows 1935 -> 1895 us) take the records, the
// mixed single-star row the arrays (2^22 x 50: 394 us, with records 415).
// LONE: the row of a launch of at most one wave per SIMD (k_lnl).
// U: epochs per turn of the loop, four where every fourth renormalises the
// product and the registers allow it (2^24 rows x 16 epochs 936 -> 930 us), else
// two.
template <int L, bool PHYS, bool MIXED, bool SAFE = false, bool BOUND = false, bool ONE = false,
          bool LONE = false, bool REC = !MIXED && !LONE,
          int U = LONE || (PHYS && !MIXED && ONE) ? 4 : 2>
__device__ __forceinline__ double jk_lnl_row(const StarDev &st, int64_t r,
                                             const double *__restrict__ P,
                                             const void *__restrict__ e_,
                                             const void *__restrict__ om_,
                                             const void *__restrict__ M0_,
                                             const void *__restrict__ s_,
                                             const double2 *__restrict__ tab,
                                             float *bnd = nullptr)
{
    static_assert(!BOUND || MIXED, "the error bound belongs to the mixed-precision row");
    if constexpr (BOUND) *bnd = INFINITY;
    RowOrbit o;
    if (!jk_row_orbit<PHYS>(st, r, P, e_, om_, M0_, s_, tab, o)) return __builtin_nan("");

    constexpr int LT = L > 1 ? L - 1 : 1, LT0 = L - 1;
    double Smm = 0.0, Smr = 0.0;
    double Smt[LT];
    double Stt[LT * LT], Str[LT], Srr = 0.0;
    double prod = 1.0;
    int pexp = 0;
#pragma unroll
    for (int j = 0; j < LT; ++j) {
        Smt[j] = 0.0;
        Str[j] = 0.0;
#pragma unroll
        for (int k = 0; k < LT; ++k) Stt[j * LT + k] = 0.0;
    }

    const int N = st.n;
    bool bad = false;
    double Sw = 0.0;       // sum w (BOUND only; with ONE it is Stt[0])
    float dmx = 0.0f;      // largest 1 / (1 - e cos E) (BOUND only)
#pragma unroll U
    for (int k = 0; k < N; ++k) {
        const double *__restrict__ ep = st.ep + (size_t)k * (JK_EP_T + LT0);
        const double vk = PHYS ? (REC ? ep[JK_EP_SIG2] : st.sig2[k]) + o.s2 : 0.0;
        double w = 0.0;
        float denb = 0.0f;
        const double m = jk_row_epoch<PHYS, MIXED, SAFE>(o, REC ? ep[JK_EP_DT] : st.dt[k], vk,
                                                              tab, w, denb, bad);
        const double rp = REC ? ep[JK_EP_RP] : st.rp[k];
        if constexpr (PHYS) {
            // sum ln w = -ln of the running product of the FP64 variances,
            // renormalised every fourth epoch (frexp scales by a power of
            // two, exactly, so the product's rounding is that of
            // renormalising every epoch; four factors stay far inside the
            // exponent range)
            prod *= vk;
            if ((k & 3) == 3) {
                int ex;
                prod = frexp(prod, &ex);
                pexp += ex;
            }
        } else {
            w = REC ? ep[JK_EP_IVAR] : st.ivar[k];
        }
        if constexpr (BOUND) {
            if constexpr (!ONE) Sw += w;
            dmx = fmaxf(dmx, denb);
        }
        const double wm = w * m;
        Smm = fma(wm, m, Smm);
        Smr = fma(wm, rp, Smr);
        if constexpr (L > 1) {
#pragma unroll
            for (int j = 0; j < L - 1; ++j) {
                const double Tj =
                    ONE && j == 0 ? 1.0 : (REC ? ep[JK_EP_T + j] : st.T[j * N + k]);
                Smt[j] = fma(wm, Tj, Smt[j]);
                if constexpr (PHYS) {
                    const double wT = w * Tj;
                    Str[j] = fma(wT, rp, Str[j]);
#pragma unroll
                    for (int q = 0; q <= j; ++q) {
                        const double Tq =
                            ONE && q == 0 ? 1.0 : (REC ? ep[JK_EP_T + q] : st.T[q * N + k]);
                        Stt[j * LT + q] = fma(wT, Tq, Stt[j * LT + q]);
                    }
                }
            }
        }
        if constexpr (PHYS) {
            if constexpr (MIXED)
                Srr = fma(w * rp, rp, Srr);
            else    // r'^2 rounded once, on the host where the record holds it
                Srr = fma(w, REC ? ep[JK_EP_RP2] : rp * rp, Srr);
        }
    }

    if constexpr (BOUND && ONE) Sw = PHYS ? Stt[0] : st.S_tt[0];
    if constexpr (!MIXED && !SAFE) {
        if (bad) return jk_lnl_row<L, PHYS, false, true>(st, r, P, e_, om_, M0_, s_, tab);
    }
    return jk_row_finish<L, PHYS, BOUND>(st, o.lam0, Smm, Smr, Srr, Smt, Str, Stt, prod, pexp,
                                         Sw, dmx, tab, bnd);
}

// ---------------------------------------------------------------------------
// Few rows: a workgroup of 4 waves takes R <= 64 rows.  With one lane per row,
// n rows are n / 64 waves, and below 4096 of them (4 per SIMD) the device
// idles while each lane walks its epochs alone; its Kepler solves, which do
// not depend on one another, are nearly all of that work.  So three waves
// evaluate (row, epoch) pairs, G = 192 / R lanes to a row, and leave each
// pair's design value m and weight w in LDS, a chunk of epochs at a time; the
// fourth, one lane per row, adds the chunk before to the rows' sums, epoch
// after epoch, meanwhile (two buffers, one barrier per chunk).  Each sum
// therefore rounds exactly as in jk_lnl_row, and the row's lnL (and bound) is
// the same bits however it is evaluated.  A row that needs the bracketed
// Newton iteration is evaluated again by jk_lnl_row's own fallback.
// Tried first: one lane per (row, sum) adding up (three LDS reads per sum and
// epoch made LDS the bound), and every wave evaluating with a barrier around
// one wave's adding (the other three idle meanwhile).
// ---------------------------------------------------------------------------
#define JK_SPLIT_PAIRS 512

template <int L, bool PHYS, bool MIXED>
struct SplitLds {
    // an epoch's record: r', sigma^2 or ivar, T, dt; the epochs of a chunk at
    // most (one value of the next chunk per evaluating lane)
    static constexpr int NEP = L + 2, CMAX = 192 / NEP;
    struct Chunk {
        double m[JK_SPLIT_PAIRS];
        double w[PHYS ? JK_SPLIT_PAIRS : 1];
    } chunk[2];
    double ep[3][CMAX * NEP];      // the chunk added up, the one evaluated, the next
    float dmx[MIXED ? 192 : 1];
    int bad[64];
};

// A lane's number in the split: the workgroup's lanes counted from wave sw,
// the one that adds up (another wave in each workgroup, so that the SIMDs of
// a compute unit share that work).  Lanes 0 .. 63 add up, lane l row l; lane
// 64 + q evaluates epochs of row q mod R.
__device__ __forceinline__ int jk_split_lane(int sw)
{
    return ((int)threadIdx.x - 64 * sw) & 255;
}

// The adding wave of workgroup b.  Workgroups go round the 8 XCDs, and within
// one round its 32 compute units: those that share a compute unit differ in
// b / 256.
__device__ __forceinline__ int jk_split_wave(unsigned b)
{
    return (int)((b >> 3) + (b >> 8)) & 3;
}

__device__ __forceinline__ int jk_split_row(int lane, int R)
{
    return lane < 64 ? lane : (lane - 64) % R;
}

// Every lane of the workgroup calls this with the same star, R and sw; r: the
// cache row of the lane's row (jk_split_row), -1 for none.  The result is
// that of the lanes whose number is below R.
template <int L, bool PHYS, bool MIXED>
__device__ __forceinline__ double jk_rows_split(const StarDev &st, int R, int sw, int64_t r,
                                                const double *__restrict__ P,
                                                const void *__restrict__ e_,
                                                const void *__restrict__ om_,
                                                const void *__restrict__ M0_,
                                                const void *__restrict__ s_,
                                                const double2 *__restrict__ tab,
                                                SplitLds<L, PHYS, MIXED> &sh, float *bnd)
{
    typedef SplitLds<L, PHYS, MIXED> Sh;
    const int lane = jk_split_lane(sw), G = 192 / R, N = st.n;
    int C = min(JK_SPLIT_PAIRS / R, Sh::CMAX);      // whole rounds of the lanes, if any fit
    C = C >= 2 * G ? C / (2 * G) * (2 * G) : (C >= G ? G : C);
    const int row = jk_split_row(lane, R), g = (lane - 64) / R;
    RowOrbit o;
    const bool valid = r >= 0 && jk_row_orbit<PHYS>(st, r, P, e_, om_, M0_, s_, tab, o);
    const bool sums = lane < 64;      // wave-uniform
    constexpr int LT = L > 1 ? L - 1 : 1;
    double Smm = 0.0, Smr = 0.0, Srr = 0.0, Sw = 0.0, prod = 1.0;
    double Smt[LT], Str[LT], Stt[LT * LT];
    int pexp = 0;
#pragma unroll
    for (int j = 0; j < LT; ++j) {
        Smt[j] = 0.0;
        Str[j] = 0.0;
#pragma unroll
        for (int k = 0; k < LT; ++k) Stt[j * LT + k] = 0.0;
    }
    __syncthreads();   // the workgroup's previous rows are done with sh
    if (sums) sh.bad[lane] = 0;
    bool bad = false;
    float dmx = 0.0f;
    const int nch = (N + C - 1) / C;
    // evaluating lane 64 + q brings in value q of each chunk's records, a chunk
    // ahead of its use
    const int ev = (lane - 64) / C, ek = lane - 64 - ev * C;
    const double *esrc = nullptr;
    if (!sums && ev < Sh::NEP)
        esrc = (ev == 0 ? st.rp
                        : (ev == 1 ? (PHYS ? st.sig2 : st.ivar)
                                   : (ev == L + 1 ? st.dt : st.T + (size_t)(ev - 2) * N))) + ek;
    double enext = esrc && ek < N ? *esrc : 0.0;
    if (esrc) sh.ep[0][ek * Sh::NEP + ev] = enext;
    __syncthreads();
    for (int c = 0; c <= nch; ++c) {
        if (!sums && c < nch) {
            typename Sh::Chunk &ck = sh.chunk[c & 1];
            const int c0 = c * C, cnt = min(C, N - c0);
            if (esrc && c0 + C + ek < N) enext = esrc[c0 + C];
            if (valid && g < G) {
                const double *rec = sh.ep[c % 3];
                // two epochs at a time, both solved before either is stored:
                // the LDS stores would keep the second solve behind the first
                for (int kk = g; kk < cnt; kk += 2 * G) {
                    const bool two = kk + G < cnt;
                    const int k2 = two ? kk + G : kk;
                    const double d1 = rec[kk * Sh::NEP + L + 1], d2 = rec[k2 * Sh::NEP + L + 1];
                    const double v1 = PHYS ? rec[kk * Sh::NEP + 1] + o.s2 : 0.0;
                    const double v2 = PHYS ? rec[k2 * Sh::NEP + 1] + o.s2 : 0.0;
                    double w1 = 0.0, w2 = 0.0, m1, m2 = 0.0;
                    float b1 = 0.0f, b2 = 0.0f;
                    if (__any(two)) {
                        m1 = jk_row_epoch<PHYS, MIXED, false>(o, d1, v1, tab, w1, b1, bad);
                        m2 = jk_row_epoch<PHYS, MIXED, false>(o, d2, v2, tab, w2, b2, bad);
                    } else {
                        m1 = jk_row_epoch<PHYS, MIXED, false>(o, d1, v1, tab, w1, b1, bad);
                    }
                    ck.m[kk * R + row] = m1;
                    if constexpr (PHYS) ck.w[kk * R + row] = w1;
                    if (two) {
                        ck.m[k2 * R + row] = m2;
                        if constexpr (PHYS) ck.w[k2 * R + row] = w2;
                    }
                    if constexpr (MIXED) dmx = fmaxf(dmx, fmaxf(b1, b2));
                }
            }
        }
        if (sums && c > 0 && lane < R) {
            const typename Sh::Chunk &ck = sh.chunk[(c - 1) & 1];
            const double *rec = sh.ep[(c - 1) % 3];
            const int c0 = (c - 1) * C, cnt = min(C, N - c0);
            // the LDS reads of U epochs in flight together
            constexpr int U = L <= 4 ? 4 : 2;
            for (int k0 = 0; k0 < cnt; k0 += U) {
                double em[U], ew[U], er[U][Sh::NEP];
#pragma unroll
                for (int j = 0; j < U; ++j) {
                    const int kk = min(k0 + j, cnt - 1);
                    em[j] = ck.m[kk * R + row];
                    ew[j] = PHYS ? ck.w[kk * R + row] : rec[kk * Sh::NEP + 1];
#pragma unroll
                    for (int q = 0; q < L + 1; ++q) er[j][q] = rec[kk * Sh::NEP + q];
                }
#pragma unroll
                for (int j = 0; j < U; ++j) {
                    if (k0 + j >= cnt) break;
                    const double m = em[j], w = ew[j], rp = er[j][0];
                    const double *ep = er[j];
                    if constexpr (PHYS) {
                        prod *= ep[1] + o.s2;
                        if (((c0 + k0 + j) & 3) == 3) {
                            int ex;
                            prod = frexp(prod, &ex);
                            pexp += ex;
                        }
                    }
                    if constexpr (MIXED) Sw += w;
                    const double wm = w * m;
                    Smm = fma(wm, m, Smm);
                    Smr = fma(wm, rp, Smr);
                    if constexpr (L > 1) {
#pragma unroll
                        for (int i = 0; i < L - 1; ++i) {
                            Smt[i] = fma(wm, ep[2 + i], Smt[i]);
                            if constexpr (PHYS) {
                                const double wT = w * ep[2 + i];
                                Str[i] = fma(wT, rp, Str[i]);
#pragma unroll
                                for (int q = 0; q <= i; ++q)
                                    Stt[i * LT + q] = fma(wT, ep[2 + q], Stt[i * LT + q]);
                            }
                        }
                    }
                    if constexpr (PHYS)
                        Srr = MIXED ? fma(w * rp, rp, Srr) : fma(w, rp * rp, Srr);
                }
            }
        }
        if (esrc && c + 1 < nch) sh.ep[(c + 1) % 3][ek * Sh::NEP + ev] = enext;
        if (c == nch - 1) {
            // after the last chunk's pairs: what the adding lanes need of them
            if (bad) sh.bad[row] = 1;
            if constexpr (MIXED)
                if (!sums) sh.dmx[lane - 64] = dmx;
        }
        __syncthreads();
    }
    if constexpr (MIXED) *bnd = INFINITY;
    if (!valid || lane >= R) return __builtin_nan("");
    if constexpr (!MIXED) {
        if (sh.bad[row]) return jk_lnl_row<L, PHYS, false, true>(st, r, P, e_, om_, M0_, s_, tab);
    } else {
        for (int q = 0; q < G; ++q) dmx = fmaxf(dmx, sh.dmx[q * R + row]);
    }
    return jk_row_finish<L, PHYS, MIXED>(st, o.lam0, Smm, Smr, Srr, Smt, Str, Stt, prod, pexp, Sw,
                                         dmx, tab, bnd);
}

// Rows per workgroup of the split evaluation of n rows of N epochs, or 0 for
// the launch with one row per lane.  R = n / 512 up to 40, then n / 768 up to
// 64 (with R = 64 at 33001 rows x 149 epochs 42 us instead of 37, with n / 1024
// 41).  The line between the two was measured on one MI355X from 4 to 200 epochs,
// L = 2 (without and with jitter), 3 (both), 5 and 6, 1000 to 49152 rows: the
// split's fixed cost (staging, barriers, the adding wave's last chunk) falls on
// every workgroup, so the rows it pays for grow with the epochs; more rows
// than that fill the SIMDs by themselves, the sooner in mixed precision, whose
// solves are cheaper against the same FP64 sums.
// FP64, one row per lane / split, us (L = 2 with jitter): N = 10: 2048 rows
// 6.1 / 5.9, 8192 6.2 / 6.5; N = 17: 2048 7.7 / 6.5, 16384 7.6 / 7.7; N = 37:
// 2048 12.3 / 8.5, 20480 12.5 / 10.9, 30000 12.4 / 12.8; N = 101: 2048 27.3 /
// 14.6, 36864 27.6 / 24.8, 43008 27.7 / 30.3.  Mixed: N = 17: 2048 7.2 / 7.1,
// 8192 7.3 / 8.3; N = 37: 2048 11.4 / 9.0, 20480 11.6 / 10.6, 30000 11.6 / 12.4;
// N = 101: 2048 24.8 / 14.9, 49152 25.1 / 24.5.
#define JK_SPLIT_MAX_ROWS 49152
#define JK_SPLIT_RMIN 8
// Rows that give every SIMD one wave.
#define JK_LONE_MAX_ROWS 65536

static int64_t jk_split_max_rows(int N, bool mixed)
{
    if (!mixed) return N < 10 ? 0 : std::min<int64_t>(36864, 600 * ((int64_t)N - 3));
    if (N < 30) return N < 17 ? 0 : 2048;
    return std::min<int64_t>(JK_SPLIT_MAX_ROWS, std::max<int64_t>(20480, 490 * (int64_t)N));
}

static int jk_split_rows(int64_t n, int N, bool mixed)
{
    if (n > jk_split_max_rows(N, mixed)) return 0;
    int R = (int)((n + 511) / 512);
    if (R > 40) R = (int)((n + 767) / 768);
    return std::min(std::max(std::max(R, 192 / N), JK_SPLIT_RMIN), 64);
}

// ---------------------------------------------------------------------------
// Full-covariance rows, FP64.  With C = Q diag(lambda) Q^T, C + s^2 I is
// diagonal in the same eigenbasis (lambda + s^2), and the marginal
// likelihood ln N(y | M mu, C + s^2 I + M Lambda M^T) does not change under
// the orthogonal change of basis (|det Q| = 1).  The star's data are stored
// rotated (StarDev::Qt); the rows' design columns are computed per epoch and
// rotated, m'_i = sum_k Qt[i][k] m_k, and fed to the same moments and finish
// with the eigenvalues as the variances.
//
// The rotation of a wave's rows is a matrix product, and runs on the matrix
// cores (FP64 16x16x4): a wave takes 16 rows, lane l evaluating row l & 15 at
// epoch 4 c + (l >> 4) in step c, which is the product's right operand as it
// stands; the left one, Q^T in LDS, is read once per step and 16 rows.  The
// products accumulate in registers (16 eigenvalues a tile) while the next
// step's Kepler solves run on the vector units, so the N^2 multiply-adds per
// row cost next to nothing, and the solves bound the kernel as they do the
// diagonal one.  The weights and the design values' reciprocals are good to an
// ulp (jk_rcp2), as they were with one lane per row: the solves hide the second
// Newton step (2^18 x 40 69.5 us with one step, 71.5 with two and the variances'
// product renormalised at each factor; 524288 x 64 246 and 244).  The error of the lnL against 80-bit arithmetic, 60 stars of 4 to 64
// epochs, is 0.74 of that form's in the mean.  Against one lane per row (a serial dot product, one LDS read
// per multiply-add, 64 rows' columns in LDS): 2^18 rows x 40 epochs 182 ->
// 75 us, 524288 x 64 1383 -> 245 us, 3000 x 64 84 -> 17 us, 2^18 x 5 30 ->
// 27 us.
// ---------------------------------------------------------------------------
#define JK_COV_ROWS 64      // rows per workgroup, 16 a wave

typedef double jk_f64x4 __attribute__((ext_vector_type(4)));

// Doubles per epoch of the LDS copy of Q (epoch-major): a multiple of 16 at
// least N, = 16 mod 32, so that the four epochs a step reads fall on
// different banks.
__host__ __device__ __forceinline__ int jk_cov_pitch(int N)
{
    return (N + 15) / 32 * 32 + 16;
}

// Dynamic LDS of k_lnl_cov: Q, then per eigenvalue r', sigma^2 / ivar and T,
// and dt per epoch.
__host__ __device__ __forceinline__ int jk_cov_lds_doubles(int N, int L)
{
    return (N + 3) / 4 * 4 * jk_cov_pitch(N) + N * (L + 2);
}

// The rotated design values of the wave's rows: acc[t][r] of lane l is
// eigenvalue 16 t + 4 r + (l >> 4) of row l & 15.  With SAFE, rows marked bad
// take the bracketed Newton iteration; else bad is set where a row needs it.
template <bool SAFE>
__device__ __forceinline__ void jk_cov_rotate(const StarDev &st, const RowOrbit &o, bool valid,
                                              const double2 *__restrict__ tab,
                                              const double *s_q, const double *s_dt,
                                              jk_f64x4 acc[4], bool &bad)
{
    const int lane = threadIdx.x & 63, kq = lane >> 4, N = st.n;
    const int pitch = jk_cov_pitch(N), nt = (N + 15) / 16;
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = jk_f64x4{0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < N; k0 += 4) {
        const int k = k0 + kq;
        double m = 0.0;
        if (valid && k < N) {
            double w;
            float denb;
            bool b = false;
            m = jk_row_epoch<false, false, false, true>(o, s_dt[k], 0.0, tab, w, denb, b);
            if constexpr (SAFE) {
                if (bad)
                    m = jk_row_epoch<false, false, true, true>(o, s_dt[k], 0.0, tab, w, denb, b);
            } else {
                bad |= b;
            }
        }
        const double *q = s_q + (size_t)k * pitch + (lane & 15);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (t < nt)
                acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(q[16 * t], m, acc[t], 0, 0, 0);
    }
}

// Sum over the four lanes of a row (the same value in each).
__device__ __forceinline__ double jk_cov_sum(double v)
{
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// ---------------------------------------------------------------------------
// Block-level helpers (256 threads = 4 wavefronts of 64).
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_nanmax(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = jk_nanmax(v, __shfl_xor(v, off, 64));
    return v;
}

__device__ __forceinline__ int64_t wave_sum_i64(int64_t v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Inclusive scan across the wavefront.
__device__ __forceinline__ int64_t wave_incl_scan_i64(int64_t v, int lane)
{
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int64_t t = __shfl_up(v, off, 64);
        if (lane >= off) v += t;
    }
    return v;
}

// Dense launch: ll[i] = lnL(row rows[i] or i), one lane per row, the grid
// (jk_dense_blocks) striding over the rows so that each workgroup stages the
// sin/cos table once for several rows.  With blockmax != nullptr each wave
// also writes the NaN-propagating maximum of its rows to blockmax[wave]
// (4 jk_dense_blocks(n) entries), so the rejection step need not read the
// lnL array a second time to find the maximum.  With BOUND (mixed
// precision), bound[i] receives the row's error bound (jk_lnl_row).
//
// LONE: the FP64 instance for launches of at most one wave per SIMD
// (JK_LONE_MAX_ROWS).  Nothing else runs on the SIMD while such a wave waits,
// so its time is its own chain of dependent operations, and what shortens that
// is epochs in flight together: four at a time, scheduled for two waves per
// SIMD at most (for more, the compiler keeps registers down by finishing one
// epoch's table read before it starts the next), and the epochs from the
// arrays, several to a scalar load.  60000 rows by the other instance and by
// this one, us, for L = 2 and 3 without jitter, 2 and 3 with, 5 without, 6 with:
// 16 epochs 7.7 -> 7.3, 8.7 -> 7.7, 8.6 -> 7.4, 7.8 -> 7.8, 9.5 -> 8.7, 9.6 -> 9.5;
// 101 epochs 29.4 -> 25.8, 34.0 -> 27.8, 35.1 -> 28.2, 30.4 -> 30.2,
// 38.1 -> 31.0, 39.2 -> 38.1.  With two waves per SIMD (131072 rows) it is from
// 7 % faster (101 epochs, L = 3, no jitter) to 4 % slower (16 epochs, L = 5),
// with three up to 12 % slower.
template <int L, bool PHYS, bool MIXED, bool BOUND, bool ONE = false, bool LONE = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, LONE ? 2 : 8)))
void k_lnl(const StarDev st, int64_t n, const double *__restrict__ P, const void *__restrict__ e_,
           const void *__restrict__ om_, const void *__restrict__ M0_,
           const void *__restrict__ s_, const int64_t *__restrict__ rows,
           double *__restrict__ ll, double *__restrict__ blockmax, float *__restrict__ bound)
{
    __shared__ double2 s_tab[MIXED ? JK_TAB_LDS : JK_TAB_LDS64];
    jk_stage_tab<MIXED>(s_tab);
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    double vmax = -INFINITY;
    for (int64_t i = t; i < n; i += stride) {
        const int64_t r = rows ? rows[i] : i;
        double v;
        if constexpr (BOUND) {
            float b;
            v = jk_lnl_row<L, PHYS, MIXED, false, true, ONE>(st, r, P, e_, om_, M0_, s_, s_tab, &b);
            bound[i] = b;
        } else {
            v = jk_lnl_row<L, PHYS, MIXED, false, false, ONE, LONE>(st, r, P, e_, om_, M0_, s_,
                                                                    s_tab);
        }
        ll[i] = v;
        vmax = jk_nanmax(vmax, v);
    }
    if (blockmax) {
        // one partial per wave: no barrier, so a finished wave retires at once
        vmax = wave_nanmax(vmax);
        if ((threadIdx.x & 63) == 0) blockmax[t >> 6] = vmax;
    }
}

// The dense launch for few rows (jk_split_rows): blockmax[block] receives the
// workgroup's maximum.
template <int L, bool PHYS, bool MIXED>
__global__ __launch_bounds__(256) void k_lnl_split(const StarDev st, int64_t n, int R,
                                                   const double *__restrict__ P,
                                                   const void *__restrict__ e_,
                                                   const void *__restrict__ om_,
                                                   const void *__restrict__ M0_,
                                                   const void *__restrict__ s_,
                                                   const int64_t *__restrict__ rows,
                                                   double *__restrict__ ll,
                                                   double *__restrict__ blockmax,
                                                   float *__restrict__ bound)
{
    __shared__ double2 s_tab[MIXED ? JK_TAB_LDS : JK_TAB_LDS64];
    __shared__ SplitLds<L, PHYS, MIXED> sh;
    jk_stage_tab<MIXED>(s_tab);
    const int sw = jk_split_wave(blockIdx.x), lane = jk_split_lane(sw);
    const int row = jk_split_row(lane, R);
    const int64_t i = (int64_t)blockIdx.x * R + row;
    const int64_t r = row < R && i < n ? (rows ? rows[i] : i) : -1;
    float b = 0.0f;
    const double v =
        jk_rows_split<L, PHYS, MIXED>(st, R, sw, r, P, e_, om_, M0_, s_, s_tab, sh, &b);
    if (lane >= 64) return;
    const bool mine = lane < R && i < n;
    if (mine) {
        ll[i] = v;
        if (MIXED && bound) bound[i] = b;
    }
    if (blockmax) {
        const double vmax = wave_nanmax(mine ? v : -INFINITY);
        if ((threadIdx.x & 63) == 0) blockmax[blockIdx.x] = vmax;
    }
}

// A full-covariance row's sums over the eigenvalues.  ep: r', sigma^2 (PHYS) or
// ivar and T, N values each.
template <int L, bool PHYS>
struct CovSums {
    static constexpr int LT = L > 1 ? L - 1 : 1;
    double Smm = 0.0, Smr = 0.0, Srr = 0.0, prod = 1.0;
    double Smt[LT] = {}, Str[LT] = {}, Stt[LT * LT] = {};
    int pexp = 0;

    // eigenvalue i, with rotated design value m
    __device__ __forceinline__ void add(double m, int i, int N, const double *ep, double s2)
    {
        const double rp = ep[i];
        double w = ep[N + i];
        if constexpr (PHYS) {
            const double vk = w + s2;
            w = jk_rcp2(vk);
            // renormalised at every factor: any finite variance keeps
            // its logarithm
            int ex;
            prod = frexp(prod * vk, &ex);
            pexp += ex;
        }
        const double wm = w * m;
        Smm = fma(wm, m, Smm);
        Smr = fma(wm, rp, Smr);
        if constexpr (L > 1) {
#pragma unroll
            for (int j = 0; j < L - 1; ++j) {
                const double Tj = ep[(j + 2) * N + i];
                Smt[j] = fma(wm, Tj, Smt[j]);
                if constexpr (PHYS) {
                    const double wT = w * Tj;
                    Str[j] = fma(wT, rp, Str[j]);
#pragma unroll
                    for (int q = 0; q <= j; ++q)
                        Stt[j * LT + q] = fma(wT, ep[(q + 2) * N + i], Stt[j * LT + q]);
                }
            }
        }
        if constexpr (PHYS) Srr = fma(w * rp, rp, Srr);
    }

    // with another part of the row's sums: plus() of the parts of a row's four
    // lanes, ((0, 1), (2, 3)), gives the bits of sum4()
    __device__ __forceinline__ void plus(const CovSums &b)
    {
        Smm += b.Smm;
        Smr += b.Smr;
#pragma unroll
        for (int j = 0; j < L - 1; ++j) Smt[j] += b.Smt[j];
        if constexpr (PHYS) {
            Srr += b.Srr;
#pragma unroll
            for (int j = 0; j < L - 1; ++j) {
                Str[j] += b.Str[j];
#pragma unroll
                for (int q = 0; q <= j; ++q) Stt[j * LT + q] += b.Stt[j * LT + q];
            }
            prod *= b.prod;
            pexp += b.pexp;
        }
    }

    // over the four lanes of a row (jk_cov_sum)
    __device__ __forceinline__ void sum4()
    {
        Smm = jk_cov_sum(Smm);
        Smr = jk_cov_sum(Smr);
#pragma unroll
        for (int j = 0; j < L - 1; ++j) Smt[j] = jk_cov_sum(Smt[j]);
        if constexpr (PHYS) {
            Srr = jk_cov_sum(Srr);
#pragma unroll
            for (int j = 0; j < L - 1; ++j) {
                Str[j] = jk_cov_sum(Str[j]);
#pragma unroll
                for (int q = 0; q <= j; ++q) Stt[j * LT + q] = jk_cov_sum(Stt[j * LT + q]);
            }
            // mantissas in [1/2, 1): four of them stay far inside the range
            prod *= __shfl_xor(prod, 16, 64);
            prod *= __shfl_xor(prod, 32, 64);
            pexp += __shfl_xor(pexp, 16, 64);
            pexp += __shfl_xor(pexp, 32, 64);
        }
    }

    __device__ __forceinline__ double finish(const StarDev &st, const RowOrbit &o,
                                             const double2 *__restrict__ tab) const
    {
        return jk_row_finish<L, PHYS, false>(st, o.lam0, Smm, Smr, Srr, Smt, Str, Stt, prod, pexp,
                                             0.0, 0.0f, tab, nullptr);
    }
};

// r', sigma^2 (PHYS) or ivar and T per eigenvalue, and dt per epoch, to LDS
// (256 threads).
template <int L, bool PHYS>
__device__ __forceinline__ void jk_cov_stage_ep(const StarDev &st, double *s_ep)
{
    const int N = st.n;
    for (int q = threadIdx.x; q < N * (L + 2); q += 256) {
        const int v = q / N, i = q - v * N;
        s_ep[q] = v == 0 ? st.rp[i]
                         : (v == 1 ? (PHYS ? st.sig2[i] : st.ivar[i])
                                   : (v == L + 1 ? st.dt[i] : st.T[(size_t)(v - 2) * N + i]));
    }
}

// Full-covariance stars, FP64: 16 rows per wave (jk_cov_rotate), the
// workgroups striding over the rows so that each stages Q and the tables once.
// For L >= 7 two waves per SIMD are asked for (else 253 VGPRs and more, and one
// wave: 62689 rows x 8 epochs, L = 8 22.7 -> 15.9 us).
template <int L, bool PHYS>
__global__ __launch_bounds__(256, L >= 7 ? 2 : JK_ROW_WAVES(L)) void k_lnl_cov(const StarDev st, int64_t n,
                                                 const double *__restrict__ P,
                                                 const void *__restrict__ e_,
                                                 const void *__restrict__ om_,
                                                 const void *__restrict__ M0_,
                                                 const void *__restrict__ s_,
                                                 const int64_t *__restrict__ rows,
                                                 double *__restrict__ ll)
{
    __shared__ double2 s_tab[JK_TAB_LDS64];
    extern __shared__ double s_q[];
    const int N = st.n, pitch = jk_cov_pitch(N), K4 = (N + 3) / 4 * 4;
    double *s_ep = s_q + K4 * pitch;      // r', sigma^2 (PHYS) or ivar, T per eigenvalue
    for (int q = threadIdx.x; q < K4 * pitch; q += 256) {
        const int k = q / pitch, i = q - k * pitch;
        s_q[q] = k < N && i < N ? st.Qt[(size_t)i * N + k] : 0.0;
    }
    jk_cov_stage_ep<L, PHYS>(st, s_ep);
    const double *s_dt = s_ep + (L + 1) * N;
    jk_stage_tab<false>(s_tab);
    const int lane = threadIdx.x & 63, kq = lane >> 4;
    for (int64_t i0 = (int64_t)blockIdx.x * JK_COV_ROWS; i0 < n;
         i0 += (int64_t)gridDim.x * JK_COV_ROWS) {
        const int64_t i = i0 + (threadIdx.x >> 6) * 16 + (lane & 15);
        RowOrbit o;
        const bool valid =
            i < n && jk_row_orbit<PHYS>(st, rows ? rows[i] : i, P, e_, om_, M0_, s_, s_tab, o);
        jk_f64x4 acc[4];
        bool bad = false;
        jk_cov_rotate<false>(st, o, valid, s_tab, s_q, s_dt, acc, bad);
        if (__any(bad)) {
            // a row is bad when any of its epochs is
            const unsigned long long bw = __ballot(bad);
            bad = ((bw | bw >> 16 | bw >> 32 | bw >> 48) >> (lane & 15)) & 1;
            jk_cov_rotate<true>(st, o, valid, s_tab, s_q, s_dt, acc, bad);
        }
        // moments in the eigenbasis, a quarter of the eigenvalues per lane
        CovSums<L, PHYS> q;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (16 * t >= N) break;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ei = 16 * t + 4 * r + kq;
                if (ei >= N) continue;
                q.add(acc[t][r], ei, N, s_ep, o.s2);
            }
        }
        q.sum4();
        if (kq == 0 && i < n) ll[i] = valid ? q.finish(st, o, s_tab) : __builtin_nan("");
    }
}

// The rotated design values of one lane's row of N <= NL epochs, eigenvalue i
// in acc[i].  SAFE: with the bracketed Newton iteration; else returns whether
// the row needs it.
template <int NL, bool SAFE>
__device__ __forceinline__ bool jk_cov_rotate_lane(const StarDev &st, const RowOrbit &o,
                                                   const double2 *__restrict__ tab,
                                                   const double *s_q, const double *s_dt,
                                                   double acc[NL])
{
    const int N = st.n;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < NL; ++i) acc[i] = 0.0;
    for (int k = 0; k < N; ++k) {
        double w;
        float denb;
        const double m = jk_row_epoch<false, false, SAFE, true>(o, s_dt[k], 0.0, tab, w, denb, bad);
        const double *q = s_q + k * NL;
#pragma unroll
        for (int i0 = 0; i0 < NL; i0 += 8) {
            if (i0 >= N) break;
#pragma unroll
            for (int i = i0; i < i0 + 8; ++i) acc[i] = fma(q[i], m, acc[i]);
        }
    }
    return bad;
}

// Full-covariance stars of few epochs, N <= NL (jk_cov_lane), one lane per row:
// the rotation is N multiply-adds per epoch, its operands read by all lanes
// alike from LDS, in the order in which the matrix cores add (each rounded like
// an fma), and the sums go by the parts that the tile form's lanes hold.  A row's
// lnL is the same bits in either form.  Bound by the latency of one row's
// chain of solves up to a wave per SIMD (65536 rows), then by the vector units,
// with jitter and L >= 5 at one wave per SIMD for the parts' registers (two
// waves asked for spill them: 131072 x 8, L = 6 18 -> 22 us).
template <int L, bool PHYS, int NL>
__global__ __launch_bounds__(256) void k_lnl_cov_lane(const StarDev st, int64_t n,
                                                      const double *__restrict__ P,
                                                      const void *__restrict__ e_,
                                                      const void *__restrict__ om_,
                                                      const void *__restrict__ M0_,
                                                      const void *__restrict__ s_,
                                                      const int64_t *__restrict__ rows,
                                                      double *__restrict__ ll)
{
    __shared__ double2 s_tab[JK_TAB_LDS64];
    __shared__ double s_q[NL * NL];    // epoch-major, zero-padded
    __shared__ double s_ep[NL * (L + 2)];
    const int N = st.n;
    for (int q = threadIdx.x; q < N * NL; q += 256) {
        const int k = q / NL, i = q % NL;
        s_q[q] = i < N ? st.Qt[(size_t)i * N + k] : 0.0;
    }
    jk_cov_stage_ep<L, PHYS>(st, s_ep);
    const double *s_dt = s_ep + (L + 1) * N;
    jk_stage_tab<false>(s_tab);
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        RowOrbit o;
        if (!jk_row_orbit<PHYS>(st, rows ? rows[i] : i, P, e_, om_, M0_, s_, s_tab, o)) {
            ll[i] = __builtin_nan("");
            continue;
        }
        double acc[NL];
        if (jk_cov_rotate_lane<NL, false>(st, o, s_tab, s_q, s_dt, acc))
            jk_cov_rotate_lane<NL, true>(st, o, s_tab, s_q, s_dt, acc);
        CovSums<L, PHYS> half, sum;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            CovSums<L, PHYS> q;
#pragma unroll
            for (int j = g; j < NL; j += 4)
                if (j < N) q.add(acc[j], j, N, s_ep, o.s2);
            if (g & 1)
                half.plus(q);
            else
                half = q;
            if (g == 1) sum = half;
            if (g == 3) sum.plus(half);
        }
        ll[i] = sum.finish(st, o, s_tab);
    }
}

// Whether a launch takes one lane per row.  The tile form pays the orbit on
// four lanes per row and the finish on one lane of four, which few epochs do
// not outweigh once its waves (a row to every 4 lanes) fill the device, the
// sooner the larger L.  us, tile form -> this: 62689 rows, 4 epochs, L = 2 7.6 ->
// 6.6, L = 4 11.7 -> 6.8, L = 6 15.4 -> 7.9; 16 epochs, L = 4 15.4 -> 12.5, L = 6 19.9
// -> 15.5; 131072 rows, 16 epochs, L = 2 15.8 -> 14.3, L = 6 32.4 -> 28.5.
// Below the lines the tile form is ahead: 16384 rows, 16 epochs, L = 2 6.9 ->
// 11.0; 32768, 12 epochs, L = 5 8.6 -> 10.4; 62689, 16 epochs, L = 2 10.2 -> 11.7.  Up
// to 24 epochs for L >= 6 alone (131072 x 20 at L = 6 38.4 -> 35.0, L = 8 without
// jitter 52.0 -> 21.5): there the tile form's registers leave one or two waves
// per SIMD.
static bool jk_cov_lane(int64_t n, int N, int L)
{
    if (N <= 8) return n > (L <= 3 ? 49152 : (L <= 5 ? 36864 : 16384));
    if (N <= 16) return n > (L <= 3 ? 65536 : (L <= 5 ? 53248 : 32768));
    return N <= 24 && L >= 6 && n > 53248;
}

template <int L, bool PHYS>
static hipError_t launch_lnl_cov_t(const jk_star *st, int64_t n, const double *P, const void *e,
                                   const void *om, const void *M0, const void *s,
                                   const int64_t *rows, double *ll, hipStream_t stream)
{
    if (jk_cov_lane(n, st->dev.n, L)) {
        const int64_t blocks = std::min<int64_t>((n + 255) / 256, 1024);
        auto kernel = k_lnl_cov_lane<L, PHYS, 16>;
        if constexpr (L >= 6)
            if (st->dev.n > 16) kernel = k_lnl_cov_lane<L, PHYS, 24>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, stream, st->dev, n, P, e,
                           om, M0, s, rows, ll);
        return hipGetLastError();
    }
    // four workgroups per compute unit, then a stride: staging Q and the tables
    // costs as much as a few rows (2^18 rows x 40: 78 us with 4096 workgroups,
    // 75 with 1024; 100000 x 64: 75 and 66)
    const int64_t blocks = std::min<int64_t>((n + JK_COV_ROWS - 1) / JK_COV_ROWS, 1024);
    const size_t lds = sizeof(double) * jk_cov_lds_doubles(st->dev.n, L);
    hipLaunchKernelGGL((k_lnl_cov<L, PHYS>), dim3((unsigned)blocks), dim3(256), lds, stream,
                       st->dev, n, P, e, om, M0, s, rows, ll);
    return hipGetLastError();
}

static hipError_t launch_lnl_cov(const jk_star *st, int64_t n, const double *P, const void *e,
                                 const void *om, const void *M0, const void *s,
                                 const int64_t *rows, double *ll, hipStream_t stream)
{
    if (st->dev.n > JK_COV_NMAX) return hipErrorInvalidValue;
    const bool phys = st->dev.jitter_mode == JK_JITTER_PHYSICAL;
#define JK_CCASE(LL)                                                                           \
    case LL:                                                                                   \
        return phys ? launch_lnl_cov_t<LL, true>(st, n, P, e, om, M0, s, rows, ll, stream)     \
                    : launch_lnl_cov_t<LL, false>(st, n, P, e, om, M0, s, rows, ll, stream);
    switch (st->dev.L) {
        JK_CCASE(1)
        JK_CCASE(2)
        JK_CCASE(3)
        JK_CCASE(4)
        JK_CCASE(5)
        JK_CCASE(6)
        JK_CCASE(7)
        JK_CCASE(8)
    default:
        return hipErrorInvalidValue;
    }
#undef JK_CCASE
}

// Scatter launch over a device-resident index list: for j < *count,
// i = idx[j], ll[i] = lnL(row rows[i] or i).  Grid-stride, so the host does
// not need the count.
template <int L, bool PHYS>
__global__ __launch_bounds__(256, JK_ROW_WAVES(L)) void k_lnl_scatter_f64(const StarDev st,
                                                         const int64_t *__restrict__ count,
                                                         const int64_t *__restrict__ idx,
                                                         const double *__restrict__ P,
                                                         const void *__restrict__ e_,
                                                         const void *__restrict__ om_,
                                                         const void *__restrict__ M0_,
                                                         const void *__restrict__ s_,
                                                         const int64_t *__restrict__ rows,
                                                         double *__restrict__ ll)
{
    __shared__ double2 s_tab[JK_TAB_LDS64];
    jk_stage_tab<false>(s_tab);
    const int64_t cnt = *count;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < cnt; j += stride) {
        const int64_t i = idx[j];
        const int64_t r = rows ? rows[i] : i;
        ll[i] = jk_lnl_row<L, PHYS, false>(st, r, P, e_, om_, M0_, s_, s_tab);
    }
}

// Workgroups of a dense launch over n rows, one row per lane: up to 16384
// workgroups (2^22 rows), then a stride.
static int64_t jk_dense_blocks(int64_t n)
{
    const int64_t b = (n + 255) / 256;
    return b < 16384 ? (b < 1 ? 1 : b) : 16384;
}

// Entries of blockmax the FP64 launch over n rows of an N-epoch star writes.
static int64_t jk_lnl_partials(int64_t n, int N)
{
    const int R = jk_split_rows(n, N, false);
    return R ? (n + R - 1) / R : 4 * jk_dense_blocks(n);
}

template <int L, bool PHYS, bool MIXED>
static hipError_t launch_lnl_t(const jk_star *st, int64_t n, const double *P, const void *e,
                               const void *om, const void *M0, const void *s,
                               const int64_t *rows, double *ll, double *blockmax, float *bound,
                               hipStream_t stream)
{
    if (const int R = jk_split_rows(n, st->dev.n, MIXED)) {
        hipLaunchKernelGGL((k_lnl_split<L, PHYS, MIXED>), dim3((unsigned)((n + R - 1) / R)),
                           dim3(256), 0, stream, st->dev, n, R, P, e, om, M0, s, rows, ll,
                           blockmax, bound);
        return hipGetLastError();
    }
    const int64_t blocks = jk_dense_blocks(n);
    if constexpr (MIXED) {
        if constexpr (L == 2 || L == 3) {
            if (bound && st->dev.t0_one) {
                hipLaunchKernelGGL((k_lnl<L, PHYS, true, true, true>), dim3((unsigned)blocks),
                                   dim3(256), 0, stream, st->dev, n, P, e, om, M0, s, rows, ll,
                                   blockmax, bound);
                return hipGetLastError();
            }
        }
        if (bound) {
            hipLaunchKernelGGL((k_lnl<L, PHYS, true, true>), dim3((unsigned)blocks), dim3(256), 0,
                               stream, st->dev, n, P, e, om, M0, s, rows, ll, blockmax, bound);
            return hipGetLastError();
        }
    }
    if constexpr (!MIXED) {
        const bool lone = n <= JK_LONE_MAX_ROWS;
        if constexpr (L == 2 || L == 3) {
            // the constant offset as the first trend column (the usual v0)
            if (st->dev.t0_one) {
                hipLaunchKernelGGL((lone ? k_lnl<L, PHYS, false, false, true, true>
                                         : k_lnl<L, PHYS, false, false, true>),
                                   dim3((unsigned)blocks), dim3(256), 0, stream, st->dev, n, P, e,
                                   om, M0, s, rows, ll, blockmax, nullptr);
                return hipGetLastError();
            }
        }
        hipLaunchKernelGGL((lone ? k_lnl<L, PHYS, false, false, false, true>
                                 : k_lnl<L, PHYS, false, false>),
                           dim3((unsigned)blocks), dim3(256), 0, stream, st->dev, n, P, e, om, M0,
                           s, rows, ll, blockmax, nullptr);
    } else {
        hipLaunchKernelGGL((k_lnl<L, PHYS, true, false>), dim3((unsigned)blocks), dim3(256), 0,
                           stream, st->dev, n, P, e, om, M0, s, rows, ll, blockmax, nullptr);
    }
    return hipGetLastError();
}

template <bool MIXED>
static hipError_t launch_lnl_dispatch(const jk_star *st, int64_t n, const double *P, const void *e,
                                      const void *om, const void *M0, const void *s,
                                      const int64_t *rows, double *ll, double *bm, float *bd,
                                      hipStream_t stream)
{
    const bool phys = st->dev.jitter_mode == JK_JITTER_PHYSICAL;
#define JK_CASE(LL)                                                                                \
    case LL:                                                                                       \
        return phys                                                                                \
                   ? launch_lnl_t<LL, true, MIXED>(st, n, P, e, om, M0, s, rows, ll, bm, bd, stream) \
                   : launch_lnl_t<LL, false, MIXED>(st, n, P, e, om, M0, s, rows, ll, bm, bd,         \
                                                    stream);
    switch (st->dev.L) {
        JK_CASE(1)
        JK_CASE(2)
        JK_CASE(3)
        JK_CASE(4)
        JK_CASE(5)
        JK_CASE(6)
        JK_CASE(7)
        JK_CASE(8)
    default:
        return hipErrorInvalidValue;
    }
#undef JK_CASE
}

hipError_t jk_launch_lnl_f64(const jk_star *st, int64_t n, const double *P, const double *e,
                             const double *om, const double *M0, const double *s,
                             const int64_t *rows, double *ll, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    if (st->dev.Qt) return launch_lnl_cov(st, n, P, e, om, M0, s, rows, ll, stream);
    return launch_lnl_dispatch<false>(st, n, P, e, om, M0, s, rows, ll, nullptr, nullptr, stream);
}

hipError_t jk_launch_lnl_mixed(const jk_star *st, int64_t n, const double *P, const double *e,
                               const double *om, const double *M0, const double *s,
                               const int64_t *rows, double *ll, float *bound, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    return launch_lnl_dispatch<true>(st, n, P, e, om, M0, s, rows, ll, nullptr, bound, stream);
}


__global__ __launch_bounds__(256) void k_max_partial(const double *__restrict__ ll, int64_t n,
                                                     double *__restrict__ partials)
{
    __shared__ double red[4];
    double m = -INFINITY;
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride)
        m = jk_nanmax(m, ll[i]);
    m = wave_nanmax(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        partials[blockIdx.x] = jk_nanmax(jk_nanmax(red[0], red[1]), jk_nanmax(red[2], red[3]));
}

__global__ __launch_bounds__(256) void k_max_final(const double *__restrict__ partials, int np,
                                                   double *__restrict__ out)
{
    __shared__ double red[4];
    double m = -INFINITY;
    for (int i = threadIdx.x; i < np; i += 256) m = jk_nanmax(m, partials[i]);
    m = wave_nanmax(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) *out = jk_nanmax(jk_nanmax(red[0], red[1]), jk_nanmax(red[2], red[3]));
}

int jk_max_partials_count(int64_t n)
{
    int64_t b = (n + 255) / 256;
    if (b > 1024) b = 1024;
    if (b < 1) b = 1;
    return (int)b;
}

void jk_launch_max_partials(const double *ll, int64_t n, double *partials, int n_partials,
                            hipStream_t stream)
{
    hipLaunchKernelGGL(k_max_partial, dim3(n_partials), dim3(256), 0, stream, ll, n, partials);
}

hipError_t jk_launch_max(const double *ll, int64_t n, double *partials, int n_partials,
                         double *max_out, hipStream_t stream)
{
    hipLaunchKernelGGL(k_max_partial, dim3(n_partials), dim3(256), 0, stream, ll, n, partials);
    hipLaunchKernelGGL(k_max_final, dim3(1), dim3(256), 0, stream, partials, n_partials, max_out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// PCG64 uniforms and rejection.
// Thread g of a grid of T threads owns indices g, g + T, g + 2T, ...; its
// state starts at s_base (the state whose output is index 0) jumped by g
// with the 2^i table, then advances by the (A_T, D_T) jump per iteration.
// Waves step through 64-aligned index ranges, so one ballot word covers
// indices [64 w, 64 w + 64).
// ---------------------------------------------------------------------------
__device__ __forceinline__ u128 pcg_jump_table(u128 s, uint64_t k, u128 inc)
{
#pragma unroll 1
    for (int b = 0; k != 0; ++b, k >>= 1)
        if (k & 1) s = pcg_affine(s, c_jump.A[b], c_jump.D[b], inc);
    return s;
}

// State of thread g = blockIdx.x * 256 + threadIdx.x (256-thread workgroups):
// the workgroup's jump by blockIdx.x * 256 is the same for every lane, so its
// loop does not diverge; the lane's own jump by threadIdx.x is one step from
// the per-lane table.  Equal to pcg_jump_table(s, g, inc).
__device__ __forceinline__ u128 pcg_thread_start(u128 s, u128 inc)
{
    uint64_t k = blockIdx.x;
#pragma unroll 1
    for (int b = 8; k != 0; ++b, k >>= 1)
        if (k & 1) s = pcg_affine(s, c_jump.A[b], c_jump.D[b], inc);
    return pcg_affine(s, c_tid_A[threadIdx.x], c_tid_D[threadIdx.x], inc);
}

static int jk_rng_grid(int64_t n)
{
    int64_t b = (n + 256 * 16 - 1) / (256 * 16);
    if (b > 4096) b = 4096;
    if (b < 1) b = 1;
    return (int)b;
}

__global__ __launch_bounds__(256) void k_uniform(int64_t n, u128 s_base, u128 inc, u128 AT, u128 DT,
                                                 double *__restrict__ u)
{
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t T = (int64_t)gridDim.x * 256;
    u128 s = pcg_thread_start(s_base, inc);
    for (int64_t i = g; i < n; i += T) {
        u[i] = pcg_to_double(pcg_output(s));
        s = pcg_affine(s, AT, DT, inc);
    }
}

// Strides of the row loop whose loads the flag kernels issue together
// (k_seg_decide on 2^24 rows of ll + bound: 66 -> 51 us).
#define JK_FLAG_UNROLL 4

// The rejection test exp(x) > u of likelihood_helpers.py:108 for a uniform u
// on numpy's grid {k 2^-53} in [0, 1), evaluated exactly as written, but
// without the exp where it cannot decide anything: for x < -40 and u > 0,
// exp(x) <= exp(-40) < 4.3e-18 < 2^-53 <= u.  Most rows of a peaked
// likelihood lie that far below the maximum, so most waves skip the exp.
__device__ __forceinline__ bool jk_accept(double x, double u)
{
    bool keep = false;
    if (x >= -40.0 || u == 0.0) keep = exp(x) > u;
    return keep;
}

// Below this x = lnL - max no uniform, not even 0, passes the test: exp(x)
// is 0 in FP64 from x < -745.14 on.
#define JK_REJECT_FLOOR (-746.0)
// Marked rows among a wave's first 1024 above which k_reject_words walks the
// wave's words row by row instead of lane by lane.
#define JK_REJECT_DENSE 128

// The NaN-propagating maximum of an array's (a segment's) partials, in every thread of a
// 256-thread workgroup: each workgroup of the pass that uses it reduces the
// (at most 1024) partials itself, which is cheaper than a launch of its own.
__device__ __forceinline__ double jk_partials_max(const double *__restrict__ partials, int pb,
                                                  double *red)
{
    double m = -INFINITY;
    for (int i = threadIdx.x; i < pb; i += 256) m = jk_nanmax(m, partials[i]);
    m = wave_nanmax(m);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    return jk_nanmax(jk_nanmax(red[0], red[1]), jk_nanmax(red[2], red[3]));
}

// The maximum the rejection flags compare with: *llmax if given, else reduced
// from np partials and, by the first workgroup, left in *llmax_out.
__device__ __forceinline__ double jk_reject_max(const double *__restrict__ llmax,
                                                const double *__restrict__ partials, int np,
                                                double *__restrict__ llmax_out)
{
    __shared__ double red[4];
    if (llmax) return *llmax;
    const double mx = jk_partials_max(partials, np, red);
    if (blockIdx.x == 0 && threadIdx.x == 0) *llmax_out = mx;
    return mx;
}

// The rejection flags row by row, four rows per lane a grid stride apart: for
// up to JK_REJECT_ROWS_MAX rows, where one lane per 64 rows (k_reject_words)
// leaves most of the device idle while each lane walks its own rows.  Peaked
// / flat likelihood, this way against one lane per word: 2^12 rows 4.6 / 5.0
// against 12 / 24 us, 2^18 7.4 / 7.4 against 16 / 28, 2^20 12 / 13 against 16
// / 29, 2^21 19 / 20 against 17 / 36, 2^22 32 / 34 against 18 / 37.
#define JK_REJECT_ROWS_MAX ((int64_t)3 << 19)

__global__ __launch_bounds__(256) void k_reject_rows(const double *__restrict__ ll, int64_t n,
                                                     const double *__restrict__ llmax,
                                                     const double *__restrict__ partials, int np,
                                                     double *__restrict__ llmax_out, u128 s_base,
                                                     u128 inc, u128 AT, u128 DT,
                                                     uint64_t *__restrict__ mask)
{
    const double mx = jk_reject_max(llmax, partials, np, llmax_out);
    const int lane = threadIdx.x & 63;
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t T = (int64_t)gridDim.x * 256;
    double xs[JK_FLAG_UNROLL];
#pragma unroll
    for (int u = 0; u < JK_FLAG_UNROLL; ++u) {
        const int64_t i = g + u * T;
        xs[u] = i < n ? ll[i] - mx : -INFINITY;
    }
    u128 s = pcg_thread_start(s_base, inc);
#pragma unroll
    for (int u = 0; u < JK_FLAG_UNROLL; ++u) {
        const int64_t base = g - lane + u * T;     // the same for every lane of the wave
        if (base >= n) break;
        bool keep = false;
        if (xs[u] >= JK_REJECT_FLOOR) keep = jk_accept(xs[u], pcg_to_double(pcg_output(s)));
        const uint64_t word = __ballot(keep);
        if (lane == 0) mask[base >> 6] = word;
        if (u + 1 < JK_FLAG_UNROLL) s = pcg_affine(s, AT, DT, inc);
    }
}

// The rejection flags with one lane per 64-row mask word: lane g owns rows
// [64 g, 64 g + 64), so a wave owns 4096 contiguous rows.  First the wave
// marks, with coalesced loads and one ballot per 64 rows, the rows with
// x = lnL - max >= JK_REJECT_FLOOR, the only ones a uniform can accept:
// iteration k reads rows 64 k + lane of the wave's range, and its ballot is
// the candidate word of the wave's lane k.  Then each lane draws uniforms for
// the marked rows of its own word alone: the state of its first row is the
// workgroup's jump (the same for every lane, by the 2^i table from bit 14
// on: 256 lanes x 64 rows per workgroup) followed by the lane's own
// (A^64t, D_64t), and each marked row's state is reached from the previous
// one by one affine step per set bit of the gap.  Every row gets the uniform
// of its own index in the stream and the same jk_accept as a row-by-row pass,
// so the words are the same; a lane whose rows all lie far below the maximum
// (most, for a peaked likelihood) does no 128-bit arithmetic, where a
// row-by-row pass steps the LCG once per row (2^24 rows of a peaked
// likelihood: 46 us row by row, 33 us this way, 38 us with each lane reading
// its own 64 rows).
__global__ __launch_bounds__(256) void k_reject_words(const double *__restrict__ ll, int64_t n,
                                                      const double *__restrict__ llmax,
                                                      const double *__restrict__ partials, int np,
                                                      double *__restrict__ llmax_out,
                                                      u128 s_base, u128 inc,
                                                      uint64_t *__restrict__ mask)
{
    const double mx = jk_reject_max(llmax, partials, np, llmax_out);
    const int t = threadIdx.x, lane = t & 63;
    const int64_t g = (int64_t)blockIdx.x * 256 + t;
    const int64_t w0 = (g - lane) * 64;          // the wave's first row
    if (w0 >= n) return;                         // the whole wave
    const int64_t r0 = g * 64;
    // the workgroup's jump, the same for every lane: 256 lanes x 64 rows
    u128 s = s_base;
    uint64_t kb = blockIdx.x;
#pragma unroll 1
    for (int b = 14; kb != 0; ++b, kb >>= 1)
        if (kb & 1) s = pcg_affine(s, c_jump.A[b], c_jump.D[b], inc);
    // marks of the wave's words, sixteen loads in flight per lane before their
    // ballots; after the first sixteen words (1024 rows), a wave with many
    // rows in reach takes the row-by-row walk instead
    uint64_t cand = 0;
    bool dense = false;
    for (int k0 = 0; k0 < 64; k0 += 16) {
        double v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t r = w0 + 64 * (k0 + q) + lane;
            v[q] = r < n ? ll[r] : -INFINITY;
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const uint64_t bits = __ballot(v[q] - mx >= JK_REJECT_FLOOR);
            cand = lane == k0 + q ? bits : cand;
        }
        if (k0 == 0 && wave_sum_i64((int64_t)__popcll(cand)) > JK_REJECT_DENSE) {
            dense = true;
            break;
        }
    }
    uint64_t word = 0;
    if (dense) {
        // Many rows in reach (a flat likelihood): the wave walks its words in
        // order, lane L at row 64 k + L of word k, as a row-by-row pass does
        // with coalesced reads and one 64-row step of every state per word.
        // State of lane L at row L: the wave's jump by 4096 w (bits 12-13)
        // and the lane's (A^L, D_L).
        for (int b = 12, kw = t >> 6; kw != 0; ++b, kw >>= 1)
            if (kw & 1) s = pcg_affine(s, c_jump.A[b], c_jump.D[b], inc);
        s = pcg_affine(s, c_tid_A[lane], c_tid_D[lane], inc);
        const u128 A64 = c_jump.A[6], D64 = c_jump.D[6];
        for (int k0 = 0; k0 < 64; k0 += JK_FLAG_UNROLL) {
            double xv[JK_FLAG_UNROLL];
#pragma unroll
            for (int q = 0; q < JK_FLAG_UNROLL; ++q) {
                const int64_t r = w0 + 64 * (k0 + q) + lane;
                xv[q] = r < n ? ll[r] - mx : -INFINITY;
            }
#pragma unroll
            for (int q = 0; q < JK_FLAG_UNROLL; ++q) {
                bool keep = false;
                if (xv[q] >= JK_REJECT_FLOOR)
                    keep = jk_accept(xv[q], pcg_to_double(pcg_output(s)));
                const uint64_t wk = __ballot(keep);
                word = lane == k0 + q ? wk : word;
                s = pcg_affine(s, A64, D64, inc);
            }
        }
    } else if (cand != 0) {
        // Few: each lane draws the uniforms of its own marked rows.
        s = pcg_affine(s, c_tid64_A[t], c_tid64_D[t], inc);
        int p = 0;
        while (cand != 0) {
            const int j = __builtin_ctzll(cand);
            cand &= cand - 1;
            for (int d = j - p, b = 0; d != 0; ++b, d >>= 1)
                if (d & 1) s = pcg_affine(s, c_jump.A[b], c_jump.D[b], inc);
            p = j;
            if (jk_accept(ll[r0 + j] - mx, pcg_to_double(pcg_output(s)))) word |= 1ull << j;
        }
    }
    if (r0 < n) mask[g] = word;
}

// Rows to re-evaluate in FP64 after a mixed-precision pass: every row not
// below max - window, and every row when the maximum itself is not finite.
__global__ __launch_bounds__(256) void k_window_flags(const double *__restrict__ ll, int64_t n,
                                                      int64_t first,
                                                      const double *__restrict__ llmax,
                                                      double window,
                                                      uint64_t *__restrict__ mask)
{
    const int lane = threadIdx.x & 63;
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t T = (int64_t)gridDim.x * 256;
    const double mx = *llmax;
    const bool all = !isfinite(mx);
    const double thr = mx - window;
    for (int64_t base = g - lane; base < n; base += T) {
        const int64_t i = base + lane;
        const bool keep = i < n && i >= first && (all || !(ll[i] < thr));
        const uint64_t word = __ballot(keep);
        if (lane == 0) mask[base >> 6] = word;
    }
}

#define JK_WORDS_PER_BLOCK 4096   // 16 words per thread

// This thread's share of the set bits of a workgroup's words, its loads in
// flight together.
__device__ __forceinline__ int64_t jk_count_words(const uint64_t *__restrict__ mask, int64_t w0,
                                                  int64_t nwords)
{
    uint64_t v[JK_WORDS_PER_BLOCK / 256];
#pragma unroll
    for (int q = 0; q < JK_WORDS_PER_BLOCK / 256; ++q) {
        const int64_t w = w0 + q * 256 + threadIdx.x;
        v[q] = w < nwords ? mask[w] : 0ull;
    }
    int64_t c = 0;
#pragma unroll
    for (int q = 0; q < JK_WORDS_PER_BLOCK / 256; ++q) c += __popcll(v[q]);
    return c;
}

__global__ __launch_bounds__(256) void k_reject_bsum(const uint64_t *__restrict__ mask,
                                                     int64_t nwords, int64_t *__restrict__ bsum)
{
    __shared__ int64_t red[4];
    const int64_t w0 = (int64_t)blockIdx.x * JK_WORDS_PER_BLOCK;
    int64_t c = jk_count_words(mask, w0, nwords);
    c = wave_sum_i64(c);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) bsum[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(256) void k_reject_compact(const uint64_t *__restrict__ mask,
                                                        int64_t nwords,
                                                        const int64_t *__restrict__ bsum,
                                                        int nblocks, int64_t max_keep,
                                                        int64_t *__restrict__ idx_out,
                                                        int64_t *__restrict__ n_pass_out)
{
    __shared__ int64_t red[4];
    __shared__ int64_t s_off;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;

    // Offset of this block = sum of the counts of the blocks before it; block
    // 0 also publishes the total.
    int64_t c = 0;
    const int lim = blockIdx.x == 0 ? nblocks : (int)blockIdx.x;
    for (int b = threadIdx.x; b < lim; b += 256) c += bsum[b];
    c = wave_sum_i64(c);
    if (lane == 0) red[wid] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int64_t tot = red[0] + red[1] + red[2] + red[3];
        if (blockIdx.x == 0) {
            *n_pass_out = tot;
            s_off = 0;
        } else {
            s_off = tot;
        }
    }
    __syncthreads();
    const int64_t off = s_off;
    if (off >= max_keep) return;   // uniform across the block

    const int64_t w0 = (int64_t)blockIdx.x * JK_WORDS_PER_BLOCK + (int64_t)threadIdx.x * 16;
    uint64_t words[16];
    int64_t cnt = 0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int64_t w = w0 + q;
        words[q] = w < nwords ? mask[w] : 0ull;
        cnt += __popcll(words[q]);
    }
    // Exclusive block scan of cnt.
    const int64_t incl = wave_incl_scan_i64(cnt, lane);
    __syncthreads();
    if (lane == 63) red[wid] = incl;
    __syncthreads();
    int64_t pre = incl - cnt;
    for (int k = 0; k < wid; ++k) pre += red[k];
    int64_t rank = off + pre;
#pragma unroll 1
    for (int q = 0; q < 16 && rank < max_keep; ++q) {
        uint64_t word = words[q];
        while (word != 0ull && rank < max_keep) {
            const int bit = __builtin_ctzll(word);
            idx_out[rank++] = ((w0 + q) << 6) + bit;
            word &= word - 1ull;
        }
    }
}

int64_t jk_reject_mask_words(int64_t n) { return (n + 63) / 64; }
int64_t jk_reject_bsum_count(int64_t n)
{
    return (jk_reject_mask_words(n) + JK_WORDS_PER_BLOCK - 1) / JK_WORDS_PER_BLOCK;
}

// ---------------------------------------------------------------------------
// Host-side PCG64 jump arithmetic.
// ---------------------------------------------------------------------------
static u128 h_mul(u128 a, u128 b)
{
    unsigned __int128 x = ((unsigned __int128)a.hi << 64) | a.lo;
    unsigned __int128 y = ((unsigned __int128)b.hi << 64) | b.lo;
    unsigned __int128 z = x * y;
    u128 r;
    r.lo = (uint64_t)z;
    r.hi = (uint64_t)(z >> 64);
    return r;
}

static u128 h_add(u128 a, u128 b)
{
    unsigned __int128 x = ((unsigned __int128)a.hi << 64) | a.lo;
    unsigned __int128 y = ((unsigned __int128)b.hi << 64) | b.lo;
    unsigned __int128 z = x + y;
    u128 r;
    r.lo = (uint64_t)z;
    r.hi = (uint64_t)(z >> 64);
    return r;
}

static const u128 kPcgMult = {0x4385DF649FCCF645ULL, 0x2360ED051FC65DA4ULL};

// A^k and D_k = sum_{j<k} A^j (mod 2^128).
void jk_pcg_jump_coeffs(uint64_t k, u128 *A, u128 *D)
{
    u128 accA = {1, 0}, accD = {0, 0};
    u128 curA = kPcgMult, curD = {1, 0};
    const u128 one = {1, 0};
    while (k) {
        if (k & 1) {
            // acc <- cur o acc:  A = curA accA,  D = curA accD + curD
            accD = h_add(h_mul(curA, accD), curD);
            accA = h_mul(curA, accA);
        }
        // cur <- cur o cur:  D = curA curD + curD = (curA + 1) curD
        curD = h_mul(h_add(curA, one), curD);
        curA = h_mul(curA, curA);
        k >>= 1;
    }
    *A = accA;
    *D = accD;
}

static u128 h_jump(u128 s, u128 inc, uint64_t k)
{
    u128 A, D;
    jk_pcg_jump_coeffs(k, &A, &D);
    return h_add(h_mul(A, s), h_mul(D, inc));
}

hipError_t jk_upload_pcg_table(int device)
{
    PcgJump tab;
    for (int b = 0; b < 64; ++b) jk_pcg_jump_coeffs(1ull << b, &tab.A[b], &tab.D[b]);
    hipError_t err =
        hipMemcpyToSymbol(HIP_SYMBOL(c_jump), &tab, sizeof(tab), 0, hipMemcpyHostToDevice);
    if (err != hipSuccess) return err;
    u128 tA[256], tD[256];
    for (int t = 0; t < 256; ++t) jk_pcg_jump_coeffs((uint64_t)t, &tA[t], &tD[t]);
    err = hipMemcpyToSymbol(HIP_SYMBOL(c_tid_A), tA, sizeof(tA), 0, hipMemcpyHostToDevice);
    if (err != hipSuccess) return err;
    err = hipMemcpyToSymbol(HIP_SYMBOL(c_tid_D), tD, sizeof(tD), 0, hipMemcpyHostToDevice);
    if (err != hipSuccess) return err;
    for (int t = 0; t < 256; ++t) jk_pcg_jump_coeffs(64 * (uint64_t)t, &tA[t], &tD[t]);
    err = hipMemcpyToSymbol(HIP_SYMBOL(c_tid64_A), tA, sizeof(tA), 0, hipMemcpyHostToDevice);
    if (err != hipSuccess) return err;
    return hipMemcpyToSymbol(HIP_SYMBOL(c_tid64_D), tD, sizeof(tD), 0, hipMemcpyHostToDevice);
}

// The sin / cos grids of jk_sincos_tab and jk_sincos_tab_f32, and the log
// table of jk_log_tab, from 80-bit long double on the host rounded once to
// FP64 / FP32.
hipError_t jk_upload_sincos_table(int device)
{
    double2 tab[JK_TAB_N + 1];
    float2 tab32[JK_TAB_N + 1];
    for (int i = 0; i <= JK_TAB_N; ++i) {
        const long double g = (long double)i * (long double)JK_TAB_H;
        tab[i] = make_double2((double)sinl(g), (double)cosl(g));
        const long double g32 = (long double)i * (long double)JK_TAB_H32;
        tab32[i] = make_float2((float)sinl(g32), (float)cosl(g32));
    }
    double2 ltab[JK_LOG_TAB_N];
    for (int i = 0; i < JK_LOG_TAB_N; ++i) {
        const double R = (double)(1.0L / (1.0L + (i + 0.5L) / JK_LOG_TAB_N));
        ltab[i] = make_double2(R, (double)(-logl((long double)R)));
    }
    hipError_t err = hipMemcpyToSymbol(HIP_SYMBOL(g_sincos_tab), tab, sizeof(tab), 0,
                                       hipMemcpyHostToDevice);
    if (err != hipSuccess) return err;
    err = hipMemcpyToSymbol(HIP_SYMBOL(g_log_tab), ltab, sizeof(ltab), 0, hipMemcpyHostToDevice);
    if (err != hipSuccess) return err;
    return hipMemcpyToSymbol(HIP_SYMBOL(g_sincos_tab32), tab32, sizeof(tab32), 0,
                             hipMemcpyHostToDevice);
}

hipError_t jk_launch_uniform(u128 state, u128 inc, uint64_t offset, int64_t n, double *u,
                             hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    const int grid = jk_rng_grid(n);
    u128 AT, DT;
    jk_pcg_jump_coeffs((uint64_t)grid * 256, &AT, &DT);
    const u128 s_base = h_jump(state, inc, offset + 1);
    hipLaunchKernelGGL(k_uniform, dim3(grid), dim3(256), 0, stream, n, s_base, inc, AT, DT, u);
    return hipGetLastError();
}

// llmax: the maximum, or nullptr and it is reduced from np (at most 1024)
// partials and left in *llmax_out.
hipError_t jk_launch_reject(const double *ll, int64_t n, const double *llmax,
                            const double *partials, int np, double *llmax_out, u128 state,
                            u128 inc, uint64_t offset, int64_t max_keep, int64_t *idx_out,
                            int64_t *n_pass_out, uint64_t *mask, int64_t *bsum,
                            hipStream_t stream)
{
    const u128 s_base = h_jump(state, inc, offset + 1);
    const int64_t nwords = jk_reject_mask_words(n);
    const int64_t nb = jk_reject_bsum_count(n);
    if (n <= JK_REJECT_ROWS_MAX) {
        const unsigned grid = (unsigned)((n + 256 * JK_FLAG_UNROLL - 1) / (256 * JK_FLAG_UNROLL));
        u128 AT, DT;
        jk_pcg_jump_coeffs((uint64_t)grid * 256, &AT, &DT);
        hipLaunchKernelGGL(k_reject_rows, dim3(grid), dim3(256), 0, stream, ll, n, llmax, partials,
                           np, llmax_out, s_base, inc, AT, DT, mask);
    } else {
        hipLaunchKernelGGL(k_reject_words, dim3((unsigned)((nwords + 255) / 256)), dim3(256), 0,
                           stream, ll, n, llmax, partials, np, llmax_out, s_base, inc, mask);
    }
    hipLaunchKernelGGL(k_reject_bsum, dim3((unsigned)nb), dim3(256), 0, stream, mask, nwords, bsum);
    hipLaunchKernelGGL(k_reject_compact, dim3((unsigned)nb), dim3(256), 0, stream, mask, nwords, bsum,
                       (int)nb, max_keep, idx_out, n_pass_out);
    return hipGetLastError();
}

// FP64 lnL plus the rejection step of the same rows, with the maximum reduced
// inside the likelihood launch (one partial per wave).
int64_t jk_lnl_reject_scratch_bytes(int64_t n)
{
    // the most partials a launch over n rows writes, whatever its epochs
    int64_t parts = 4 * jk_dense_blocks(n);
    if (n <= JK_SPLIT_MAX_ROWS) parts = std::max(parts, n / JK_SPLIT_RMIN + 1);
    return (int64_t)sizeof(double) * (parts + 1024) +
           (int64_t)sizeof(uint64_t) * jk_reject_mask_words(n) +
           (int64_t)sizeof(int64_t) * jk_reject_bsum_count(n);
}

hipError_t jk_launch_lnl_reject_f64(const jk_star *st, int64_t n, const double *P, const double *e,
                                    const double *om, const double *M0, const double *s,
                                    const int64_t *rows, double *ll, u128 state, u128 inc,
                                    uint64_t offset, int64_t max_keep, int64_t *idx_out,
                                    int64_t *n_pass_out, double *llmax_out, void *scratch,
                                    hipStream_t stream)
{
    const int64_t parts = jk_lnl_partials(n, st->dev.n);
    double *partials = (double *)scratch;       // one per likelihood wave or workgroup
    double *partials2 = partials + parts;       // second level, at most 1024
    const double *level = partials;             // at most 1024 for the rejection step
    int64_t n_level = parts;
    uint64_t *mask = (uint64_t *)(partials2 + 1024);
    int64_t *bsum = (int64_t *)(mask + jk_reject_mask_words(n));
    hipError_t err;
    if (st->dev.Qt) {
        // full covariance: the partial maxima in a pass over ll
        err = launch_lnl_cov(st, n, P, e, om, M0, s, rows, ll, stream);
        if (err != hipSuccess) return err;
        level = partials2;
        n_level = jk_max_partials_count(n);
        jk_launch_max_partials(ll, n, partials2, (int)n_level, stream);
    } else {
        err = launch_lnl_dispatch<false>(st, n, P, e, om, M0, s, rows, ll, partials, nullptr,
                                         stream);
        if (err != hipSuccess) return err;
        if (parts > 1024) {
            level = partials2;
            n_level = jk_max_partials_count(parts);
            jk_launch_max_partials(partials, parts, partials2, (int)n_level, stream);
        }
    }
    return jk_launch_reject(ll, n, nullptr, level, (int)n_level, llmax_out, state, inc, offset,
                            max_keep, idx_out, n_pass_out, mask, bsum, stream);
}

template <int L, bool PHYS>
static void launch_scatter_t(const jk_star *st, const int64_t *count, const int64_t *idx, int grid,
                             const double *P, const void *e, const void *om, const void *M0,
                             const void *s, const int64_t *rows, double *ll, hipStream_t stream)
{
    hipLaunchKernelGGL((k_lnl_scatter_f64<L, PHYS>), dim3(grid), dim3(256), 0, stream, st->dev,
                       count, idx, P, e, om, M0, s, rows, ll);
}

int64_t jk_polish_scratch_bytes(int64_t n)
{
    return (int64_t)sizeof(double) * (jk_max_partials_count(n) + 1) +
           (int64_t)sizeof(uint64_t) * jk_reject_mask_words(n) +
           (int64_t)sizeof(int64_t) * (jk_reject_bsum_count(n) + n + 1);
}

hipError_t jk_launch_polish(const jk_star *st, int64_t n, const double *P, const double *e,
                            const double *om, const double *M0, const double *s,
                            const int64_t *rows, double *ll, double window, int64_t first,
                            void *scratch, int64_t *n_polished, hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    const int np = jk_max_partials_count(n);
    const int64_t nwords = jk_reject_mask_words(n);
    const int64_t nb = jk_reject_bsum_count(n);
    char *p = (char *)scratch;
    double *partials = (double *)p;
    double *mx = partials + np;
    uint64_t *mask = (uint64_t *)(mx + 1);
    int64_t *bsum = (int64_t *)(mask + nwords);
    int64_t *idx = bsum + nb;
    int64_t *count = n_polished;
    hipError_t err = jk_launch_max(ll, n, partials, np, mx, stream);
    if (err != hipSuccess) return err;
    const int grid = jk_rng_grid(n);
    hipLaunchKernelGGL(k_window_flags, dim3(grid), dim3(256), 0, stream, ll, n, first, mx, window,
                       mask);
    hipLaunchKernelGGL(k_reject_bsum, dim3((unsigned)nb), dim3(256), 0, stream, mask, nwords, bsum);
    hipLaunchKernelGGL(k_reject_compact, dim3((unsigned)nb), dim3(256), 0, stream, mask, nwords, bsum,
                       (int)nb, n, idx, count);
    int64_t sgrid = (n + 255) / 256;
    if (sgrid > 2048) sgrid = 2048;
    const bool phys = st->dev.jitter_mode == JK_JITTER_PHYSICAL;
#define JK_SCASE(LL)                                                                                 \
    case LL:                                                                                         \
        if (phys)                                                                                    \
            launch_scatter_t<LL, true>(st, count, idx, (int)sgrid, P, e, om, M0, s, rows, ll, stream); \
        else                                                                                         \
            launch_scatter_t<LL, false>(st, count, idx, (int)sgrid, P, e, om, M0, s, rows, ll, stream); \
        break;
    switch (st->dev.L) {
        JK_SCASE(1)
        JK_SCASE(2)
        JK_SCASE(3)
        JK_SCASE(4)
        JK_SCASE(5)
        JK_SCASE(6)
        JK_SCASE(7)
        JK_SCASE(8)
    default:
        return hipErrorInvalidValue;
    }
#undef JK_SCASE
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Up to JK_SEG_ARGS segment descriptors to the device as kernel arguments:
// they are copied into the launch's argument buffer at the call, so the host
// array need not outlive it and nothing waits.
// ---------------------------------------------------------------------------
struct SegArgs {
    uint64_t w[JK_SEG_ARGS * sizeof(SegDev) / sizeof(uint64_t)];
};

__global__ __launch_bounds__(256) void k_put_segs(uint64_t *__restrict__ dst, const SegArgs a,
                                                  int n_words)
{
    for (int i = threadIdx.x; i < n_words; i += 256) dst[i] = a.w[i];
}

hipError_t jk_put_segs(SegDev *dst, const SegDev *src, int n, hipStream_t stream)
{
    SegArgs a;
    if (n > JK_SEG_ARGS) return hipErrorInvalidValue;
    memcpy(a.w, src, sizeof(SegDev) * n);
    hipLaunchKernelGGL(k_put_segs, dim3(1), dim3(256), 0, stream, (uint64_t *)dst, a,
                       (int)(n * sizeof(SegDev) / sizeof(uint64_t)));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Many stars per launch: one workgroup per work item (star, row tile), or per
// part of an item's rows, in the items' order; it reads the star's constants
// through scalar loads and evaluates its rows one lane per row.  The hardware
// dispatcher hands the entries out: a persistent grid that took them from a
// device counter paid about 10 ns per fetch (one address, so one after
// another: 20 us before the last of 2048 workgroups had its first item, as
// much for the fetches that found the queue empty) and a launch to clear the
// counter, more than staging the tables again costs.
// ---------------------------------------------------------------------------
// Entries [first, end) of a launch, each work item as 1 << lg_parts parts: one
// workgroup per entry, or (CAPPED) the caller's most workgroups, each taking
// every gridDim.x-th entry.  An instance of its own, since the loop over the
// entries costs the other registers (L = 4 with jitter, FP64: 126 -> 163 VGPRs).
struct WorkSplit {
    int64_t first, end;
    unsigned lg_parts;
};

// The rows [lo, hi) that entry q takes of its item's n_rows: parts of whole
// workgroup passes.
__device__ __forceinline__ void jk_split_item(const WorkSplit &ws, int64_t q, int n_rows, int &lo,
                                              int &hi)
{
    lo = 0;
    hi = n_rows;
    if (ws.lg_parts) {
        const unsigned parts = 1u << ws.lg_parts, part = (unsigned)q & (parts - 1), bd = blockDim.x;
        const int64_t passes = (n_rows + (int64_t)bd - 1) / bd;
        const int64_t chunk = ((passes + parts - 1) >> ws.lg_parts) * bd;
        lo = (int)std::min<int64_t>(n_rows, part * chunk);
        hi = (int)std::min<int64_t>(n_rows, (part + 1) * chunk);
    }
}

// Parts per item: two, four or eight where that leaves at most 2 grid entries
// (grid: 8 workgroups per CU unless the caller says otherwise), so that few
// items still fill the chip and end together.  Whole items from the counter ->
// parts from the dispatcher, 2048 rows per item: 40 items (FP64, 3 to 12
// epochs, L = 2) 67 -> 27 us, 500 82 -> 37, 2400 155 -> 132; mixed, 3 to 64
// epochs, L = 3: 40 items 210 -> 28, 600 268 -> 122, 8192 1425 -> 1411.  More
// parts than that cost more than they level out: 2400 FP64 items in 8 parts
// 240 us.  A capped launch splits for the cap.
// grid < 0: -grid workgroups fill the device; grid > 0: the caller's cap, which
// is then what items are split for.
#define JK_ITEM_LAUNCH ((int64_t)1 << 23)   // entries per launch (x 256 threads < 2^32)
static unsigned jk_item_parts(int64_t n_items, int grid)
{
    unsigned lg = 0;
    while (lg < 3 && (n_items << (lg + 1)) <= 2 * std::abs((int64_t)grid)) ++lg;
    return lg;
}

// Parts per item of a pruned launch: two or four where that leaves at most a
// quarter of grid (512 entries).  An item's survivors are gathered to fill
// waves, and a part has fewer of them: each part ends on waves of a few lanes
// that walk all the star's epochs.  Against a persistent grid of whole items,
// live thresholds (the star's maximum - 40), 2048 rows per item, L = 2 to 5, 24 to
// 150 epochs, FP64, geometric mean (worst), for whole items, two parts, four:
// 1024 items 1.14 (0.92), 0.97 (0.66), 0.76 (0.47); 512 1.54 (1.18), 1.44
// (0.93), 1.12 (0.73); 256 1.91, 2.10 (1.49), 1.80 (1.09); 128 1.88, 2.51, 2.62.
// With no survivors parts only help: 1024 items 1.21, 1.26, 1.25; 512
// 1.66, 1.87, 1.90.
static unsigned jk_prune_parts(int64_t n_items, int grid)
{
    return std::min(2u, jk_item_parts(n_items, grid / 8));
}

// The end of the launch that starts at ws.first, and its workgroups (cap: 0 for
// none).
static unsigned jk_item_launch(int64_t entries, int cap, WorkSplit &ws)
{
    ws.end = cap ? entries : std::min(entries, ws.first + JK_ITEM_LAUNCH);
    return (unsigned)std::min(cap ? cap : ws.end - ws.first, JK_ITEM_LAUNCH);
}

// One row of a mixed-precision batched launch: in FP64 with error bound 0
// for a star whose table slot is marked exact (jk_batch_set_exact; a star
// whose rows nearly all land within the settling margin of its maximum, so
// that mixed values would be re-evaluated anyway), else in mixed precision
// with its bound.  The branch is uniform over a work item.
template <int L, bool PHYS, int U = 2>
__device__ __forceinline__ double jk_lnl_row_sel(const StarDev &st, int64_t r,
                                                 const double *__restrict__ P,
                                                 const void *__restrict__ e_,
                                                 const void *__restrict__ om_,
                                                 const void *__restrict__ M0_,
                                                 const void *__restrict__ s_,
                                                 const double2 *__restrict__ tab, float *bnd)
{
    if (st.exact) {
        *bnd = 0.0f;
        return jk_lnl_row<L, PHYS, false>(st, r, P, e_, om_, M0_, s_, tab);
    }
    return jk_lnl_row<L, PHYS, true, false, true, false, false, true, U>(st, r, P, e_, om_, M0_,
                                                                         s_, tab, bnd);
}

// Slot `slot` of a star table evaluated in FP64 (exact != 0) or as the launch
// asks (jk_batch_set_exact); a kernel, so that it is ordered on the stream and
// reads no host memory after it returns.
__global__ void k_set_exact(StarDev *stars, int slot, int exact) { stars[slot].exact = exact; }

template <int L, bool PHYS, bool MIXED, bool BOUND, bool CAPPED>
__global__ __launch_bounds__(256, JK_ROW_WAVES(L)) void k_lnl_batch(const StarDev *__restrict__ stars,
                                                   const jk_work_item *__restrict__ items,
                                                   WorkSplit ws,
                                                   const double *__restrict__ P,
                                                   const void *__restrict__ e_,
                                                   const void *__restrict__ om_,
                                                   const void *__restrict__ M0_,
                                                   const void *__restrict__ s_,
                                                   const int64_t *__restrict__ rows,
                                                   double *__restrict__ ll,
                                                   float *__restrict__ bound)
{
    __shared__ double2 s_tab[MIXED ? JK_TAB_LDS : JK_TAB_LDS64];
    if (CAPPED) jk_stage_tab<MIXED>(s_tab);
    for (int64_t q0 = ws.first + blockIdx.x; q0 < ws.end; q0 += gridDim.x) {
        const jk_work_item w = items[q0 >> ws.lg_parts];
        int lo, hi;
        jk_split_item(ws, q0, w.n_rows, lo, hi);
        if (!CAPPED) {
            if (lo >= hi) return;
            jk_stage_tab<MIXED>(s_tab);
        }
        const StarDev &st = stars[w.star];
        for (int j = lo + threadIdx.x; j < hi; j += blockDim.x) {
            const int64_t q = w.row_begin + j;
            const int64_t r = rows ? rows[q] : q;
            if constexpr (BOUND) {
                float b;
                ll[w.out_offset + j] = jk_lnl_row_sel<L, PHYS>(st, r, P, e_, om_, M0_, s_, s_tab, &b);
                bound[w.out_offset + j] = b;
            } else if constexpr (MIXED) {
                ll[w.out_offset + j] =
                    st.exact ? jk_lnl_row<L, PHYS, false>(st, r, P, e_, om_, M0_, s_, s_tab)
                             : jk_lnl_row<L, PHYS, true, false, false, false, false, true>(
                                   st, r, P, e_, om_, M0_, s_, s_tab);
            } else {
                ll[w.out_offset + j] = jk_lnl_row<L, PHYS, false>(st, r, P, e_, om_, M0_, s_, s_tab);
            }
        }
        if (!CAPPED) return;
    }
}

hipError_t jk_launch_set_exact(const jk_batch *b, int slot, int exact, hipStream_t stream)
{
    hipLaunchKernelGGL(k_set_exact, dim3(1), dim3(1), 0, stream, b->d_stars, slot, exact ? 1 : 0);
    return hipGetLastError();
}

template <int L, bool PHYS, bool MIXED>
static void launch_batch_t(const jk_batch *b, int64_t n_items, const jk_work_item *items,
                           const double *P, const void *e, const void *om, const void *M0,
                           const void *s, const int64_t *rows, double *ll, float *bound,
                           int block, int grid, hipStream_t stream)
{
    WorkSplit ws{0, 0, jk_item_parts(n_items, grid)};
    const int64_t entries = n_items << ws.lg_parts;
    const bool capped = grid > 0 && entries > grid;
    for (; ws.first < entries; ws.first = ws.end) {
        const dim3 blocks(jk_item_launch(entries, capped ? grid : 0, ws));
        if (MIXED && bound)
            hipLaunchKernelGGL((capped ? k_lnl_batch<L, PHYS, MIXED, MIXED, true>
                                       : k_lnl_batch<L, PHYS, MIXED, MIXED, false>),
                               blocks, dim3(block), 0, stream, b->d_stars, items, ws, P, e, om, M0,
                               s, rows, ll, bound);
        else
            hipLaunchKernelGGL((capped ? k_lnl_batch<L, PHYS, MIXED, false, true>
                                       : k_lnl_batch<L, PHYS, MIXED, false, false>),
                               blocks, dim3(block), 0, stream, b->d_stars, items, ws, P, e, om, M0,
                               s, rows, ll, nullptr);
    }
}

template <bool MIXED>
static hipError_t launch_batch_dispatch(const jk_batch *b, int64_t n_items,
                                        const jk_work_item *items, const double *P,
                                        const void *e, const void *om, const void *M0,
                                        const void *s, const int64_t *rows, double *ll,
                                        float *bd, int block, int grid,
                                        hipStream_t stream)
{
    const bool phys = b->jitter_mode == JK_JITTER_PHYSICAL;
#define JK_BCASE(LL)                                                                              \
    case LL:                                                                                      \
        if (phys)                                                                                 \
            launch_batch_t<LL, true, MIXED>(b, n_items, items, P, e, om, M0, s, rows, ll, bd,      \
                                            block, grid, stream);                        \
        else                                                                                      \
            launch_batch_t<LL, false, MIXED>(b, n_items, items, P, e, om, M0, s, rows, ll, bd,     \
                                             block, grid, stream);                       \
        break;
    switch (b->L) {
        JK_BCASE(1)
        JK_BCASE(2)
        JK_BCASE(3)
        JK_BCASE(4)
        JK_BCASE(5)
        JK_BCASE(6)
        JK_BCASE(7)
        JK_BCASE(8)
    default:
        return hipErrorInvalidValue;
    }
#undef JK_BCASE
    return hipGetLastError();
}

hipError_t jk_launch_lnl_batch(const jk_batch *b, int precision, int64_t n_items,
                               const jk_work_item *items, const double *P, const void *e,
                               const void *om, const void *M0, const void *s,
                               const int64_t *rows, double *ll, float *bound, int block, int grid,
                               hipStream_t stream)
{
    if (n_items <= 0) return hipSuccess;
    if (precision == 0)
        return launch_batch_dispatch<false>(b, n_items, items, P, e, om, M0, s, rows, ll, nullptr,
                                            block, grid, stream);
    return launch_batch_dispatch<true>(b, n_items, items, P, e, om, M0, s, rows, ll, bound, block,
                                       grid, stream);
}

// ---------------------------------------------------------------------------
// Many stars per launch with pruning by an upper bound.  probes[k] holds star
// k's data on a subset S of its epochs.  The marginal likelihood factors as
// p(y) = p(y_S) p(y_rest | y_S), and the conditional covariance of y_rest is
// at least the noise covariance C_rest, so
//   lnL <= lnL_S - 1/2 sum_{n not in S} ln(2 pi sigma_n^2) = lnL_S + add,
// for every prior row (with jitter the variances only grow).  prune[k] =
// (thr, add): a row whose bound lnL_S (+ its mixed error bound) + add is
// finite and below thr gets that bound as its value and is not evaluated
// further (bound JK_BOUND_UPPER in mixed precision: the value is an upper
// bound on the row's lnL, nothing more, and the settling kernels treat it so); every other row is evaluated as in k_lnl_batch.  Rows
// are probed a chunk of blockDim at a time and the survivors are gathered in
// LDS over several chunks, so the full evaluations run on dense waves.  thr = -inf
// turns the probe off for the star.  n_full (optional, one entry per star)
// accumulates each star's rows evaluated in full.
// ---------------------------------------------------------------------------
#define JK_PRUNE_LIST 2048   // survivors held in LDS before their evaluation

template <int L, bool PHYS, bool MIXED, bool CAPPED>
__global__ __launch_bounds__(256, JK_PRUNE_WAVES(L, PHYS, MIXED))
                                                    void k_lnl_prune_batch(const StarDev *__restrict__ stars,
                                                         const StarDev *__restrict__ probes,
                                                         const double2 *__restrict__ prune,
                                                         const jk_work_item *__restrict__ items,
                                                         WorkSplit ws,
                                                         const double *__restrict__ P,
                                                         const void *__restrict__ e_,
                                                         const void *__restrict__ om_,
                                                         const void *__restrict__ M0_,
                                                         const void *__restrict__ s_,
                                                         double *__restrict__ ll,
                                                         float *__restrict__ bound,
                                                         unsigned long long *__restrict__ n_full)
{
    constexpr int U = JK_PRUNE_UNROLL(L, PHYS);   // of the mixed rows
    __shared__ int s_n;
    __shared__ int s_list[JK_PRUNE_LIST];
    __shared__ double2 s_tab[MIXED ? JK_TAB_LDS : JK_TAB_LDS64];
    if (CAPPED) jk_stage_tab<MIXED>(s_tab);
    for (int64_t q0 = ws.first + blockIdx.x; q0 < ws.end; q0 += gridDim.x) {
        const jk_work_item w = items[q0 >> ws.lg_parts];
        int lo, hi;
        jk_split_item(ws, q0, w.n_rows, lo, hi);
        if (!CAPPED) {
            if (lo >= hi) return;
            jk_stage_tab<MIXED>(s_tab);
        }
        const StarDev &st = stars[w.star];
        const double2 pr = prune[w.star];
        if (!(pr.x > -INFINITY)) {
            for (int j = lo + (int)threadIdx.x; j < hi; j += blockDim.x) {
                const int64_t r = w.row_begin + j;
                if constexpr (MIXED) {
                    float b;
                    ll[w.out_offset + j] =
                        jk_lnl_row_sel<L, PHYS, U>(st, r, P, e_, om_, M0_, s_, s_tab, &b);
                    bound[w.out_offset + j] = b;
                } else {
                    ll[w.out_offset + j] = jk_lnl_row<L, PHYS, false>(st, r, P, e_, om_, M0_, s_, s_tab);
                    if (bound) bound[w.out_offset + j] = 0.0f;
                }
            }
            if (n_full && threadIdx.x == 0)
                atomicAdd(n_full + w.star, (unsigned long long)(hi - lo));
            if (CAPPED) continue;
            return;
        }
        const StarDev &pb = probes[w.star];
        unsigned n_surv = 0;
        if (threadIdx.x == 0) s_n = 0;
        __syncthreads();
        for (int base = lo; base < hi; base += blockDim.x) {
            const int j = base + (int)threadIdx.x;
            if (j < hi) {
                const int64_t r = w.row_begin + j;
                double v;
                if constexpr (MIXED) {
                    float b;
                    v = jk_lnl_row<L, PHYS, true, false, true, false, false, true, U>(
                        pb, r, P, e_, om_, M0_, s_, s_tab, &b);
                    v += (double)b + pr.y;
                } else {
                    v = jk_lnl_row<L, PHYS, false>(pb, r, P, e_, om_, M0_, s_, s_tab);
                    // FP64 rounding of both evaluations, far below this slack
                    v += pr.y + 1e-9 * (1.0 + fabs(v));
                }
                if (isfinite(v) && v < pr.x) {
                    ll[w.out_offset + j] = v;
                    if (bound) bound[w.out_offset + j] = JK_BOUND_UPPER;
                } else {
                    s_list[atomicAdd(&s_n, 1)] = j;
                }
            }
            __syncthreads();
            // Survivors gather over chunks and are evaluated once another
            // chunk might overflow the list, or at the item's end: the full
            // evaluations then run on whole waves.
            const int ns = s_n;
            __syncthreads();   // every thread holds ns before the next append
            if (ns > JK_PRUNE_LIST - (int)blockDim.x || base + (int)blockDim.x >= hi) {
                n_surv += (unsigned)ns;
                for (int k = threadIdx.x; k < ns; k += blockDim.x) {
                    const int jj = s_list[k];
                    const int64_t r = w.row_begin + jj;
                    if constexpr (MIXED) {
                        float b;
                        ll[w.out_offset + jj] =
                            jk_lnl_row_sel<L, PHYS, U>(st, r, P, e_, om_, M0_, s_, s_tab, &b);
                        bound[w.out_offset + jj] = b;
                    } else {
                        ll[w.out_offset + jj] =
                            jk_lnl_row<L, PHYS, false>(st, r, P, e_, om_, M0_, s_, s_tab);
                        if (bound) bound[w.out_offset + jj] = 0.0f;
                    }
                }
                __syncthreads();   // every read of s_list before it is reset
                if (threadIdx.x == 0) s_n = 0;
                __syncthreads();
            }
        }
        if (n_full && threadIdx.x == 0 && n_surv)
            atomicAdd(n_full + w.star, (unsigned long long)n_surv);
        if (!CAPPED) return;
    }
}

template <int L, bool PHYS, bool MIXED>
static void launch_prune_t(const jk_batch *b, const jk_batch *pb, const double2 *prune,
                           int64_t n_items, const jk_work_item *items, const double *P,
                           const void *e, const void *om, const void *M0, const void *s,
                           double *ll, float *bound, unsigned long long *n_full, int block,
                           int grid, hipStream_t stream)
{
    WorkSplit ws{0, 0, jk_prune_parts(n_items, grid)};
    const int64_t entries = n_items << ws.lg_parts;
    const bool capped = grid > 0 && entries > grid;
    for (; ws.first < entries; ws.first = ws.end) {
        const dim3 blocks(jk_item_launch(entries, capped ? grid : 0, ws));
        hipLaunchKernelGGL((capped ? k_lnl_prune_batch<L, PHYS, MIXED, true>
                                   : k_lnl_prune_batch<L, PHYS, MIXED, false>),
                           blocks, dim3(block), 0, stream, b->d_stars, pb->d_stars, prune, items,
                           ws, P, e, om, M0, s, ll, bound, n_full);
    }
}

hipError_t jk_launch_lnl_prune_batch(const jk_batch *b, const jk_batch *pb, const double *prune,
                                     int precision, int64_t n_items, const jk_work_item *items,
                                     const double *P, const void *e, const void *om,
                                     const void *M0, const void *s, double *ll, float *bound,
                                     unsigned long long *n_full, int block, int grid,
                                     hipStream_t stream)
{
    if (n_items <= 0) return hipSuccess;
    const bool phys = b->jitter_mode == JK_JITTER_PHYSICAL;
    const double2 *pr = reinterpret_cast<const double2 *>(prune);
#define JK_PCASE(LL)                                                                              \
    case LL:                                                                                      \
        if (precision == 1) {                                                                     \
            if (phys)                                                                             \
                launch_prune_t<LL, true, true>(b, pb, pr, n_items, items, P, e, om, M0, s, ll,     \
                                               bound, n_full, block, grid, stream);      \
            else                                                                                  \
                launch_prune_t<LL, false, true>(b, pb, pr, n_items, items, P, e, om, M0, s, ll,    \
                                                bound, n_full, block, grid, stream);     \
        } else {                                                                                  \
            if (phys)                                                                             \
                launch_prune_t<LL, true, false>(b, pb, pr, n_items, items, P, e, om, M0, s, ll,    \
                                                bound, n_full, block, grid, stream);     \
            else                                                                                  \
                launch_prune_t<LL, false, false>(b, pb, pr, n_items, items, P, e, om, M0, s, ll,   \
                                                 bound, n_full, block, grid, stream);    \
        }                                                                                         \
        break;
    switch (b->L) {
        JK_PCASE(1)
        JK_PCASE(2)
        JK_PCASE(3)
        JK_PCASE(4)
        JK_PCASE(5)
        JK_PCASE(6)
        JK_PCASE(7)
        JK_PCASE(8)
    default:
        return hipErrorInvalidValue;
    }
#undef JK_PCASE
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Segmented rejection: the steps of jk_launch_reject with blockIdx.y picking
// the segment.  Blocks past a segment's extent exit at once.
// ---------------------------------------------------------------------------
#define JK_SEG_MAX_BLOCKS 1024

__global__ __launch_bounds__(256) void k_seg_max_partial(const double *__restrict__ ll,
                                                         const SegDev *__restrict__ segs,
                                                         double *__restrict__ partials, int pb)
{
    __shared__ double red[4];
    const SegDev sg = segs[blockIdx.y];
    double m = -INFINITY;
    const int64_t stride = (int64_t)pb * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < sg.n; i += stride)
        m = jk_nanmax(m, ll[sg.off + i]);
    m = wave_nanmax(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        partials[(int64_t)blockIdx.y * pb + blockIdx.x] =
            jk_nanmax(jk_nanmax(red[0], red[1]), jk_nanmax(red[2], red[3]));
}

__global__ __launch_bounds__(64) void k_seg_max_final(const double *__restrict__ partials, int pb,
                                                      double *__restrict__ llmax)
{
    double m = -INFINITY;
    for (int i = threadIdx.x; i < pb; i += 64) m = jk_nanmax(m, partials[(int64_t)blockIdx.x * pb + i]);
    m = wave_nanmax(m);
    if (threadIdx.x == 0) llmax[blockIdx.x] = m;
}

// Every workgroup reduces its segment's maximum from the partials (one launch
// less: 96 segments of 50000 rows with their likelihood 334 -> 311 us, 8 of
// 20000 117 -> 98); the segment's first one writes it.
// zero_u (optional): zero_u[segment] is set to 1 when one of the segment's
// uniforms is exactly 0 (probability 2^-53 per row), the one case settling
// with a margin below 746 leaves open.
__global__ __launch_bounds__(256) void k_seg_flags(const double *__restrict__ ll,
                                                   const SegDev *__restrict__ segs,
                                                   const double *__restrict__ partials, int pb,
                                                   double *__restrict__ llmax, u128 AT, u128 DT,
                                                   uint64_t *__restrict__ mask,
                                                   int64_t *__restrict__ zero_u)
{
    __shared__ double red[4];
    const SegDev sg = segs[blockIdx.y];
    const double mx = jk_partials_max(partials + (int64_t)blockIdx.y * pb, pb, red);
    if (blockIdx.x == 0 && threadIdx.x == 0) llmax[blockIdx.y] = mx;
    const int lane = threadIdx.x & 63;
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t T = (int64_t)gridDim.x * 256;
    if (g - lane >= sg.n) return;
    u128 s = pcg_thread_start(sg.s_base, sg.inc);
    for (int64_t base0 = g - lane; base0 < sg.n; base0 += JK_FLAG_UNROLL * T) {
        // the loads of JK_FLAG_UNROLL strides first
        double xs[JK_FLAG_UNROLL];
#pragma unroll
        for (int u = 0; u < JK_FLAG_UNROLL; ++u) {
            const int64_t i = base0 + u * T + lane;
            xs[u] = i < sg.n ? ll[sg.off + i] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < JK_FLAG_UNROLL; ++u) {
            const int64_t base = base0 + u * T;     // the same for every lane of the wave
            if (base >= sg.n) break;
            bool keep = false;
            if (base + lane < sg.n) {
                const double uu = pcg_to_double(pcg_output(s));
                keep = jk_accept(xs[u] - mx, uu);
                if (zero_u != nullptr && uu == 0.0) zero_u[blockIdx.y] = 1;
            }
            const uint64_t word = __ballot(keep);
            if (lane == 0) mask[sg.mask_off + (base >> 6)] = word;
            s = pcg_affine(s, AT, DT, sg.inc);
        }
    }
}

// With n_settled_out, the segment's results that later launches of a settling
// sequence no longer change are written too: the rows of both its lists and the
// settled maximum.
__global__ __launch_bounds__(256) void k_seg_bsum(const SegDev *__restrict__ segs,
                                                  const uint64_t *__restrict__ mask,
                                                  int64_t *__restrict__ bsum,
                                                  const int64_t *__restrict__ count1 = nullptr,
                                                  const int64_t *__restrict__ count2 = nullptr,
                                                  const double *__restrict__ llmax = nullptr,
                                                  int64_t *__restrict__ n_settled_out = nullptr,
                                                  double *__restrict__ llmax_out = nullptr)
{
    __shared__ int64_t red[4];
    const SegDev sg = segs[blockIdx.y];
    if (n_settled_out && blockIdx.x == 0 && threadIdx.x == 0) {
        n_settled_out[blockIdx.y] = count1[blockIdx.y] + count2[blockIdx.y];
        llmax_out[blockIdx.y] = llmax[blockIdx.y];
    }
    if ((int64_t)blockIdx.x >= sg.nb) return;
    const int64_t nwords = (sg.n + 63) / 64;
    const int64_t w0 = (int64_t)blockIdx.x * JK_WORDS_PER_BLOCK;
    int64_t c = jk_count_words(mask + sg.mask_off, w0, nwords);
    c = wave_sum_i64(c);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) bsum[sg.bsum_off + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(256) void k_seg_compact(const SegDev *__restrict__ segs,
                                                     const uint64_t *__restrict__ mask,
                                                     const int64_t *__restrict__ bsum,
                                                     int64_t *__restrict__ idx_out,
                                                     int64_t *__restrict__ n_pass_out)
{
    __shared__ int64_t red[4];
    __shared__ int64_t s_off;
    const SegDev sg = segs[blockIdx.y];
    if ((int64_t)blockIdx.x >= sg.nb) return;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t nwords = (sg.n + 63) / 64;
    int64_t c = 0;
    const int64_t lim = blockIdx.x == 0 ? sg.nb : (int64_t)blockIdx.x;
    for (int64_t b = threadIdx.x; b < lim; b += 256) c += bsum[sg.bsum_off + b];
    c = wave_sum_i64(c);
    if (lane == 0) red[wid] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        const int64_t tot = red[0] + red[1] + red[2] + red[3];
        if (blockIdx.x == 0) {
            n_pass_out[blockIdx.y] = tot;
            s_off = 0;
        } else {
            s_off = tot;
        }
    }
    __syncthreads();
    const int64_t off = s_off;
    if (off >= sg.max_keep) return;
    const int64_t w0 = (int64_t)blockIdx.x * JK_WORDS_PER_BLOCK + (int64_t)threadIdx.x * 16;
    uint64_t words[16];
    int64_t cnt = 0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int64_t w = w0 + q;
        words[q] = w < nwords ? mask[sg.mask_off + w] : 0ull;
        cnt += __popcll(words[q]);
    }
    const int64_t incl = wave_incl_scan_i64(cnt, lane);
    __syncthreads();
    if (lane == 63) red[wid] = incl;
    __syncthreads();
    int64_t pre = incl - cnt;
    for (int k = 0; k < wid; ++k) pre += red[k];
    int64_t rank = off + pre;
#pragma unroll 1
    for (int q = 0; q < 16 && rank < sg.max_keep; ++q) {
        uint64_t word = words[q];
        while (word != 0ull && rank < sg.max_keep) {
            const int bit = __builtin_ctzll(word);
            idx_out[sg.idx_off + rank++] = ((w0 + q) << 6) + bit;
            word &= word - 1ull;
        }
    }
}

int jk_seg_flag_blocks(int64_t max_n)
{
    int64_t b = (max_n + 256 * 16 - 1) / (256 * 16);
    if (b > JK_SEG_MAX_BLOCKS) b = JK_SEG_MAX_BLOCKS;
    if (b < 1) b = 1;
    return (int)b;
}

__global__ __launch_bounds__(256) void k_fill_i64(int64_t *__restrict__ p, int n, int64_t v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

hipError_t jk_launch_reject_batch(const double *ll, int n_seg, const SegDev *d_segs,
                                  int64_t max_n, int64_t max_nb, double *partials, int pb,
                                  uint64_t *mask, int64_t *bsum, int64_t *idx_out,
                                  int64_t *n_pass_out, double *llmax_out, hipStream_t stream,
                                  int64_t *zero_u)
{
    if (n_seg <= 0) return hipSuccess;
    const int fb = jk_seg_flag_blocks(max_n);
    u128 AT, DT;
    jk_pcg_jump_coeffs((uint64_t)fb * 256, &AT, &DT);
    if (zero_u)
        hipLaunchKernelGGL(k_fill_i64, dim3((n_seg + 255) / 256), dim3(256), 0, stream, zero_u,
                           n_seg, (int64_t)0);
    hipLaunchKernelGGL(k_seg_max_partial, dim3(pb, n_seg), dim3(256), 0, stream, ll, d_segs,
                       partials, pb);
    hipLaunchKernelGGL(k_seg_flags, dim3(fb, n_seg), dim3(256), 0, stream, ll, d_segs, partials,
                       pb, llmax_out, AT, DT, mask, zero_u);
    hipLaunchKernelGGL(k_seg_bsum, dim3((unsigned)max_nb, n_seg), dim3(256), 0, stream, d_segs,
                       mask, bsum, nullptr, nullptr, nullptr, nullptr, nullptr);
    hipLaunchKernelGGL(k_seg_compact, dim3((unsigned)max_nb, n_seg), dim3(256), 0, stream, d_segs,
                       mask, bsum, idx_out, n_pass_out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Lists of rows to re-evaluate in FP64.  Their order does not matter (each row
// is evaluated by itself and written to its own place), so the kernels that
// pick the rows append them to the segment's list as they find them: a wave
// gathers its rows in LDS and claims room for up to JK_APPEND_CAP of them with
// one atomic, its workgroup for the rest.  Flag words with a block-count and an ordered compaction pass
// took two launches and a pass over the words more (2^21 rows: 7 + 6.5 + 6 us
// for each of four lists; 6 to 12 us this way).
// ---------------------------------------------------------------------------
#define JK_APPEND_CAP 512

struct WaveAppend {
    int64_t *buf;      // the wave's JK_APPEND_CAP entries of LDS
    int n;             // entries held, the same in every lane
};

__device__ __forceinline__ void jk_append_flush(WaveAppend &w, int64_t *__restrict__ list,
                                                int64_t *__restrict__ count)
{
    const int lane = threadIdx.x & 63;
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd((unsigned long long *)count, (unsigned long long)w.n);
    base = __shfl(base, 0, 64);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int q = lane; q < w.n; q += 64) list[base + q] = w.buf[q];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    w.n = 0;
}

// Every lane of the wave: appends i where keep is set.
__device__ __forceinline__ void jk_append(WaveAppend &w, bool keep, int64_t i,
                                          int64_t *__restrict__ list,
                                          int64_t *__restrict__ count)
{
    const uint64_t word = __ballot(keep);
    if (word == 0) return;
    const int lane = threadIdx.x & 63;
    if (keep) w.buf[w.n + __popcll(word & ((1ull << lane) - 1ull))] = i;
    w.n += __popcll(word);
    if (w.n > JK_APPEND_CAP - 64) jk_append_flush(w, list, count);
}

// What the workgroup's four waves still hold, with one atomic for all of them
// (an atomic per wave on the segment's one counter took 20 us for 2048 waves).
// Every wave of the workgroup, once, at the end.
__device__ __forceinline__ void jk_append_end(WaveAppend &w, int64_t *__restrict__ list,
                                              int64_t *__restrict__ count)
{
    __shared__ int held[4];
    __shared__ unsigned long long base;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) held[wid] = w.n;
    __syncthreads();
    const int total = held[0] + held[1] + held[2] + held[3];
    if (total == 0) return;
    if (threadIdx.x == 0)
        base = atomicAdd((unsigned long long *)count, (unsigned long long)total);
    __syncthreads();
    int64_t at = (int64_t)base;
    for (int k = 0; k < wid; ++k) at += held[k];
    for (int q = lane; q < w.n; q += 64) list[at + q] = w.buf[q];
}

// FP64 values as unsigned integers in the same order, every NaN above all
// numbers, 0 below: the maximum of re-evaluated rows by integer atomics.
__device__ __forceinline__ unsigned long long jk_max_key(double v)
{
    if (v != v) return ~0ull;
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : b | (1ull << 63);
}

__device__ __forceinline__ double jk_max_of_key(unsigned long long k)
{
    if (k == ~0ull) return __builtin_nan("");
    if (k == 0ull) return -INFINITY;
    return __longlong_as_double((long long)((k >> 63) ? k & ~(1ull << 63) : ~k));
}

__device__ __forceinline__ void jk_wave_max_key(double v, bool some, unsigned long long *key)
{
    unsigned long long k = some ? jk_max_key(v) : 0ull;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_xor(k, off, 64);
        k = o > k ? o : k;
    }
    if ((threadIdx.x & 63) == 0 && k != 0ull) atomicMax(key, k);
}

// Segmented FP64 re-evaluation window (jk_polish_f64 per segment): flags,
// the segmented compaction above, then a scatter of FP64 lnL over each
// segment's selected entries.
__global__ __launch_bounds__(256) void k_seg_window_flags(const double *__restrict__ ll,
                                                          const SegDev *__restrict__ segs,
                                                          const double *__restrict__ llmax,
                                                          double window,
                                                          uint64_t *__restrict__ mask)
{
    const SegDev sg = segs[blockIdx.y];
    const int lane = threadIdx.x & 63;
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t T = (int64_t)gridDim.x * 256;
    if (g - lane >= sg.n) return;
    const double mx = llmax[blockIdx.y];
    const bool all = !isfinite(mx);
    const double thr = mx - window;
    for (int64_t base = g - lane; base < sg.n; base += T) {
        const int64_t i = base + lane;
        const bool keep = i < sg.n && i >= sg.first && (all || !(ll[sg.off + i] < thr));
        const uint64_t word = __ballot(keep);
        if (lane == 0) mask[sg.mask_off + (base >> 6)] = word;
    }
}

// Padded exclusive prefix of the per-segment counts: cum[s] = sum over t < s
// of count[t] rounded up to a multiple of 64, so that a wavefront of the
// scatter below never straddles two segments.  One workgroup of 256; cum is
// its LDS or device memory (the scatter scans up to JK_SCAN_SEGS segments
// itself, a launch of one workgroup scans more).
#define JK_SCAN_SEGS 64

__device__ __forceinline__ void jk_count_scan(const int64_t *__restrict__ count, int n_seg,
                                              int64_t *cum)
{
    __shared__ int64_t wsum[4];
    const int per = (n_seg + 255) / 256;
    const int lo = min((int)threadIdx.x * per, n_seg);
    const int hi = min(lo + per, n_seg);
    int64_t mine = 0;
    for (int i = lo; i < hi; ++i) mine += (count[i] + 63) & ~(int64_t)63;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t incl = wave_incl_scan_i64(mine, lane);
    if (lane == 63) wsum[wid] = incl;
    __syncthreads();
    int64_t run = incl - mine;
    for (int k = 0; k < wid; ++k) run += wsum[k];
    for (int i = lo; i < hi; ++i) {
        cum[i] = run;
        run += (count[i] + 63) & ~(int64_t)63;
    }
    if (threadIdx.x == 255) cum[n_seg] = run;
    __syncthreads();
}

__global__ __launch_bounds__(256) void k_seg_count_scan(const int64_t *__restrict__ count,
                                                        int n_seg, int64_t *__restrict__ cum)
{
    jk_count_scan(count, n_seg, cum);
}

// The segment of padded position j0: the last one that starts at or before it.
__device__ __forceinline__ int jk_seg_of(const int64_t *__restrict__ cum, int n_seg, int64_t j0)
{
    int lo = 0, hi = n_seg;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cum[mid] <= j0) lo = mid; else hi = mid;
    }
    return lo;
}

// Most padded waves of a scatter that take the split evaluation, 16 rows to a
// workgroup (with 8 or 32 the same within 1 us), for a table of L parameters
// whose longest star has N epochs: what the split saves grows with the epochs
// that one lane would walk alone, what it costs with the rows, and with more
// workgroups than the compute units hold at once (the LDS of one grows with L)
// it falls behind.  The FP64 re-evaluations around a maximum are a few hundred
// rows.  One lane per row minus the split, us, L = 2 with jitter: N = 5: 4000
// rows -2; N = 12: 300 2.8, 4000 -0.7; N = 24: 2000 5.7, 12000 -1.7; N = 40: 6000
// 7.7, 16000 -0.8; N = 100: 1000 29, 12000 22, 16000 16, 20000 2, 30000 -4; N = 200: 20000 24.
// L = 6: N = 12: 300 2.7, 4000 -2; N = 24: 2000 6.2, 8000 -3; N = 100: 8000 27,
// 12000 22, 16000 -3, 30000 -52.
// (16 as a constant also leaves the one-lane half its own registers: with the
// rows per workgroup chosen on the device, <3, true> spilled two and <2, false>
// took 121 VGPRs instead of 97.)
#define JK_SPLIT_SCATTER_R 16
static int jk_split_scatter_waves(int N, int L)
{
    return std::min(std::max(4 * (N - 8), 0), L <= 3 ? 320 : 192);
}

// Workgroups of the scatter: at least 4 for each wave of the split.
#define JK_SCATTER_GRID 2048

// FP64 re-evaluation of every segment's selected entries as one flat list
// spread over the whole grid: wavefront w takes padded positions
// [64 w, 64 w + 64), all in one segment (found by binary search in cum and
// made wave-uniform, so the star's constants stay in scalar loads).
template <int L, bool PHYS>
__global__ __launch_bounds__(256, JK_ROW_WAVES(L)) void k_seg_scatter_f64(const StarDev *__restrict__ stars,
                                                         const SegDev *__restrict__ segs,
                                                         int n_seg, int split_waves,
                                                         const int64_t *__restrict__ count,
                                                         const int64_t *__restrict__ cum_in,
                                                         const int64_t *__restrict__ idx,
                                                         unsigned long long *__restrict__ key,
                                                         const double *__restrict__ P,
                                                         const void *__restrict__ e_,
                                                         const void *__restrict__ om_,
                                                         const void *__restrict__ M0_,
                                                         const void *__restrict__ s_,
                                                         const int64_t *__restrict__ rows,
                                                         double *__restrict__ ll,
                                                         float *__restrict__ bound)
{
    __shared__ double2 s_tab[JK_TAB_LDS64];
    __shared__ SplitLds<L, PHYS, false> sh;
    __shared__ int64_t s_cum[JK_SCAN_SEGS + 1];
    const int lane = threadIdx.x & 63;
    const int64_t *cum = cum_in;
    if (!cum_in) {
        jk_count_scan(count, n_seg, s_cum);
        cum = s_cum;
    }
    const int64_t total_waves = cum[n_seg] >> 6;
    if (total_waves <= split_waves) {
        // Few rows: each 64 positions over 64 / R workgroups, a row's epochs
        // over many lanes (jk_rows_split; the same bits).
        constexpr int R = JK_SPLIT_SCATTER_R;
        const int sw = jk_split_wave(blockIdx.x), sl = jk_split_lane(sw),
                  row = jk_split_row(sl, R);
        const int64_t j0 = (int64_t)blockIdx.x * R;
        if (j0 >= total_waves * 64) return;
        jk_stage_tab<false>(s_tab);
        const int sidx = __builtin_amdgcn_readfirstlane(jk_seg_of(cum, n_seg, j0));
        const SegDev &sg = segs[sidx];
        const int64_t local = j0 - cum[sidx] + row;
        const bool some = row < R && local < count[sidx];
        const int64_t p = some ? idx[sg.idx_off + local] : 0, q = sg.row0 + p;
        const double v = jk_rows_split<L, PHYS, false>(
            stars[sg.star], R, sw, some ? (rows ? rows[q] : q) : -1, P, e_, om_, M0_, s_, s_tab,
            sh, nullptr);
        if (some && sl < R) {
            ll[sg.off + p] = v;
            if (bound) bound[sg.off + p] = 0.0f;
        }
        if (key && sl < 64) jk_wave_max_key(v, some && sl < R, key + sidx);
        return;
    }
    jk_stage_tab<false>(s_tab);
    const int64_t wstride = (int64_t)gridDim.x * (blockDim.x >> 6);
    for (int64_t w = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
         w < total_waves; w += wstride) {
        const int64_t j0 = w << 6;
        const int sidx = __builtin_amdgcn_readfirstlane(jk_seg_of(cum, n_seg, j0));
        const SegDev &sg = segs[sidx];
        const int64_t local = j0 - cum[sidx] + lane;
        const bool some = local < count[sidx];
        double v = 0.0;
        if (some) {
            const int64_t p = idx[sg.idx_off + local];
            const int64_t q = sg.row0 + p;
            const int64_t r = rows ? rows[q] : q;
            v = jk_lnl_row<L, PHYS, false>(stars[sg.star], r, P, e_, om_, M0_, s_, s_tab);
            ll[sg.off + p] = v;
            if (bound) bound[sg.off + p] = 0.0f;
        }
        if (key) jk_wave_max_key(v, some, key + sidx);
    }
}

template <int L, bool PHYS>
static void launch_seg_scatter_t(const jk_batch *b, int n_seg, const SegDev *d_segs,
                                 const int64_t *count, const int64_t *cum, const int64_t *idx,
                                 unsigned long long *key, const double *P, const void *e,
                                 const void *om, const void *M0, const void *s,
                                 const int64_t *rows, double *ll, float *bound,
                                 hipStream_t stream)
{
    hipLaunchKernelGGL((k_seg_scatter_f64<L, PHYS>), dim3(JK_SCATTER_GRID), dim3(256), 0, stream,
                       b->d_stars, d_segs, n_seg,
                       jk_split_scatter_waves(
                           __atomic_load_n(&b->max_epochs, __ATOMIC_RELAXED), L),
                       count, cum, idx, key, P, e, om, M0, s, rows, ll, bound);
}

// FP64 re-evaluation of every segment's list idx (counts in count) as one flat
// launch; bound entries of re-evaluated rows are set to zero, and key (if
// given) receives each segment's maximum over them (jk_max_key).
static hipError_t launch_seg_scatter(const jk_batch *b, int n_seg, const SegDev *d_segs,
                                     const int64_t *count, int64_t *cum, const int64_t *idx,
                                     const double *P, const double *e, const double *om,
                                     const double *M0, const double *s, const int64_t *rows,
                                     double *ll, float *bound, hipStream_t stream,
                                     unsigned long long *key = nullptr)
{
    if (n_seg > JK_SCAN_SEGS)
        hipLaunchKernelGGL(k_seg_count_scan, dim3(1), dim3(256), 0, stream, count, n_seg, cum);
    else
        cum = nullptr;
    const bool phys = b->jitter_mode == JK_JITTER_PHYSICAL;
#define JK_SCASE2(LL)                                                                             \
    case LL:                                                                                      \
        if (phys)                                                                                 \
            launch_seg_scatter_t<LL, true>(b, n_seg, d_segs, count, cum, idx, key, P, e, om, M0,   \
                                           s, rows, ll, bound, stream);                           \
        else                                                                                      \
            launch_seg_scatter_t<LL, false>(b, n_seg, d_segs, count, cum, idx, key, P, e, om, M0,  \
                                            s, rows, ll, bound, stream);                          \
        break;
    switch (b->L) {
        JK_SCASE2(1)
        JK_SCASE2(2)
        JK_SCASE2(3)
        JK_SCASE2(4)
        JK_SCASE2(5)
        JK_SCASE2(6)
        JK_SCASE2(7)
        JK_SCASE2(8)
    default:
        return hipErrorInvalidValue;
    }
#undef JK_SCASE2
    return hipGetLastError();
}

hipError_t jk_launch_polish_batch(const jk_batch *b, int n_seg, const SegDev *d_segs,
                                  int64_t max_n, int64_t max_nb, double *partials, int pb,
                                  uint64_t *mask, int64_t *bsum, int64_t *idx, double *llmax,
                                  int64_t *cum, const double *P, const double *e, const double *om,
                                  const double *M0, const double *s, const int64_t *rows,
                                  double *ll, double window, int64_t *n_polished,
                                  hipStream_t stream)
{
    if (n_seg <= 0) return hipSuccess;
    const int fb = jk_seg_flag_blocks(max_n);
    hipLaunchKernelGGL(k_seg_max_partial, dim3(pb, n_seg), dim3(256), 0, stream, ll, d_segs,
                       partials, pb);
    hipLaunchKernelGGL(k_seg_max_final, dim3(n_seg), dim3(64), 0, stream, partials, pb, llmax);
    hipLaunchKernelGGL(k_seg_window_flags, dim3(fb, n_seg), dim3(256), 0, stream, ll, d_segs, llmax,
                       window, mask);
    hipLaunchKernelGGL(k_seg_bsum, dim3((unsigned)max_nb, n_seg), dim3(256), 0, stream, d_segs,
                       mask, bsum, nullptr, nullptr, nullptr, nullptr, nullptr);
    hipLaunchKernelGGL(k_seg_compact, dim3((unsigned)max_nb, n_seg), dim3(256), 0, stream, d_segs,
                       mask, bsum, idx, n_polished);
    return launch_seg_scatter(b, n_seg, d_segs, n_polished, cum, idx, P, e, om, M0, s, rows, ll,
                              nullptr, stream);
}

// ---------------------------------------------------------------------------
// Settling a mixed-precision lnL buffer for the rejection step
// (jk_settle_batch).  Per segment, with B the per-row bounds on
// |lnL(mixed) - lnL(FP64)| (0 for rows already FP64):
//   1. lo = max(ll - B) is a lower bound on the FP64 maximum; a row with
//      ll + B >= lo could be the maximum: re-evaluate it in FP64 (B := 0).
//      So is a row with ll + B >= lo - 40 and B > 1e-3 (k_seg_shell_list).
//      A NaN anywhere makes lo NaN and every unsettled row is re-evaluated.
//   2. mx = max(ll) is then the FP64 maximum.
//   3. u = the row's numpy uniform (the stream the rejection step draws); a
//      row whose decision exp(x - mx) > u differs between x = ll - B and
//      x = ll + B is re-evaluated in FP64 (B := 0).
// Afterwards exp(ll - mx) > u holds for exactly the rows for which it holds
// with every row's FP64 likelihood, and every row within 40 of mx is within
// 1e-3 of its FP64 lnL.
// ---------------------------------------------------------------------------
// lo = max(ll - b) over the rows that bound the maximum from below (b >= 0), in
// partials, and (partials2 given) the maximum over the rows no settling
// re-evaluates (b = 0) in partials2.  The first workgroup of a segment clears
// the counters of the passes that follow.
__global__ __launch_bounds__(256) void k_seg_lo_partial(const double *__restrict__ ll,
                                                        const float *__restrict__ bound,
                                                        const SegDev *__restrict__ segs,
                                                        double *__restrict__ partials,
                                                        double *__restrict__ partials2, int pb,
                                                        int64_t *__restrict__ count1,
                                                        int64_t *__restrict__ count2,
                                                        unsigned long long *__restrict__ key)
{
    __shared__ double red[4], red2[4];
    const SegDev sg = segs[blockIdx.y];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        count1[blockIdx.y] = 0;
        if (count2) count2[blockIdx.y] = 0;
        if (key) key[blockIdx.y] = 0ull;
    }
    double m = -INFINITY, m2 = -INFINITY;
    const int64_t stride = (int64_t)pb * 256;
    for (int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x; i0 < sg.n;
         i0 += JK_FLAG_UNROLL * stride) {
        float bs[JK_FLAG_UNROLL];
        double xs[JK_FLAG_UNROLL];
#pragma unroll
        for (int u = 0; u < JK_FLAG_UNROLL; ++u) {
            const int64_t i = i0 + u * stride;
            bs[u] = i < sg.n ? bound[sg.off + i] : -1.0f;
            xs[u] = i < sg.n ? ll[sg.off + i] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < JK_FLAG_UNROLL; ++u) {
            // an upper-bound row gives no lower bound on the maximum
            if (!(bs[u] < 0.0f)) {
                m = jk_nanmax(m, xs[u] - (double)bs[u]);
                if (!(bs[u] > 0.0f)) m2 = jk_nanmax(m2, xs[u]);
            }
        }
    }
    m = wave_nanmax(m);
    if (partials2) m2 = wave_nanmax(m2);
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = m;
        red2[threadIdx.x >> 6] = m2;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int64_t o = (int64_t)blockIdx.y * pb + blockIdx.x;
        partials[o] = jk_nanmax(jk_nanmax(red[0], red[1]), jk_nanmax(red[2], red[3]));
        if (partials2)
            partials2[o] = jk_nanmax(jk_nanmax(red2[0], red2[1]), jk_nanmax(red2[2], red2[3]));
    }
}

// Rows the settling re-evaluates besides the shell of the maximum: those that
// may lie within JK_LIVE_WINDOW of it (rows with a non-negligible chance of
// acceptance, exp(-40) < 4.3e-18) and whose bound exceeds JK_LIVE_TOL, so
// that after settling every such row is within JK_LIVE_TOL of its FP64 lnL.
#define JK_LIVE_WINDOW 40.0
#define JK_LIVE_TOL 1e-3f

// The list kernels below share a frame: the segment's level from its partials,
// then strides of the grid with the loads of JK_FLAG_UNROLL of them together.
// ROW(x, b, i): whether row i with value x and bound b goes on the list.
#define JK_LIST_ROWS(NEED_X, ROW)                                                              \
    __shared__ int64_t s_buf[4][JK_APPEND_CAP];                                                \
    WaveAppend wa{s_buf[threadIdx.x >> 6], 0};                                                 \
    const int lane = threadIdx.x & 63;                                                         \
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;                                 \
    const int64_t T = (int64_t)gridDim.x * 256;                                                \
    int64_t *list = idx + sg.idx_off, *cnt = count + blockIdx.y;                               \
    for (int64_t base0 = g - lane; base0 < sg.n; base0 += JK_FLAG_UNROLL * T) {                \
        double xs[JK_FLAG_UNROLL];                                                             \
        float bs[JK_FLAG_UNROLL];                                                              \
        _Pragma("unroll") for (int u = 0; u < JK_FLAG_UNROLL; ++u) {                           \
            const int64_t i = base0 + u * T + lane;                                            \
            xs[u] = NEED_X && i < sg.n ? ll[sg.off + i] : 0.0;                                 \
            bs[u] = i < sg.n ? bound[sg.off + i] : 0.0f;                                       \
        }                                                                                      \
        _Pragma("unroll") for (int u = 0; u < JK_FLAG_UNROLL; ++u) {                           \
            const int64_t i = base0 + u * T + lane;                                            \
            const double x = xs[u];                                                            \
            const float b = bs[u];                                                             \
            jk_append(wa, i < sg.n && (ROW), i, list, cnt);                                    \
        }                                                                                      \
    }                                                                                          \
    jk_append_end(wa, list, cnt)

__global__ __launch_bounds__(256) void k_seg_shell_list(const double *__restrict__ ll,
                                                        const float *__restrict__ bound,
                                                        const SegDev *__restrict__ segs,
                                                        const double *__restrict__ partials, int pb,
                                                        int64_t *__restrict__ count,
                                                        int64_t *__restrict__ idx)
{
    __shared__ double red[4];
    const SegDev sg = segs[blockIdx.y];
    if ((int64_t)blockIdx.x * 256 >= sg.n) return;
    const double l0 = jk_partials_max(partials + (int64_t)blockIdx.y * pb, pb, red);
    // could be the maximum; or within JK_LIVE_WINDOW of it with a bound above
    // JK_LIVE_TOL (an upper-bound row: x bounds it from above only)
    JK_LIST_ROWS(true, b > 0.0f ? (!(x + (double)b < l0) ||
                                   (b > JK_LIVE_TOL && !(x + (double)b < l0 - JK_LIVE_WINDOW)))
                                : (b < 0.0f && !(x < l0 - JK_LIVE_WINDOW)));
}

// The FP64 maximum of a settled segment: over the rows that were FP64 before
// (partials2) and those the settling re-evaluated (key).  A row left with a
// bound lies below lo, and so does not hold it.
__device__ __forceinline__ double jk_settled_max(const double *__restrict__ partials2, int pb,
                                                 const unsigned long long *__restrict__ key,
                                                 double *red)
{
    return jk_nanmax(jk_partials_max(partials2 + (int64_t)blockIdx.y * pb, pb, red),
                     jk_max_of_key(key[blockIdx.y]));
}

__global__ __launch_bounds__(256) void k_seg_uncertain_list(const double *__restrict__ ll,
                                                            const float *__restrict__ bound,
                                                            const SegDev *__restrict__ segs,
                                                            const double *__restrict__ partials2,
                                                            int pb,
                                                            const unsigned long long *__restrict__ key,
                                                            u128 AT, u128 DT,
                                                            int64_t *__restrict__ count,
                                                            int64_t *__restrict__ idx)
{
    __shared__ double red[4];
    __shared__ int64_t s_buf[4][JK_APPEND_CAP];
    const SegDev sg = segs[blockIdx.y];
    if ((int64_t)blockIdx.x * 256 >= sg.n) return;
    const double mx = jk_settled_max(partials2, pb, key, red);
    const bool live = !(mx != mx);     // a NaN maximum rejects every row anyway
    WaveAppend wa{s_buf[threadIdx.x >> 6], 0};
    const int lane = threadIdx.x & 63;
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t T = (int64_t)gridDim.x * 256;
    u128 s = pcg_thread_start(sg.s_base, sg.inc);
    for (int64_t base = g - lane; base < sg.n; base += T) {
        const int64_t i = base + lane;
        bool keep = false;
        if (i < sg.n) {
            const double uu = pcg_to_double(pcg_output(s));
            const float bf = bound[sg.off + i];
            if (live && bf > 0.0f) {
                const double x = ll[sg.off + i];
                const double b = fma((double)bf, 1e-6, (double)bf) + 1e-12;
                keep = jk_accept(x - b - mx, uu) != jk_accept(x + b - mx, uu);
            } else if (live && bf < 0.0f) {
                // an upper bound decides a rejection only
                keep = jk_accept(ll[sg.off + i] - mx, uu);
            }
        }
        jk_append(wa, keep, i, idx + sg.idx_off, count + blockIdx.y);
        s = pcg_affine(s, AT, DT, sg.inc);
    }
    jk_append_end(wa, idx + sg.idx_off, count + blockIdx.y);
}

__global__ void k_seg_add_counts(const int64_t *__restrict__ a, int64_t *__restrict__ b, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] += a[i];
}

hipError_t jk_launch_settle_batch(const jk_batch *b, int n_seg, const SegDev *d_segs,
                                  int64_t max_n, double *partials, int pb, int64_t *idx,
                                  unsigned long long *key, int64_t *cum, int64_t *count1,
                                  const double *P, const double *e, const double *om,
                                  const double *M0, const double *s, const int64_t *rows,
                                  double *ll, float *bound, int64_t *n_settled,
                                  hipStream_t stream)
{
    if (n_seg <= 0) return hipSuccess;
    const int fb = jk_seg_flag_blocks(max_n);
    double *partials2 = partials + (size_t)pb * n_seg;
    // 1. the rows that could hold the FP64 maximum
    hipLaunchKernelGGL(k_seg_lo_partial, dim3(pb, n_seg), dim3(256), 0, stream, ll, bound, d_segs,
                       partials, partials2, pb, count1, n_settled, key);
    hipLaunchKernelGGL(k_seg_shell_list, dim3(fb, n_seg), dim3(256), 0, stream, ll, bound, d_segs,
                       partials, pb, count1, idx);
    hipError_t err = launch_seg_scatter(b, n_seg, d_segs, count1, cum, idx, P, e, om, M0, s, rows,
                                        ll, bound, stream, key);
    if (err != hipSuccess) return err;
    // 2. the rows whose decision the bound leaves open
    u128 AT, DT;
    jk_pcg_jump_coeffs((uint64_t)fb * 256, &AT, &DT);
    hipLaunchKernelGGL(k_seg_uncertain_list, dim3(fb, n_seg), dim3(256), 0, stream, ll, bound,
                       d_segs, partials2, pb, key, AT, DT, n_settled, idx);
    err = launch_seg_scatter(b, n_seg, d_segs, n_settled, cum, idx, P, e, om, M0, s, rows, ll,
                             bound, stream);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(k_seg_add_counts, dim3((n_seg + 255) / 256), dim3(256), 0, stream, count1,
                       n_settled, n_seg);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Settling for every future uniform (the iterative rejection loop redraws
// the uniforms of all rows each round).  For each segment's new rows:
//   1. lo = max(floor, max(ll - B)) is a lower bound on the FP64 maximum of
//      the segment (floor: the FP64 maximum of the rows settled before);
//   2. every new row with ll + B >= lo - margin is re-evaluated in FP64.
// A row left in mixed precision then has lnL(FP64) <= ll + B < max - margin,
// and so does ll itself: with margin >= 746, exp(x - max) is 0 for both, so
// the row is rejected whatever its uniform, and it cannot be the maximum.
// The maximum row itself is always re-evaluated.  A NaN in lo re-evaluates
// every new row still in mixed precision.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_seg_live_list(const double *__restrict__ ll,
                                                       const float *__restrict__ bound,
                                                       const SegDev *__restrict__ segs,
                                                       const double *__restrict__ partials, int pb,
                                                       double margin, int64_t *__restrict__ count,
                                                       int64_t *__restrict__ idx)
{
    __shared__ double red[4];
    const SegDev sg = segs[blockIdx.y];
    if ((int64_t)blockIdx.x * 256 >= sg.n) return;
    const double lo = jk_partials_max(partials + (int64_t)blockIdx.y * pb, pb, red);
    const double thr = jk_nanmax(lo, sg.floor) - margin;
    // an upper-bound row (b < 0): its value bounds lnL from above
    JK_LIST_ROWS(true, b != 0.0f && !(x + (double)fmaxf(b, 0.0f) < thr));
}

// ---------------------------------------------------------------------------
// Settling and rejection in one sequence (jk_settle_reject_batch): after the
// rows that could hold the maximum are settled and the FP64 maximum found
// (step 1 of jk_settle_batch), one pass draws every row's uniform once
// and decides it -- directly where the bound leaves no doubt, else puts it on
// the list of open rows.  The open rows (a few per million) are re-evaluated in FP64 and
// their decisions set from a uniform jumped to their index.  The accepted
// set is the one jk_settle_batch + jk_reject_batch give, with one pass over
// the rows and one PCG64 stream fewer.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_seg_decide(const double *__restrict__ ll,
                                                    const float *__restrict__ bound,
                                                    const SegDev *__restrict__ segs,
                                                    const double *__restrict__ partials2, int pb,
                                                    const unsigned long long *__restrict__ key,
                                                    u128 AT, u128 DT, double *__restrict__ llmax,
                                                    uint64_t *__restrict__ mask,
                                                    int64_t *__restrict__ count,
                                                    int64_t *__restrict__ idx)
{
    __shared__ double red[4];
    __shared__ int64_t s_buf[4][JK_APPEND_CAP];
    const SegDev sg = segs[blockIdx.y];
    if ((int64_t)blockIdx.x * 256 >= sg.n) return;
    const double mx = jk_settled_max(partials2, pb, key, red);
    if (blockIdx.x == 0 && threadIdx.x == 0) llmax[blockIdx.y] = mx;
    WaveAppend wa{s_buf[threadIdx.x >> 6], 0};
    const int lane = threadIdx.x & 63;
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t T = (int64_t)gridDim.x * 256;
    u128 s = pcg_thread_start(sg.s_base, sg.inc);
    for (int64_t base0 = g - lane; base0 < sg.n; base0 += JK_FLAG_UNROLL * T) {
        // the loads of JK_FLAG_UNROLL strides first
        double xs[JK_FLAG_UNROLL];
        float bs[JK_FLAG_UNROLL];
#pragma unroll
        for (int u = 0; u < JK_FLAG_UNROLL; ++u) {
            const int64_t i = base0 + u * T + lane;
            xs[u] = i < sg.n ? ll[sg.off + i] : 0.0;
            bs[u] = i < sg.n ? bound[sg.off + i] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < JK_FLAG_UNROLL; ++u) {
            const int64_t base = base0 + u * T;     // the same for every lane of the wave
            if (base >= sg.n) break;
            const int64_t i = base + lane;
            bool acc = false, open = false;
            if (i < sg.n) {
                const double uu = pcg_to_double(pcg_output(s));
                const double x = xs[u];
                const float bf = bs[u];
                if (bf > 0.0f) {
                    // a NaN maximum makes both sides false: nothing accepted, nothing open
                    const double b = fma((double)bf, 1e-6, (double)bf) + 1e-12;
                    const bool lo = jk_accept(x - b - mx, uu), hi = jk_accept(x + b - mx, uu);
                    open = lo != hi;
                    acc = lo && hi;
                } else if (bf < 0.0f) {
                    // an upper bound decides a rejection only
                    open = jk_accept(x - mx, uu);
                } else {
                    acc = jk_accept(x - mx, uu);
                }
            }
            const uint64_t word = __ballot(acc);
            if (lane == 0) mask[sg.mask_off + (base >> 6)] = word;
            jk_append(wa, open, i, idx + sg.idx_off, count + blockIdx.y);
            s = pcg_affine(s, AT, DT, sg.inc);
        }
    }
    jk_append_end(wa, idx + sg.idx_off, count + blockIdx.y);
}

// The decisions of the open rows, now in FP64: each row's uniform from the
// segment's stream jumped to its index; accepted rows set their bit.
__global__ __launch_bounds__(256) void k_seg_patch(const SegDev *__restrict__ segs,
                                                   const int64_t *__restrict__ count,
                                                   const int64_t *__restrict__ idx,
                                                   const double *__restrict__ ll,
                                                   const double *__restrict__ llmax,
                                                   uint64_t *__restrict__ mask)
{
    const SegDev sg = segs[blockIdx.y];
    const int64_t cnt = count[blockIdx.y];
    const double mx = llmax[blockIdx.y];
    for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < cnt;
         j += (int64_t)gridDim.x * 256) {
        const int64_t i = idx[sg.idx_off + j];
        const u128 st = pcg_jump_table(sg.s_base, (uint64_t)i, sg.inc);
        const double uu = pcg_to_double(pcg_output(st));
        if (jk_accept(ll[sg.off + i] - mx, uu))
            atomicOr((unsigned long long *)&mask[sg.mask_off + (i >> 6)], 1ull << (i & 63));
    }
}

// The outputs are written once and never read: they may be in host memory.
hipError_t jk_launch_settle_reject_batch(const jk_batch *b, int n_seg, const SegDev *d_settle,
                                         const SegDev *d_reject, int64_t max_n, int64_t max_nb,
                                         double *partials, int pb, uint64_t *mask, int64_t *bsum,
                                         int64_t *idx, unsigned long long *key, int64_t *cum,
                                         int64_t *count1, int64_t *count2, double *llmax,
                                         const double *P, const double *e, const double *om,
                                         const double *M0, const double *s, const int64_t *rows,
                                         double *ll, float *bound, int64_t *idx_out,
                                         int64_t *n_pass_out, double *llmax_out,
                                         int64_t *n_settled_out, hipStream_t stream)
{
    if (n_seg <= 0) return hipSuccess;
    const int fb = jk_seg_flag_blocks(max_n);
    double *partials2 = partials + (size_t)pb * n_seg;
    // 1. the rows that could hold the FP64 maximum, settled
    hipLaunchKernelGGL(k_seg_lo_partial, dim3(pb, n_seg), dim3(256), 0, stream, ll, bound,
                       d_settle, partials, partials2, pb, count1, count2, key);
    hipLaunchKernelGGL(k_seg_shell_list, dim3(fb, n_seg), dim3(256), 0, stream, ll, bound,
                       d_settle, partials, pb, count1, idx);
    hipError_t err = launch_seg_scatter(b, n_seg, d_settle, count1, cum, idx, P, e, om, M0, s,
                                        rows, ll, bound, stream, key);
    if (err != hipSuccess) return err;
    // 2. every row decided against the FP64 maximum or listed as open, one
    // uniform each
    u128 AT, DT;
    jk_pcg_jump_coeffs((uint64_t)fb * 256, &AT, &DT);
    hipLaunchKernelGGL(k_seg_decide, dim3(fb, n_seg), dim3(256), 0, stream, ll, bound, d_settle,
                       partials2, pb, key, AT, DT, llmax, mask, count2, idx);
    // 3. the open rows in FP64, then their decisions
    err = launch_seg_scatter(b, n_seg, d_settle, count2, cum, idx, P, e, om, M0, s, rows, ll,
                             bound, stream);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(k_seg_patch, dim3(4, n_seg), dim3(256), 0, stream, d_settle, count2, idx,
                       ll, llmax, mask);
    // 4. the ordered compaction of the accepted rows
    hipLaunchKernelGGL(k_seg_bsum, dim3((unsigned)max_nb, n_seg), dim3(256), 0, stream, d_reject,
                       mask, bsum, count1, count2, llmax, n_settled_out, llmax_out);
    hipLaunchKernelGGL(k_seg_compact, dim3((unsigned)max_nb, n_seg), dim3(256), 0, stream,
                       d_reject, mask, bsum, idx_out, n_pass_out);
    return hipGetLastError();
}

hipError_t jk_launch_settle_live_batch(const jk_batch *b, int n_seg, const SegDev *d_segs,
                                       int64_t max_n, double *partials, int pb, int64_t *idx,
                                       int64_t *cum, const double *P, const double *e,
                                       const double *om, const double *M0, const double *s,
                                       const int64_t *rows, double *ll, float *bound,
                                       double margin, int64_t *n_settled, hipStream_t stream)
{
    if (n_seg <= 0) return hipSuccess;
    const int fb = jk_seg_flag_blocks(max_n);
    hipLaunchKernelGGL(k_seg_lo_partial, dim3(pb, n_seg), dim3(256), 0, stream, ll, bound, d_segs,
                       partials, nullptr, pb, n_settled, nullptr, nullptr);
    hipLaunchKernelGGL(k_seg_live_list, dim3(fb, n_seg), dim3(256), 0, stream, ll, bound, d_segs,
                       partials, pb, margin, n_settled, idx);
    return launch_seg_scatter(b, n_seg, d_segs, n_settled, cum, idx, P, e, om, M0, s, rows, ll,
                              bound, stream);
}

// ---------------------------------------------------------------------------
// Settling to a tolerance (jk_settle_tol_batch): every entry of a segment
// whose error bound exceeds tol, or whose value is only an upper bound
// (negative bound), is re-evaluated in FP64.  Afterwards every entry is
// within tol of its FP64 lnL, whatever its distance from the maximum: the
// form for lnL arrays handed to a caller.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_seg_tol_list(const double *__restrict__ ll,
                                                      const float *__restrict__ bound,
                                                      const SegDev *__restrict__ segs, float tol,
                                                      int64_t *__restrict__ count,
                                                      int64_t *__restrict__ idx)
{
    const SegDev sg = segs[blockIdx.y];
    if ((int64_t)blockIdx.x * 256 >= sg.n) return;
    JK_LIST_ROWS(false, b < 0.0f || b > tol || b != b);
}

hipError_t jk_launch_settle_tol_batch(const jk_batch *b, int n_seg, const SegDev *d_segs,
                                      int64_t max_n, int64_t *idx, int64_t *cum, const double *P,
                                      const double *e, const double *om, const double *M0,
                                      const double *s, const int64_t *rows, double *ll,
                                      float *bound, float tol, int64_t *n_settled,
                                      hipStream_t stream)
{
    if (n_seg <= 0) return hipSuccess;
    const int fb = jk_seg_flag_blocks(max_n);
    hipLaunchKernelGGL(k_fill_i64, dim3((n_seg + 255) / 256), dim3(256), 0, stream, n_settled,
                       n_seg, (int64_t)0);
    hipLaunchKernelGGL(k_seg_tol_list, dim3(fb, n_seg), dim3(256), 0, stream, ll, bound, d_segs,
                       tol, n_settled, idx);
    return launch_seg_scatter(b, n_seg, d_segs, n_settled, cum, idx, P, e, om, M0, s, rows, ll,
                              bound, stream);
}

// ---------------------------------------------------------------------------
// Settling a buffer whose entries are values or upper bounds
// (jk_settle_pruned_batch): a probe launch leaves every row's upper bound
// (bound < 0); the rows that can matter are then evaluated in FP64 around the
// maximum, found in two steps.
//   1. hi = max over the segment of (ll + max(b, 0)) bounds the FP64 maximum
//      from above; the upper-bound rows with ll >= hi - window are evaluated.
//   2. lo = max over the value rows (b >= 0) of ll - b bounds it from below;
//      the upper-bound rows with ll >= lo - margin are evaluated.
// Afterwards every upper-bound row lies more than margin below the maximum.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_seg_hi_partial(const double *__restrict__ ll,
                                                        const float *__restrict__ bound,
                                                        const SegDev *__restrict__ segs,
                                                        double *__restrict__ partials, int pb,
                                                        int64_t *__restrict__ count)
{
    __shared__ double red[4];
    const SegDev sg = segs[blockIdx.y];
    if (blockIdx.x == 0 && threadIdx.x == 0) count[blockIdx.y] = 0;
    double m = -INFINITY;
    const int64_t stride = (int64_t)pb * 256;
    for (int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x; i0 < sg.n;
         i0 += JK_FLAG_UNROLL * stride) {
        double xs[JK_FLAG_UNROLL];
#pragma unroll
        for (int u = 0; u < JK_FLAG_UNROLL; ++u) {
            const int64_t i = i0 + u * stride;
            xs[u] = i < sg.n ? ll[sg.off + i] + (double)fmaxf(bound[sg.off + i], 0.0f) : -INFINITY;
        }
#pragma unroll
        for (int u = 0; u < JK_FLAG_UNROLL; ++u) m = jk_nanmax(m, xs[u]);
    }
    m = wave_nanmax(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        partials[(int64_t)blockIdx.y * pb + blockIdx.x] =
            jk_nanmax(jk_nanmax(red[0], red[1]), jk_nanmax(red[2], red[3]));
}

// Upper-bound rows (b < 0) not below the segment's level - margin; every
// upper-bound row when the level is NaN.
__global__ __launch_bounds__(256) void k_seg_upper_list(const double *__restrict__ ll,
                                                        const float *__restrict__ bound,
                                                        const SegDev *__restrict__ segs,
                                                        const double *__restrict__ partials, int pb,
                                                        double margin, int64_t *__restrict__ count,
                                                        int64_t *__restrict__ idx)
{
    __shared__ double red[4];
    const SegDev sg = segs[blockIdx.y];
    if ((int64_t)blockIdx.x * 256 >= sg.n) return;
    const double thr = jk_partials_max(partials + (int64_t)blockIdx.y * pb, pb, red) - margin;
    JK_LIST_ROWS(true, b < 0.0f && !(x < thr));
}

hipError_t jk_launch_settle_pruned_batch(const jk_batch *b, int n_seg, const SegDev *d_segs,
                                         int64_t max_n, double *partials, int pb, int64_t *idx,
                                         int64_t *cum, int64_t *count1, const double *P,
                                         const double *e, const double *om, const double *M0,
                                         const double *s, const int64_t *rows, double *ll,
                                         float *bound, double window, double margin,
                                         int64_t *n_settled, hipStream_t stream)
{
    if (n_seg <= 0) return hipSuccess;
    const int fb = jk_seg_flag_blocks(max_n);
    // 1. the rows whose bound reaches the window below the upper bound on the maximum
    hipLaunchKernelGGL(k_seg_hi_partial, dim3(pb, n_seg), dim3(256), 0, stream, ll, bound, d_segs,
                       partials, pb, count1);
    hipLaunchKernelGGL(k_seg_upper_list, dim3(fb, n_seg), dim3(256), 0, stream, ll, bound, d_segs,
                       partials, pb, window, count1, idx);
    hipError_t err = launch_seg_scatter(b, n_seg, d_segs, count1, cum, idx, P, e, om, M0, s, rows,
                                        ll, bound, stream);
    if (err != hipSuccess) return err;
    // 2. the rows whose bound reaches the margin below the lower bound on the maximum
    hipLaunchKernelGGL(k_seg_lo_partial, dim3(pb, n_seg), dim3(256), 0, stream, ll, bound, d_segs,
                       partials, nullptr, pb, n_settled, nullptr, nullptr);
    hipLaunchKernelGGL(k_seg_upper_list, dim3(fb, n_seg), dim3(256), 0, stream, ll, bound, d_segs,
                       partials, pb, margin, n_settled, idx);
    err = launch_seg_scatter(b, n_seg, d_segs, n_settled, cum, idx, P, e, om, M0, s, rows, ll,
                             bound, stream);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(k_seg_add_counts, dim3((n_seg + 255) / 256), dim3(256), 0, stream, count1,
                       n_settled, n_seg);
    return hipGetLastError();
}

void jk_host_pcg_jump(u128 state, u128 inc, uint64_t k, u128 *out) { *out = h_jump(state, inc, k); }

// ---------------------------------------------------------------------------
// On-device prior cache fill.  Philox4x32-10 (Salmon, Moraes, Dror & Shaw,
// "Parallel random numbers: as easy as 1, 2, 3", SC 2011): counter = (row,
// block, 0, 0), key = seed; three blocks per row give six 53-bit uniforms.
//   P     = exp(u0 (ln P_max - ln P_min) + ln P_min)    (log-uniform)
//   e     = inverse Beta CDF, linear interpolation in a table of n_tab + 1
//           equally spaced quantiles built on the host
//   omega = 2 pi u2,  M0 = 2 pi u3
//   s     = exp(mu + sigma z), z = sqrt(-2 ln(1 - u4)) cos(2 pi u5), or 0
// FP64 master columns and their FP32 copy are written in one pass.
// ---------------------------------------------------------------------------
struct Philox4 {
    uint32_t v[4];
};

__device__ __forceinline__ Philox4 philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                                 uint32_t k0, uint32_t k1)
{
    const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint32_t hi0 = __umulhi(M0, c0), lo0 = M0 * c0;
        const uint32_t hi1 = __umulhi(M1, c2), lo1 = M1 * c2;
        const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
        c0 = n0;
        c1 = lo1;
        c2 = n2;
        c3 = lo0;
        k0 += W0;
        k1 += W1;
    }
    Philox4 o;
    o.v[0] = c0;
    o.v[1] = c1;
    o.v[2] = c2;
    o.v[3] = c3;
    return o;
}

__device__ __forceinline__ double u53(uint32_t a, uint32_t b)
{
    return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) * (1.0 / 9007199254740992.0);
}

__global__ __launch_bounds__(256) void k_prior_fill(int64_t n, int64_t row0, uint32_t k0,
                                                    uint32_t k1, double lnPmin, double lnPspan,
                                                    const double *__restrict__ e_tab, int n_tab,
                                                    double s_mu, double s_sigma,
                                                    double *__restrict__ P, double *__restrict__ e,
                                                    double *__restrict__ om,
                                                    double *__restrict__ M0,
                                                    double *__restrict__ s, float *__restrict__ e32,
                                                    float *__restrict__ om32,
                                                    float *__restrict__ M032,
                                                    float *__restrict__ s32)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t row = (uint64_t)(row0 + i);
    const uint32_t lo = (uint32_t)row, hi = (uint32_t)(row >> 32);
    const Philox4 a = philox4x32_10(lo, hi, 0u, 0u, k0, k1);
    const Philox4 b = philox4x32_10(lo, hi, 1u, 0u, k0, k1);
    const Philox4 c = philox4x32_10(lo, hi, 2u, 0u, k0, k1);
    const double u0 = u53(a.v[0], a.v[1]), u1 = u53(a.v[2], a.v[3]);
    const double u2 = u53(b.v[0], b.v[1]), u3 = u53(b.v[2], b.v[3]);
    const double u4 = u53(c.v[0], c.v[1]), u5 = u53(c.v[2], c.v[3]);
    const double Pv = exp(fma(u0, lnPspan, lnPmin));
    const double x = u1 * n_tab;
    int k = (int)x;
    if (k >= n_tab) k = n_tab - 1;
    const double f = x - k;
    const double ev = fma(f, e_tab[k + 1] - e_tab[k], e_tab[k]);
    const double omv = JK_TWO_PI * u2, M0v = JK_TWO_PI * u3;
    double sv = 0.0;
    if (s_sigma >= 0.0) {
        const double z = sqrt(-2.0 * log1p(-u4)) * cos(JK_TWO_PI * u5);
        sv = exp(fma(s_sigma, z, s_mu));
    }
    P[i] = Pv;
    e[i] = ev;
    om[i] = omv;
    M0[i] = M0v;
    s[i] = sv;
    if (e32) {
        e32[i] = (float)ev;
        om32[i] = (float)omv;
        M032[i] = (float)M0v;
        s32[i] = (float)sv;
    }
}

hipError_t jk_launch_prior_fill(int64_t n, int64_t row0, uint64_t seed, double P_min, double P_max,
                                const double *e_tab, int n_tab, double s_mu, double s_sigma,
                                double *P, double *e, double *om, double *M0, double *s,
                                float *e32, float *om32, float *M032, float *s32,
                                hipStream_t stream)
{
    if (n <= 0) return hipSuccess;
    const double lnPmin = log(P_min);
    const double span = log(P_max) - lnPmin;
    hipLaunchKernelGGL(k_prior_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, n,
                       row0, (uint32_t)seed, (uint32_t)(seed >> 32), lnPmin, span, e_tab, n_tab,
                       s_mu, s_sigma, P, e, om, M0, s, e32, om32, M032, s32);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Linear-parameter posterior of accepted rows, FP64.  Lambda[0] is not clipped
// here (fast_likelihood.pyx:519-521).
//
// Hundreds to thousands of rows of up to a few hundred epochs: the time is one
// row's chain of dependent operations, not the arithmetic.  A group of 16
// lanes takes a row's epochs, lane l the epochs l, l + 16, ..., with the
// Kepler solve of the FP64 likelihood rows (LDS tables) and L at compile time,
// so the sums stay in registers.  The lanes' sums are combined by a butterfly
// of DPP moves that halves the number of quantities a lane holds at each step
// (NP - 1 exchanges for NP quantities, instead of 4 NP), they go to LDS, and
// one wave finishes the workgroup's rows, a lane per row.  The order of every
// sum depends on the row's star only, so the one-star and the many-star
// launches give the same bits.  16 lanes per row: at 64 a row's setup and its
// exchanges took 200 us of 65536 rows of 6 epochs (now 22), with 2048 rows of
// 64 epochs at 12 us (now 8.2).  Against a wave per row with the sums in
// scratch and the library's sine and cosine, L = 3: 2048 rows of 6 epochs
// 37 -> 6.0 us, of 64 36 -> 8.2, of 200 47 -> 15; 65536 rows of 64 epochs
// 738 -> 42.  Full covariance (was a lane per row, the rotation from global
// memory): 2048 rows of 64 epochs 237 -> 14 us, 65536 327 -> 112.
// The design value comes from the likelihood's tables and one-step solve
// instead of the library's sine and cosine and the converged iteration: against
// 80-bit arithmetic, 100 stars of 3 to 200 epochs, the errors are those of that
// form within their scatter (norm of a 0.98, of cov 1.04 +- 0.04, median of cov
// 1.01 +- 0.01, of the lnL 0.92 times).  The finish divides by the pivots:
// products with their reciprocals put the median of cov at 1.04 +- 0.01 and
// save nothing.
// ---------------------------------------------------------------------------
#define JK_POST_WG 256                 // threads per workgroup
#define JK_POST_G 16                   // lanes per row (one DPP row)
#define JK_POST_NG (JK_POST_WG / JK_POST_G)   // rows in flight per workgroup
#define JK_POST_RPG 4                  // most rows per group: NG x 4 lanes finish
#define JK_POST_FULL 16384             // rows that fill the chip at one per group

// The quantities of a row, in order: chi0, sum ln w, rhs[L], u[L], G's lower
// triangle by rows; padded to a power of two for the butterfly.
template <int L>
struct PostSums {
    static constexpr int NQ = 2 + 2 * L + L * (L + 1) / 2;
    static constexpr int LG = NQ <= 8 ? 3 : NQ <= 16 ? 4 : NQ <= 32 ? 5 : 6;
    static constexpr int NP = 1 << LG;
};

// The end of a row's linear posterior from its sums over the epochs: the prior
// added, Cholesky, cov = G^-1, a = cov rhs, and the row's lnL.
template <int L>
__device__ __forceinline__ void jk_posterior_finish(const StarDev &st, int64_t i, double Pv,
                                                    double ev, const double *__restrict__ q,
                                                    const double2 *__restrict__ ltab,
                                                    double *__restrict__ a_out,
                                                    double *__restrict__ cov_out,
                                                    double *__restrict__ ll_out)
{
    const double lam0 = st.k_prior_mode == JK_KPRIOR_FIXED_COMPANION_MASS
                            ? jk_k_variance(&st, Pv, ev, false)
                            : st.lam0;
    double G[L][L], rhs[L], u[L];
#pragma unroll
    for (int a = 0; a < L; ++a) {
        rhs[a] = q[2 + a];
        u[a] = q[2 + L + a];
#pragma unroll
        for (int b = 0; b <= a; ++b) G[a][b] = q[2 + 2 * L + a * (a + 1) / 2 + b];
    }
    const double il0 = 1.0 / lam0;
    G[0][0] += il0;
    rhs[0] = fma(st.mu0, il0, rhs[0]);
#pragma unroll
    for (int a = 1; a < L; ++a) {
        G[a][a] += st.lam_inv[a];
        rhs[a] += st.mu[a] * st.lam_inv[a];
    }
    // Cholesky G = R R^T (lower, in place; the diagonal holds 1 / R_jj);
    // lam0 det G as a mantissa and an exponent.
    int dexp;
    double detm = frexp(lam0, &dexp);
    bool ok = true;
#pragma unroll
    for (int j = 0; j < L; ++j) {
        double d = G[j][j];
#pragma unroll
        for (int k = 0; k < j; ++k) d = fma(-G[j][k], G[j][k], d);
        ok = ok && d > 0.0;
        int ex;
        detm = frexp(detm * d, &ex);
        dexp += ex;
        const double rj = sqrt(d);
        G[j][j] = 1.0 / rj;
#pragma unroll
        for (int c = j + 1; c < L; ++c) {
            double v = G[c][j];
#pragma unroll
            for (int k = 0; k < j; ++k) v = fma(-G[c][k], G[j][k], v);
            G[c][j] = v / rj;
        }
    }
    double *__restrict__ ao = a_out + i * L;
    double *__restrict__ co = cov_out + i * L * L;
    if (!ok) {
        for (int c = 0; c < L; ++c) ao[c] = __builtin_nan("");
        for (int c = 0; c < L * L; ++c) co[c] = __builtin_nan("");
        ll_out[i] = INFINITY;
        return;
    }
    // R^-1 (lower) by forward substitution, z = R^-1 u for chi2.
    double Ri[L][L];
    double zz = 0.0;
#pragma unroll
    for (int c = 0; c < L; ++c) {
        Ri[c][c] = G[c][c];
#pragma unroll
        for (int a = c + 1; a < L; ++a) {
            double v = 0.0;
#pragma unroll
            for (int k = c; k < a; ++k) v = fma(-G[a][k], Ri[k][c], v);
            Ri[a][c] = v * G[a][a];
        }
    }
#pragma unroll
    for (int a = 0; a < L; ++a) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k <= a; ++k) v = fma(Ri[a][k], u[k], v);
        zz = fma(v, v, zz);
    }
    // cov = R^-T R^-1 (symmetric), a = cov rhs.
    double am[L];
#pragma unroll
    for (int a = 0; a < L; ++a) am[a] = 0.0;
#pragma unroll
    for (int a = 0; a < L; ++a)
#pragma unroll
        for (int b = 0; b <= a; ++b) {
            double v = 0.0;
#pragma unroll
            for (int k = a; k < L; ++k) v = fma(Ri[k][a], Ri[k][b], v);
            co[a * L + b] = v;
            am[a] = fma(v, rhs[b], am[a]);
            if (b < a) {
                co[b * L + a] = v;
                am[b] = fma(v, rhs[a], am[b]);
            }
        }
#pragma unroll
    for (int a = 0; a < L; ++a) ao[a] = am[a];
    const double lnd = jk_log_tab(detm, ltab) + (double)dexp * JK_LN2;
    ll_out[i] = -0.5 * (q[0] - zz + (double)st.n * JK_LN_TWO_PI - q[1] + st.ln_lam_trend + lnd);
}

// sin E, cos E and the design value of one epoch.
__device__ __forceinline__ double jk_posterior_design(double dtk, double nP, double M0v, double ev,
                                                      float ef, float omef, float a1f, double dmax,
                                                      double sq, double cw, double sw, double ecw,
                                                      const double2 *__restrict__ tab)
{
    const double x = jk_reduce_2pi(fma(nP, dtk, -M0v));
    double sE, cE;
    if (!jk_kepler_markley_f64(x, ev, ef, omef, a1f, dmax, tab, sE, cE))
        jk_kepler_poly_f64(x, ev, tab, sE, cE);
    return jk_design_f64(sE, cE, ev, sq, cw, sw, ecw);
}

// v of the lane that DPP control CTRL names (all lanes active).
template <int CTRL>
__device__ __forceinline__ double jk_dpp(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// One step of the butterfly over v[0 .. 2 HALF): the lanes with `up` keep the
// upper half, the others the lower, each adding its partner's partials of it;
// a single quantity (HALF == 0) is added to the partner's.
template <int HALF, int CTRL>
__device__ __forceinline__ void jk_post_fold(double *v, bool up)
{
    if constexpr (HALF == 0) {
        v[0] += jk_dpp<CTRL>(v[0]);
    } else {
#pragma unroll
        for (int j = 0; j < HALF; ++j) {
            const double keep = up ? v[j + HALF] : v[j], send = up ? v[j] : v[j + HALF];
            v[j] = keep + jk_dpp<CTRL>(send);
        }
    }
}

// One row's sums over the epochs by a group of JK_POST_G lanes, into q[NQ] of
// LDS; pe = (P, e), P NaN for an invalid row.  live: false for a group with no
// row (it only takes part in the exchanges).  COV (a full-covariance star,
// n <= JK_COV_NMAX): the design column is computed in epoch order in m_col (n
// doubles of LDS of this group) and rotated into the eigenbasis the star's
// data are in, with s_Q the eigenvectors (element (k, c) of Q^T at
// c (n | 1) + k).
template <int L, bool COV>
__device__ __forceinline__ void jk_posterior_sums(const StarDev &st, int64_t r,
                                                  const double *__restrict__ P,
                                                  const double *__restrict__ E_,
                                                  const double *__restrict__ OM,
                                                  const double *__restrict__ MM,
                                                  const double *__restrict__ S,
                                                  const double2 *__restrict__ tab, double *m_col,
                                                  const double *s_Q, bool live, double *q, double2 *pe)
{
    constexpr int NQ = PostSums<L>::NQ, NP = PostSums<L>::NP, G = JK_POST_G;
    const int lane = threadIdx.x & (G - 1);
    const bool phys = st.jitter_mode == JK_JITTER_PHYSICAL;
    const double Pv = P[r], ev = E_[r], omv = OM[r], M0v = MM[r];
    const double sv = phys ? S[r] : 0.0;
    const bool valid = isfinite(Pv) && Pv != 0.0 && ev >= 0.0 && ev < 1.0 && isfinite(omv) &&
                       isfinite(M0v) && isfinite(sv);
    const int N = valid && live ? st.n : 0;
    if (lane == 0 && live) *pe = make_double2(valid ? Pv : __builtin_nan(""), ev);
    double sw, cw;
    jk_sincos_tab_f64(omv, tab, sw, cw);
    const double ecw = ev * cw, sq = sqrt((1.0 - ev) * (1.0 + ev));
    const double nP = JK_TWO_PI / Pv, s2 = sv * sv;
    // the FP32 starter's copies, as in jk_row_orbit
    const float ef = fminf((float)ev, 0.99999994f);
    const float omef = fmaxf((float)(1.0 - ev), 5.9604645e-08f);
    const float a1f = JK_MARKLEY_A1N * __builtin_amdgcn_rcpf(1.0f + ef);
    const double dmax = ev > 0.9999999 ? -1.0 : 1e-3;
    if constexpr (COV) {
        for (int k = lane; k < N; k += G)
            m_col[k] = jk_posterior_design(st.dt[k], nP, M0v, ev, ef, omef, a1f, dmax, sq, cw, sw,
                                           ecw, tab);
        // one wave's LDS writes and reads are in order
        __builtin_amdgcn_wave_barrier();
        double acc[JK_COV_NMAX / G];
#pragma unroll
        for (int j = 0; j < JK_COV_NMAX / G; ++j) acc[j] = 0.0;
        const int QP = N | 1;
        for (int c = 0; c < N; ++c) {
            const double mc = m_col[c];
#pragma unroll
            for (int j = 0; j < JK_COV_NMAX / G; ++j)
                acc[j] = fma(s_Q[c * QP + min(lane + j * G, N - 1)], mc, acc[j]);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < JK_COV_NMAX / G; ++j)
            if (lane + j * G < N) m_col[lane + j * G] = acc[j];
        __builtin_amdgcn_wave_barrier();
    }
    double v[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) v[j] = 0.0;
#pragma unroll 1
    for (int k = lane; k < N; k += G) {
        double x[L];
        if constexpr (COV) {
            x[0] = m_col[k];
        } else {
            x[0] = jk_posterior_design(st.dt[k], nP, M0v, ev, ef, omef, a1f, dmax, sq, cw, sw, ecw,
                                       tab);
        }
#pragma unroll
        for (int j = 1; j < L; ++j) x[j] = st.T[(j - 1) * N + k];
        const double iv = st.ivar[k], yk = st.y[k];
        const double w = phys ? iv / fma(s2, iv, 1.0) : iv;
        const double rr = st.rp[k] - st.mu0 * x[0];
        v[0] = fma(w * rr, rr, v[0]);
        v[1] += jk_log_tab(w, tab + JK_TAB_LOG_OFF);
#pragma unroll
        for (int a = 0; a < L; ++a) {
            const double wx = w * x[a];
            v[2 + a] = fma(wx, yk, v[2 + a]);
            v[2 + L + a] = fma(wx, rr, v[2 + L + a]);
#pragma unroll
            for (int b = 0; b <= a; ++b)
                v[2 + 2 * L + a * (a + 1) / 2 + b] = fma(wx, x[b], v[2 + 2 * L + a * (a + 1) / 2 + b]);
        }
    }
    // partners: lane ^ 8 (row_ror 8), ^ 7 (half mirror), ^ 2 and ^ 1 (quad
    // permutes), which between them reach all 16 lanes
    jk_post_fold<NP / 2, 0x128>(v, lane & 8);
    jk_post_fold<NP / 4, 0x141>(v, lane & 4);
    jk_post_fold<NP / 8, 0x4e>(v, lane & 2);
    jk_post_fold<NP / 16, 0xb1>(v, lane & 1);
    constexpr int K = NP > G ? NP / G : 1;   // quantities a lane ends with
    const int q0 = lane * NP / G;
#pragma unroll
    for (int j = 0; j < K; ++j)
        if (q0 + j < NQ && live) q[q0 + j] = v[j];
}

// Doubles from one group's design column to the next's (full covariance).
__host__ __device__ inline int jk_post_cov_pitch(int N, int NP)
{
    return N > NP ? N | 1 : NP | 1;
}

// This workgroup's rows of [i0, n), rpg per group; star(i): the row's star.
template <int L, bool COV, typename Star>
__device__ __forceinline__ void jk_posterior_rows(Star star, int64_t i0, int64_t n, int rpg,
                                                  const double *__restrict__ P,
                                                  const double *__restrict__ E_,
                                                  const double *__restrict__ OM,
                                                  const double *__restrict__ MM,
                                                  const double *__restrict__ S,
                                                  const int64_t *__restrict__ rows,
                                                  double *__restrict__ a_out,
                                                  double *__restrict__ cov_out,
                                                  double *__restrict__ ll_out, double *s_m)
{
    constexpr int NP = PostSums<L>::NP, RWG = COV ? 1 : JK_POST_NG * JK_POST_RPG;
    __shared__ double2 s_tab[JK_TAB_LDS64];
    // odd pitch: the finishing lanes read one quantity of many rows at a time
    __shared__ double s_qd[RWG * (NP + 1)];
    __shared__ double2 s_pe[COV ? JK_POST_NG : RWG];
    // a full-covariance star's rows (one per group): the eigenvectors, then
    // each group's design column, which its sums then replace
    double *s_q = s_qd;
    int qp = NP + 1;
    if constexpr (COV) {
        const StarDev &st = star(0);
        const int N = st.n, QP = N | 1;
        s_q = s_m + N * QP;
        qp = jk_post_cov_pitch(N, NP);
        for (int t = threadIdx.x; t < N * N; t += JK_POST_WG)
            s_m[(t % N) * QP + t / N] = st.Qt[t];
    }
    jk_stage_tab<false>(s_tab);
    const int group = threadIdx.x / JK_POST_G;
    const int64_t ib = i0 + (int64_t)blockIdx.x * (JK_POST_NG * rpg);
#pragma unroll 1
    for (int t = 0; t < rpg; ++t) {
        const int slot = t * JK_POST_NG + group;
        const bool live = ib + slot < n;
        const int64_t i = live ? ib + slot : n - 1;
        const StarDev &st = star(i);
        jk_posterior_sums<L, COV>(st, rows ? rows[i] : i, P, E_, OM, MM, S, s_tab,
                                  s_q + slot * qp, s_m, live,
                                  s_q + slot * qp, s_pe + slot);
    }
    __syncthreads();
    const int slot = threadIdx.x;
    const int64_t i = ib + slot;
    if (slot >= JK_POST_NG * rpg || i >= n) return;
    const double2 pe = s_pe[slot];
    if (isnan(pe.x)) {
        for (int c = 0; c < L; ++c) a_out[i * L + c] = __builtin_nan("");
        for (int c = 0; c < L * L; ++c) cov_out[i * L * L + c] = __builtin_nan("");
        ll_out[i] = __builtin_nan("");
        return;
    }
    jk_posterior_finish<L>(star(i), i, pe.x, pe.y, s_q + slot * qp, s_tab + JK_TAB_LOG_OFF,
                           a_out, cov_out, ll_out);
}

template <int L, bool COV>
__global__ __launch_bounds__(JK_POST_WG) void k_linear_posterior(
    const StarDev st, int64_t i0, int64_t n, int rpg, const double *__restrict__ P,
    const double *__restrict__ E_, const double *__restrict__ OM, const double *__restrict__ MM,
    const double *__restrict__ S, const int64_t *__restrict__ rows, double *__restrict__ a_out,
    double *__restrict__ cov_out, double *__restrict__ ll_out)
{
    extern __shared__ double s_m[];
    jk_posterior_rows<L, COV>([&](int64_t) -> const StarDev & { return st; }, i0, n, rpg, P, E_,
                              OM, MM, S, rows, a_out, cov_out, ll_out, s_m);
}

// Accepted rows of many stars of a table in one launch: row i belongs to
// table entry star_idx[i] (diagonal-covariance stars only).
template <int L>
__global__ __launch_bounds__(JK_POST_WG) void k_linear_posterior_batch(
    const StarDev *__restrict__ stars, const int32_t *__restrict__ star_idx, int64_t i0, int64_t n,
    int rpg, const double *__restrict__ P, const double *__restrict__ E_,
    const double *__restrict__ OM, const double *__restrict__ MM, const double *__restrict__ S,
    const int64_t *__restrict__ rows, double *__restrict__ a_out, double *__restrict__ cov_out,
    double *__restrict__ ll_out)
{
    jk_posterior_rows<L, false>([&](int64_t i) -> const StarDev & { return stars[star_idx[i]]; },
                                i0, n, rpg, P, E_, OM, MM, S, rows, a_out, cov_out, ll_out,
                                nullptr);
}

// Rows per launch of the posterior kernels (the grid's threads stay far inside
// 2^32).
#define JK_POST_CHUNK ((int64_t)1 << 24)

// One row per group until that fills the chip, then more: a workgroup stages
// the tables once, and its finishing wave has more lanes at work.
static int jk_post_rpg(int64_t n)
{
    const int64_t r = n / JK_POST_FULL;
    return r < 1 ? 1 : r > JK_POST_RPG ? JK_POST_RPG : (int)r;
}

#define JK_POST_SWITCH(L_, LAUNCH)                                                                 \
    switch (L_) {                                                                                  \
    case 1: LAUNCH(1); break;                                                                      \
    case 2: LAUNCH(2); break;                                                                      \
    case 3: LAUNCH(3); break;                                                                      \
    case 4: LAUNCH(4); break;                                                                      \
    case 5: LAUNCH(5); break;                                                                      \
    case 6: LAUNCH(6); break;                                                                      \
    case 7: LAUNCH(7); break;                                                                      \
    case 8: LAUNCH(8); break;                                                                      \
    default: return hipErrorInvalidValue;                                                          \
    }

hipError_t jk_launch_linear_posterior_batch(const jk_batch *b, int64_t n, const int32_t *star_idx,
                                            const double *P, const double *e, const double *om,
                                            const double *M0, const double *s,
                                            const int64_t *rows, double *a_out, double *cov_out,
                                            double *ll_out, hipStream_t stream)
{
    const int rpg = jk_post_rpg(n), rwg = JK_POST_NG * rpg;
    for (int64_t i0 = 0; i0 < n; i0 += JK_POST_CHUNK) {
        const int64_t nb = n - i0 < JK_POST_CHUNK ? n - i0 : JK_POST_CHUNK;
        const dim3 grid((unsigned)((nb + rwg - 1) / rwg));
        const int64_t end = i0 + nb;
#define LAUNCH(LL)                                                                                 \
    hipLaunchKernelGGL(k_linear_posterior_batch<LL>, grid, dim3(JK_POST_WG), 0, stream,    \
                       b->d_stars, star_idx, i0, end, rpg, P, e, om, M0, s, rows, a_out, cov_out,  \
                       ll_out)
        JK_POST_SWITCH(b->L, LAUNCH)
#undef LAUNCH
    }
    return hipGetLastError();
}

hipError_t jk_launch_linear_posterior(const jk_star *st, int64_t n, const double *P,
                                      const double *e, const double *om, const double *M0,
                                      const double *s, const int64_t *rows, double *a_out,
                                      double *cov_out, double *ll_out, hipStream_t stream)
{
    const bool cov = st->dev.Qt != nullptr;
    const int rpg = cov ? 1 : jk_post_rpg(n), rwg = JK_POST_NG * rpg;
    const int N = st->dev.n;
    for (int64_t i0 = 0; i0 < n; i0 += JK_POST_CHUNK) {
        const int64_t nb = n - i0 < JK_POST_CHUNK ? n - i0 : JK_POST_CHUNK;
        const dim3 grid((unsigned)((nb + rwg - 1) / rwg));
        const int64_t end = i0 + nb;
#define LAUNCH(LL)                                                                                 \
    if (cov)                                                                                       \
        hipLaunchKernelGGL((k_linear_posterior<LL, true>), grid, dim3(JK_POST_WG),                 \
                           sizeof(double) * (N * (N | 1) + JK_POST_NG * jk_post_cov_pitch(         \
                                                                      N, PostSums<LL>::NP)),       \
                           stream, st->dev, i0, end, rpg, P, e, om, M0, s, rows, a_out, cov_out,   \
                           ll_out);                                                                \
    else                                                                                           \
        hipLaunchKernelGGL((k_linear_posterior<LL, false>), grid, dim3(JK_POST_WG), 0,     \
                           stream, st->dev, i0, end, rpg, P, e, om, M0, s, rows, a_out, cov_out,   \
                           ll_out)
        JK_POST_SWITCH(st->dev.L, LAUNCH)
#undef LAUNCH
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// One prior row in full detail (jk_debug_single): the quantities
// CJokerHelper.test_likelihood_worker leaves in its public members
// (fast_likelihood.pyx:109-114, 255-425, 547-576), for tests.  One lane, FP64,
// diagonal data covariance C = diag(1/w) (w = ivar, or ivar / (1 + s^2 ivar)
// in the physical jitter mode).  Lambda[0] is not clipped to max_K^2 here, as
// in test_likelihood_worker (:567-569).
//   M_T   (L x N)  design matrix, row 0 the unit-K Keplerian column
//   Ainv  (L x L)  Lambda^-1 + M_T C^-1 M_T^T                  (:262-276)
//   A     (L x L)  inverse of Ainv (here from its Cholesky factor)
//   a     (L)      Ainv^-1 (M_T C^-1 y + Lambda^-1 mu)         (:394-420)
//   b     (N)      M mu                                        (:305-309)
//   B     (N x N)  C + M Lambda M^T (optional)                 (:315-327)
//   Binv  (N x N)  C^-1 - C^-1 M A M^T C^-1 (optional)         (:329-337)
//   sc    lnL, chi2 = (b - y)^T Binv (b - y), ln det(2 pi B), Lambda[0]
// ln det(2 pi B) comes from the determinant lemma,
// N ln 2 pi - sum ln w + sum ln Lambda + ln det Ainv, and chi2 from the same
// algebra, sum w r^2 - v^T A v with v = M_T C^-1 r; the reference takes the
// LU of B (:342-353) and sums over Binv (:387-392), the same quantities.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(64) void k_debug_row(const StarDev st, const double *__restrict__ row,
                                                 double *__restrict__ MT,
                                                 double *__restrict__ Ainv,
                                                 double *__restrict__ A,
                                                 double *__restrict__ a,
                                                 double *__restrict__ b,
                                                 double *__restrict__ B,
                                                 double *__restrict__ Binv,
                                                 double *__restrict__ sc)
{
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const int L = st.L, N = st.n;
    const bool phys = st.jitter_mode == JK_JITTER_PHYSICAL;
    const double Pv = row[0], ev = row[1], omv = row[2], M0v = row[3];
    const double sv = phys ? row[4] : 0.0;
    const double nan = __builtin_nan("");
    const bool valid = isfinite(Pv) && Pv != 0.0 && ev >= 0.0 && ev < 1.0 && isfinite(omv) &&
                       isfinite(M0v) && isfinite(sv);
    const double lam0 = st.k_prior_mode == JK_KPRIOR_FIXED_COMPANION_MASS
                            ? (valid ? jk_k_variance(&st, Pv, ev, false) : nan)
                            : st.lam0;
    double lam[JK_LMAX];
    lam[0] = lam0;
    for (int i = 1; i < L; ++i) lam[i] = 1.0 / st.lam_inv[i];
    double sw = 0.0, cw = 1.0;
    if (valid) sincos(omv, &sw, &cw);
    const double ecw = ev * cw, sq = valid ? sqrt((1.0 - ev) * (1.0 + ev)) : nan;
    const double nP = JK_TWO_PI / Pv;
    double G[JK_LMAX * JK_LMAX], rhs[JK_LMAX], v[JK_LMAX];
    for (int q = 0; q < JK_LMAX * JK_LMAX; ++q) G[q] = 0.0;
    for (int q = 0; q < JK_LMAX; ++q) rhs[q] = v[q] = 0.0;
    double wrr = 0.0, sum_ln_w = 0.0;
    for (int k = 0; k < N; ++k) {
        double x0 = nan;
        if (valid) {
            double sE, cE;
            jk_kepler_f64(jk_reduce_2pi(fma(nP, st.dt[k], -M0v)), ev, sE, cE);
            x0 = jk_design_f64(sE, cE, ev, sq, cw, sw, ecw);
        }
        MT[k] = x0;
        for (int j = 1; j < L; ++j) MT[(size_t)j * N + k] = st.T[(size_t)(j - 1) * N + k];
        const double iv = st.ivar[k];
        const double w = phys ? iv / fma(sv * sv, iv, 1.0) : iv;
        double bk = 0.0;
        for (int i = 0; i < L; ++i) bk = fma(MT[(size_t)i * N + k], st.mu[i], bk);
        b[k] = bk;
        const double r = bk - st.y[k];
        wrr = fma(w * r, r, wrr);
        sum_ln_w += log(w);
        for (int i = 0; i < L; ++i) {
            const double wx = w * MT[(size_t)i * N + k];
            rhs[i] = fma(wx, st.y[k], rhs[i]);
            v[i] = fma(wx, r, v[i]);
            for (int j = 0; j < L; ++j) G[i * JK_LMAX + j] = fma(wx, MT[(size_t)j * N + k], G[i * JK_LMAX + j]);
        }
    }
    double lnlam = 0.0;
    for (int i = 0; i < L; ++i) {
        G[i * JK_LMAX + i] += 1.0 / lam[i];
        rhs[i] += st.mu[i] / lam[i];
        lnlam += log(lam[i]);
    }
    for (int i = 0; i < L; ++i)
        for (int j = 0; j < L; ++j) Ainv[i * L + j] = G[i * JK_LMAX + j];
    // Cholesky Ainv = R R^T (R lower, kept in Rl)
    double Rl[JK_LMAX * JK_LMAX];
    for (int q = 0; q < JK_LMAX * JK_LMAX; ++q) Rl[q] = 0.0;
    double lndet = 0.0;
    bool ok = valid;
    for (int j = 0; j < L && ok; ++j) {
        double d = G[j * JK_LMAX + j];
        for (int k = 0; k < j; ++k) d -= Rl[j * JK_LMAX + k] * Rl[j * JK_LMAX + k];
        if (!(d > 0.0)) { ok = false; break; }
        d = sqrt(d);
        Rl[j * JK_LMAX + j] = d;
        lndet += 2.0 * log(d);
        for (int q = j + 1; q < L; ++q) {
            double t = G[q * JK_LMAX + j];
            for (int k = 0; k < j; ++k) t -= Rl[q * JK_LMAX + k] * Rl[j * JK_LMAX + k];
            Rl[q * JK_LMAX + j] = t / d;
        }
    }
    double Am[JK_LMAX * JK_LMAX];
    if (ok) {
        // A = R^-T R^-1 from the lower inverse Ri
        double Ri[JK_LMAX * JK_LMAX];
        for (int q = 0; q < JK_LMAX * JK_LMAX; ++q) Ri[q] = 0.0;
        for (int c = 0; c < L; ++c)
            for (int r = c; r < L; ++r) {
                double t = r == c ? 1.0 : 0.0;
                for (int k = c; k < r; ++k) t -= Rl[r * JK_LMAX + k] * Ri[k * JK_LMAX + c];
                Ri[r * JK_LMAX + c] = t / Rl[r * JK_LMAX + r];
            }
        for (int i = 0; i < L; ++i)
            for (int j = 0; j < L; ++j) {
                double t = 0.0;
                for (int k = (i > j ? i : j); k < L; ++k) t += Ri[k * JK_LMAX + i] * Ri[k * JK_LMAX + j];
                Am[i * JK_LMAX + j] = t;
            }
    } else {
        for (int q = 0; q < JK_LMAX * JK_LMAX; ++q) Am[q] = nan;
    }
    double chi2 = wrr;
    for (int i = 0; i < L; ++i) {
        double ai = 0.0;
        for (int j = 0; j < L; ++j) {
            A[i * L + j] = Am[i * JK_LMAX + j];
            ai = fma(Am[i * JK_LMAX + j], rhs[j], ai);
            chi2 -= v[i] * Am[i * JK_LMAX + j] * v[j];
        }
        a[i] = ai;
    }
    if (B) {
        for (int n = 0; n < N; ++n)
            for (int m = 0; m < N; ++m) {
                double t = 0.0;
                for (int i = 0; i < L; ++i)
                    t = fma(MT[(size_t)i * N + n] * lam[i], MT[(size_t)i * N + m], t);
                if (n == m) {
                    const double iv = st.ivar[n];
                    t += phys ? fma(sv, sv, 1.0 / iv) : 1.0 / iv;
                }
                B[(size_t)n * N + m] = t;
            }
    }
    if (Binv) {
        for (int n = 0; n < N; ++n) {
            const double ivn = st.ivar[n];
            const double wn = phys ? ivn / fma(sv * sv, ivn, 1.0) : ivn;
            for (int m = 0; m < N; ++m) {
                const double ivm = st.ivar[m];
                const double wm = phys ? ivm / fma(sv * sv, ivm, 1.0) : ivm;
                double t = 0.0;
                for (int i = 0; i < L; ++i)
                    for (int j = 0; j < L; ++j)
                        t = fma(MT[(size_t)i * N + n] * Am[i * JK_LMAX + j], MT[(size_t)j * N + m], t);
                Binv[(size_t)n * N + m] = (n == m ? wn : 0.0) - wn * t * wm;
            }
        }
    }
    const double logdet = (double)N * JK_LN_TWO_PI - sum_ln_w + lnlam + lndet;
    double ll = -0.5 * (chi2 + logdet);
    if (!valid) ll = nan;
    else if (!ok) ll = INFINITY;
    sc[0] = ll;
    sc[1] = ok ? chi2 : nan;
    sc[2] = ok ? logdet : nan;
    sc[3] = lam0;
}

hipError_t jk_launch_debug_row(const jk_star *st, const double *row, double *MT, double *Ainv,
                               double *A, double *a, double *b, double *B, double *Binv,
                               double *sc, hipStream_t stream)
{
    hipLaunchKernelGGL(k_debug_row, dim3(1), dim3(64), 0, stream, st->dev, row, MT, Ainv, A, a,
                       b, B, Binv, sc);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Per-sample failure counts of an lnL array (the reference writes +INF when
// its L x L or N x N factorisation fails, fast_likelihood.pyx:283-291,
// 347-348, 381-382, 422-423; invalid rows are NaN here): counts[0] += rows
// at +inf, counts[1] += rows at -inf, counts[2] += NaN rows.  counts is
// cleared by the launcher's first kernel.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_zero_counts3(unsigned long long *counts)
{
    if (threadIdx.x < 3) counts[threadIdx.x] = 0ull;
}

__global__ __launch_bounds__(256) void k_count_failures(const double *__restrict__ ll, int64_t n,
                                                        unsigned long long *__restrict__ counts)
{
    unsigned long long c[3] = {0ull, 0ull, 0ull};
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const double x = ll[i];
        c[0] += x == INFINITY;
        c[1] += x == -INFINITY;
        c[2] += x != x;
    }
    for (int q = 0; q < 3; ++q) {
        unsigned long long t = c[q];
        for (int off = 32; off > 0; off >>= 1) t += __shfl_down(t, off, 64);
        if ((threadIdx.x & 63) == 0 && t) atomicAdd(counts + q, t);
    }
}

hipError_t jk_launch_count_failures(const double *ll, int64_t n, unsigned long long *counts,
                                    hipStream_t stream)
{
    hipLaunchKernelGGL(k_zero_counts3, dim3(1), dim3(256), 0, stream, counts);
    if (n > 0) {
        int64_t blocks = (n + 255) / 256;
        if (blocks > 2048) blocks = 2048;
        hipLaunchKernelGGL(k_count_failures, dim3((unsigned)blocks), dim3(256), 0, stream, ll, n,
                           counts);
    }
    return hipGetLastError();
}
