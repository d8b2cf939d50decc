// Device-side value types and per-column scalar recurrences of the block
// Krylov kernels: shared by the launch-sequence kernels (krylov_kernels.hip)
// and the resident solve (krylov_resident.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "krylov.hpp"

namespace tmi {

// ------------------------------------------------------------ value types
__device__ inline float2 vadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ inline double2 vadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline float vadd(float a, float b) { return a + b; }
__device__ inline double vadd(double a, double b) { return a + b; }
__device__ inline float2 vsub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ inline double2 vsub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ inline float vsub(float a, float b) { return a - b; }
__device__ inline double vsub(double a, double b) { return a - b; }
__device__ inline float2 vmul(float2 a, float2 b) { return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ inline double2 vmul(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ inline float vmul(float a, float b) { return a * b; }
// acc + a * b with four fused multiply-adds (complex) / one (real)
__device__ inline float2 vfma(float2 acc, float2 a, float2 b)
{
    acc.x = __builtin_fmaf(a.x, b.x, acc.x);
    acc.x = __builtin_fmaf(-a.y, b.y, acc.x);
    acc.y = __builtin_fmaf(a.x, b.y, acc.y);
    acc.y = __builtin_fmaf(a.y, b.x, acc.y);
    return acc;
}
__device__ inline double2 vfma(double2 acc, double2 a, double2 b)
{
    acc.x = __builtin_fma(a.x, b.x, acc.x);
    acc.x = __builtin_fma(-a.y, b.y, acc.x);
    acc.y = __builtin_fma(a.x, b.y, acc.y);
    acc.y = __builtin_fma(a.y, b.x, acc.y);
    return acc;
}
__device__ inline float vfma(float acc, float a, float b) { return __builtin_fmaf(a, b, acc); }
__device__ inline double vfma(double acc, double a, double b) { return __builtin_fma(a, b, acc); }
__device__ inline double vmul(double a, double b) { return a * b; }

// acc + c x as four fused multiply-adds (complex) or one (real): the
// accumulation of the SpMM kernels
__device__ inline float2 vmac(float2 acc, float2 c, float2 x)
{
    acc.x = fmaf(c.x, x.x, acc.x);
    acc.x = fmaf(-c.y, x.y, acc.x);
    acc.y = fmaf(c.x, x.y, acc.y);
    acc.y = fmaf(c.y, x.x, acc.y);
    return acc;
}
__device__ inline double2 vmac(double2 acc, double2 c, double2 x)
{
    acc.x = fma(c.x, x.x, acc.x);
    acc.x = fma(-c.y, x.y, acc.x);
    acc.y = fma(c.x, x.y, acc.y);
    acc.y = fma(c.y, x.x, acc.y);
    return acc;
}
__device__ inline float vmac(float acc, float c, float x) { return fmaf(c, x, acc); }
__device__ inline double vmac(double acc, double c, double x) { return fma(c, x, acc); }

// scalar type of a vector element type
template <class V> struct ScalarOf { using type = V; };
template <> struct ScalarOf<float2> { using type = float; };
template <> struct ScalarOf<double2> { using type = double; };
// Multi-frequency operator (MF): the stored coefficient holds the real part
// and the imaginary part at omega = 1 (the mass term); a column at omega w
// uses re + i w im.  Real types and MF = false pass the coefficient through.
template <bool MF, class V>
__device__ inline V mfc(V c, typename ScalarOf<V>::type w)
{
    if constexpr (MF && (std::is_same<V, float2>::value || std::is_same<V, double2>::value)) {
        c.y *= w;
        return c;
    } else {
        (void)w;
        return c;
    }
}
// the column's omega (1 without MF)
template <bool MF, class V>
__device__ inline typename ScalarOf<V>::type mf_omega(const double *omg, int c)
{
    using S = typename ScalarOf<V>::type;
    if constexpr (MF) return (S)omg[c];
    else return (S)1;
}
__device__ inline float2 vscale(float2 a, double s) { float f = (float)s; return make_float2(a.x * f, a.y * f); }
__device__ inline double2 vscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__device__ inline float vscale(float a, double s) { return a * (float)s; }
__device__ inline double vscale(double a, double s) { return a * s; }
__device__ inline double dotR(float2 a, float2 b) { return (double)a.x * (double)b.x + (double)a.y * (double)b.y; }
__device__ inline double dotR(double2 a, double2 b) { return a.x * b.x + a.y * b.y; }
__device__ inline double dotR(float a, float b) { return (double)a * (double)b; }
__device__ inline double dotR(double a, double b) { return a * b; }
// SpMM epilogue dots of one entry: mode 0: d1 += <w, y>_R; mode 1: also
// d2 += <y, y>_R; mode DOT_BIL (complex): d1, d2 += Re, Im of w y
// (unconjugated, COCG's p^T A p)
template <class V>
__device__ inline void dot_epi(V w, V y, int mode, double &d1, double &d2)
{
    if constexpr (std::is_same<V, float2>::value || std::is_same<V, double2>::value) {
        if (mode == DOT_BIL) {
            d1 += (double)w.x * (double)y.x - (double)w.y * (double)y.y;
            d2 += (double)w.x * (double)y.y + (double)w.y * (double)y.x;
            return;
        }
    }
    d1 += dotR(w, y);
    if (mode) d2 += dotR(y, y);
}

// sign pattern of the initial residual (-1, 0, +1 per real component), the
// shadow residual of the mixed-precision BiCGSTAB: any fixed shadow vector
// with <rd, r0> != 0 defines the method, and <sign(r0), r0> = ||r0||_1 > 0.
// On the diffusion systems it needs fewer iterations than rd = r0 (100 vs
// 109 per source at 250k nodes, 61 vs 66 at 103k), and its entries are
// exact in any precision.
__device__ inline float sgn3(float v) { return v > 0.f ? 1.f : (v < 0.f ? -1.f : 0.f); }
__device__ inline double sgn3(double v) { return v > 0.0 ? 1.0 : (v < 0.0 ? -1.0 : 0.0); }
__device__ inline float2 shadow_sign(float2 v) { return make_float2(sgn3(v.x), sgn3(v.y)); }
__device__ inline double2 shadow_sign(double2 v) { return make_double2(sgn3(v.x), sgn3(v.y)); }
__device__ inline float shadow_sign(float v) { return sgn3(v); }
__device__ inline double shadow_sign(double v) { return sgn3(v); }

// The shadow residual of a 64-column complex FP32 tile packed to 4 bits per
// entry (2 per real component: 0 -> 0, 1 -> +1, 3 -> -1), 32 bytes per row
// instead of 512: the kernels that stream it every iteration (the dot of
// the first SpMM, the x/r update) read the packed copy, the others the FP32
// one; both hold the same values, so every dot is bit-identical.
__device__ inline unsigned sh_code(float x) { return x > 0.f ? 1u : (x < 0.f ? 3u : 0u); }
__device__ inline float sh_val(unsigned b) { return (b & 1u) ? ((b & 2u) ? -1.f : 1.f) : 0.f; }
__device__ inline float2 sh_unpack(const unsigned char *__restrict__ q, size_t row, int c)
{
    const unsigned nib = (q[row * 32 + (c >> 1)] >> ((c & 1) * 4)) & 15u;
    return make_float2(sh_val(nib & 3u), sh_val(nib >> 2));
}

template <class V> __device__ inline V vzero();
template <> __device__ inline float2 vzero<float2>() { return make_float2(0.f, 0.f); }
template <> __device__ inline double2 vzero<double2>() { return make_double2(0.0, 0.0); }
template <> __device__ inline float vzero<float>() { return 0.f; }
template <> __device__ inline double vzero<double>() { return 0.0; }
__device__ inline float2 to32(double2 a) { return make_float2((float)a.x, (float)a.y); }
__device__ inline float to32(double a) { return (float)a; }
__device__ inline double2 to64(float2 a) { return make_double2(a.x, a.y); }
__device__ inline double to64(float a) { return a; }
__device__ inline double2 to64(double2 a) { return a; }
__device__ inline double to64(double a) { return a; }
__device__ inline float2 cvt32(double2 a) { return make_float2((float)a.x, (float)a.y); }
__device__ inline float cvt32(double a) { return (float)a; }
template <class To> __device__ inline To cvt(double2 a);
template <> __device__ inline float2 cvt<float2>(double2 a) { return make_float2((float)a.x, (float)a.y); }
template <> __device__ inline double2 cvt<double2>(double2 a) { return a; }
template <class To> __device__ inline To cvt(double a);
template <> __device__ inline float cvt<float>(double a) { return (float)a; }
template <> __device__ inline double cvt<double>(double a) { return a; }
__device__ inline float2 shfl_add(float2 a, int off) { a.x += __shfl_xor(a.x, off); a.y += __shfl_xor(a.y, off); return a; }
__device__ inline double2 shfl_add(double2 a, int off) { a.x += __shfl_xor(a.x, off); a.y += __shfl_xor(a.y, off); return a; }
__device__ inline float shfl_add(float a, int off) { return a + __shfl_xor(a, off); }
__device__ inline double shfl_add(double a, int off) { return a + __shfl_xor(a, off); }

// complex value times a complex scalar (ar + i ai)
__device__ inline float2 cscale(float2 v, double ar, double ai)
{
    const float a = (float)ar, b = (float)ai;
    return make_float2(v.x * a - v.y * b, v.x * b + v.y * a);
}
__device__ inline double2 cscale(double2 v, double ar, double ai)
{
    return make_double2(v.x * ar - v.y * ai, v.x * ai + v.y * ar);
}
// unconjugated product terms: re and im of a b
template <class V>
__device__ inline void bil_add(V a, V b, double &re, double &im)
{
    if constexpr (std::is_same<V, float2>::value || std::is_same<V, double2>::value) {
        re += (double)a.x * (double)b.x - (double)a.y * (double)b.y;
        im += (double)a.x * (double)b.y + (double)a.y * (double)b.x;
    } else {
        re += (double)a * (double)b;
    }
}

// z = D^-1 r for column c.  Without omg, di is the row's inverse diagonal;
// with omg (multi-frequency solve), di is the row's diagonal entry with its
// imaginary part at omega = 1 and the column's diagonal is re + i omg[c] im.
template <class V>
__device__ inline V prec_apply(V di, V r, const double *__restrict__ omg, int c)
{
    if constexpr (std::is_same<V, float2>::value || std::is_same<V, double2>::value) {
        if (omg) {
            using S = typename ScalarOf<V>::type;
            const S a = di.x, b = di.y * (S)omg[c], den = a * a + b * b;
            V z;
            z.x = (r.x * a + r.y * b) / den;
            z.y = (r.y * a - r.x * b) / den;
            return z;
        }
    }
    return vmul(di, r);
}

// (cr + i ci) = (ar + i ai) / (br + i bi); false when the quotient is not finite
__device__ inline bool cdiv(double ar, double ai, double br, double bi, double &cr, double &ci)
{
    const double den = br * br + bi * bi;
    cr = (ar * br + ai * bi) / den;
    ci = (ai * br - ar * bi) / den;
    return den != 0.0 && isfinite(cr) && isfinite(ci);
}

// The scalar recurrence of one column after a reduction (r0, r1, r2: the
// summed partials); S and I hold the column's scalar and flag slots
// (I[I_NSLOT]: the outer solve's active flag).
__device__ inline void fin_column(int fk, double r0, double r1, double r2, double *S, int *I, int maxit, double tol2)
{
#define SC(slot) S[slot]
#define IC(slot) I[slot]
    switch (fk) {
    case FIN_OUTER_BNORM:
        SC(S_BNORM2) = r0;
        SC(S_SCALE) = r0 > 0.0 ? 1.0 / sqrt(r0) : 1.0;
        SC(S_BEST) = -1.0;
        IC(I_STALL) = 0;
        if (r0 == 0.0) IC(I_ACTIVE) = 0;   // zero right-hand side: the field stays at the initial guess
        break;
    case FIN_OUTER_RES: {
        if (!IC(I_ACTIVE)) break;
        SC(S_RES2) = r0;
        IC(I_ITERS) += 1;   // true-residual evaluations
        if (r0 <= tol2 * SC(S_BNORM2) || !isfinite(r0)) { IC(I_ACTIVE) = 0; break; }
        // stagnation: no 2x drop of the true residual norm over 8 evaluations
        if (SC(S_BEST) < 0.0 || r0 < 0.25 * SC(S_BEST)) { SC(S_BEST) = r0; IC(I_STALL) = 0; }
        else if (++IC(I_STALL) >= 8) IC(I_ACTIVE) = 0;
        break;
    }
    case FIN_BICG_RELIABLE:
    case FIN_CG_RELIABLE: {
        const int oact = I[I_NSLOT];
        if (!oact) { IC(I_ACTIVE) = 0; break; }
        SC(S_RES2) = r0;
        if (fk == FIN_BICG_RELIABLE) {
            // recompute beta of the coming iteration with the replaced residual
            if (!IC(I_FIRST) && SC(S_RHOP) != 0.0 && SC(S_OMEGA) != 0.0 && r1 != 0.0 && isfinite(r1))
                SC(S_BETA) = (r1 * SC(S_ALPHA)) / (SC(S_RHOP) * SC(S_OMEGA));
            else
                IC(I_FIRST) = 1;   // breakdown or not started: restart the directions from r
            SC(S_RHO) = r1;
        } else {
            // PCG: the replacement sits between the beta step and the
            // direction update d = beta d + D^-1 r, so beta is recomputed
            // from the replaced residual
            SC(S_RHO) = r1;
            if (SC(S_RHOP) != 0.0 && isfinite(r1) && !IC(I_FIRST)) SC(S_BETA) = r1 / SC(S_RHOP);
            else IC(I_FIRST) = 1;
        }
        if (IC(I_BREAK)) { IC(I_FIRST) = 1; IC(I_BREAK) = 0; }
        IC(I_ACTIVE) = 1;
        if (maxit > 0 && IC(I_ITERS) >= maxit) IC(I_ACTIVE) = 0;
        break;
    }
    case FIN_BICG_INIT:
    case FIN_CG_INIT:
        if (!IC(I_ACTIVE)) break;
        SC(S_BNORM2) = 1.0;   // the inner system is scaled by 1/||b||: absolute criterion
        SC(S_RES2) = (fk == FIN_BICG_INIT) ? r0 : r1;
        SC(S_RHO) = (fk == FIN_BICG_INIT) ? r1 : r0;
        IC(I_FIRST) = 1;
        IC(I_BREAK) = 0;
        if (SC(S_RES2) <= SC(S_TOL2)) IC(I_ACTIVE) = 0;
        break;
    case FIN_BICG_ALPHA: {
        if (!IC(I_ACTIVE)) break;
        double alpha = SC(S_RHO) / r0;
        if (r0 == 0.0 || !isfinite(alpha)) { IC(I_ACTIVE) = 0; IC(I_BREAK) = 1; alpha = 0.0; }
        SC(S_ALPHA) = alpha;
        break;
    }
    case FIN_BICG_OMEGA: {
        if (!IC(I_ACTIVE)) break;
        double om = (r1 == 0.0) ? 0.0 : r0 / r1;
        if (!isfinite(om)) om = 0.0;
        SC(S_OMEGA) = om;
        break;
    }
    case FIN_BICG_RHO: {
        if (!IC(I_ACTIVE)) break;
        IC(I_ITERS) += 1;
        IC(I_FIRST) = 0;
        SC(S_RES2) = r0;
        const double rho_new = r1;
        SC(S_RHOP) = SC(S_RHO);
        if (r0 <= SC(S_TOL2)) { IC(I_ACTIVE) = 0; break; }
        if (SC(S_OMEGA) == 0.0 || rho_new == 0.0 || !isfinite(r0)) { IC(I_ACTIVE) = 0; IC(I_BREAK) = 1; break; }
        if (maxit > 0 && IC(I_ITERS) >= maxit) { IC(I_ACTIVE) = 0; break; }
        SC(S_BETA) = (rho_new * SC(S_ALPHA)) / (SC(S_RHO) * SC(S_OMEGA));
        SC(S_RHOP) = SC(S_RHO);
        SC(S_RHO) = rho_new;
        break;
    }
    case FIN_CG_ALPHA: {
        if (!IC(I_ACTIVE)) break;
        double alpha = SC(S_RHO) / r0;
        if (alpha == 0.0 || !isfinite(alpha)) { IC(I_ACTIVE) = 0; IC(I_BREAK) = 1; alpha = 0.0; }
        SC(S_ALPHA) = alpha;
        break;
    }
    case FIN_CG_BETA: {
        if (!IC(I_ACTIVE)) break;
        IC(I_ITERS) += 1;
        IC(I_FIRST) = 0;
        const double dold = SC(S_RHO), dnew = r0;
        const double beta = dnew / dold;
        SC(S_RHOP) = dold;
        SC(S_RHO) = dnew;
        SC(S_BETA) = beta;
        SC(S_RES2) = r1;
        if (beta == 0.0 || !isfinite(beta)) { IC(I_ACTIVE) = 0; IC(I_BREAK) = 1; break; }
        if (r1 <= SC(S_TOL2)) { IC(I_ACTIVE) = 0; break; }
        if (maxit > 0 && IC(I_ITERS) >= maxit) { IC(I_ACTIVE) = 0; break; }
        break;
    }
    // COCG: rho, alpha, beta are complex (real part in the slot, imaginary
    // part in its _I slot); r0, r1 = re, im of a bilinear product, r2 = ||r||^2
    case FIN_COCG_INIT:
        if (!IC(I_ACTIVE)) break;
        SC(S_BNORM2) = 1.0;   // the inner system is scaled by 1/||b||: absolute criterion
        SC(S_RES2) = r2;
        SC(S_RHO) = r0;
        SC(S_RHO_I) = r1;
        IC(I_FIRST) = 1;
        IC(I_BREAK) = 0;
        if (r2 <= SC(S_TOL2)) IC(I_ACTIVE) = 0;
        break;
    case FIN_COCG_ALPHA: {
        // I_XPEND: the columns whose x update this iteration owes, the ones
        // the update kernel runs for (the direction update applies it when
        // the update kernel defers it)
        IC(I_XPEND) = 0;
        if (!IC(I_ACTIVE)) break;
        double ar, ai;
        if (!cdiv(SC(S_RHO), SC(S_RHO_I), r0, r1, ar, ai) || (ar == 0.0 && ai == 0.0)) {
            IC(I_ACTIVE) = 0;
            IC(I_BREAK) = 1;
            ar = ai = 0.0;
        }
        SC(S_ALPHA) = ar;
        SC(S_ALPHA_I) = ai;
        IC(I_XPEND) = IC(I_ACTIVE);
        break;
    }
    case FIN_COCG_BETA: {
        if (!IC(I_ACTIVE)) break;
        IC(I_ITERS) += 1;
        IC(I_FIRST) = 0;
        double br, bi;
        const bool ok = cdiv(r0, r1, SC(S_RHO), SC(S_RHO_I), br, bi);
        SC(S_RHOP) = SC(S_RHO);
        SC(S_RHOP_I) = SC(S_RHO_I);
        SC(S_RHO) = r0;
        SC(S_RHO_I) = r1;
        SC(S_BETA) = br;
        SC(S_BETA_I) = bi;
        SC(S_RES2) = r2;
        if (!ok || (br == 0.0 && bi == 0.0)) { IC(I_ACTIVE) = 0; IC(I_BREAK) = 1; break; }
        if (r2 <= SC(S_TOL2)) { IC(I_ACTIVE) = 0; break; }
        if (maxit > 0 && IC(I_ITERS) >= maxit) { IC(I_ACTIVE) = 0; break; }
        break;
    }
    case FIN_COCG_RELIABLE: {
        // the replacement sits between the beta step and the direction
        // update, so beta is recomputed from the replaced residual
        if (!I[I_NSLOT]) { IC(I_ACTIVE) = 0; break; }
        SC(S_RES2) = r2;
        SC(S_RHO) = r0;
        SC(S_RHO_I) = r1;
        double br, bi;
        if (!IC(I_FIRST) && cdiv(r0, r1, SC(S_RHOP), SC(S_RHOP_I), br, bi)) {
            SC(S_BETA) = br;
            SC(S_BETA_I) = bi;
        } else {
            IC(I_FIRST) = 1;
        }
        if (IC(I_BREAK)) { IC(I_FIRST) = 1; IC(I_BREAK) = 0; }
        IC(I_ACTIVE) = 1;
        if (maxit > 0 && IC(I_ITERS) >= maxit) IC(I_ACTIVE) = 0;
        break;
    }
    }
#undef SC
#undef IC
}

}  // namespace tmi
