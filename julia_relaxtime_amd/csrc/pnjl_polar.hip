// pnjl_polar.hip -- the anisotropic one-loop polarization Pi(k0, k) on gfx950.
//
// One lane, or a group of them, evaluates one B0 / B0_correction /
// polarization value with the reference's fixed quadrature: the same
// breakpoints (poles of the k = 0 integrand, roots of the k > 0 logarithm,
// imaginary-part intervals), the same 16/32-node power-clustered and 33-node
// double-exponential rules, the same principal-value subtraction and the same
// skip-non-finite rule, so the results reproduce the reference's numbers, not
// the exact integrals.  All of it is FP64 arithmetic on tables in LDS, bound
// by instruction issue: B0's terms that differ only in the distribution's
// sign are evaluated together, every rule and integrand of an evaluation goes
// through one node loop, and the nodes' functions are table-driven.  On six
// 256-point x 3 pairs x 128 k0 x 64 k grids a call takes 10.6 to 11.2 ms (29.1
// to 31.0 with one loop per rule, term by term, on the library's functions).  For the
// grid call, the threads of a wavefront share (point, pair) and take an 8 x 8
// tile of (k0, k), so their segment structures differ only smoothly; the
// propagator batch sorts its work into buckets of similar (pair, mass,
// lambda, k) for the same reason.
//
// Follows src/relaxtime/OneLoopIntegrals.jl, OneLoopIntegralsAniso.jl,
// PolarizationAniso.jl, src/integration/IntervalQuadratureStrategies.jl and
// src/QuarkDistribution{,_Aniso}.jl (file:line at each function).
#include <hip/hip_runtime.h>

#include <math.h>
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "pnjl_ctx.h"

using namespace pnjl_host;

// No contraction of a*b + c into FMA here: the reference evaluates these
// expressions unfused, and some of them cancel exactly (lambda^2 + m^2 - m'^2
// with m = m'), where a fused product leaves a 1e-17 residue instead of 0.
#pragma clang fp contract(off)

#include "pnjl_meson.h"

namespace polar {

constexpr double kPi = 3.14159265358979323846;
constexpr double kEpsK = 1.0e-9;        // OneLoopIntegrals.jl:23
constexpr double kEpsSeg = 1.0e-12;     // OneLoopIntegrals.jl:24
constexpr double kPvGapRel = 1e-6;      // OneLoopIntegrals.jl:35
constexpr double kAlpha = 0.35;         // IntervalQuadratureStrategies.jl:35
constexpr double kDeH = 0.15;           // IntervalQuadratureStrategies.jl:36

// ---- tables ------------------------------------------------------------------
// The quadrature kernels' tables in LDS, one array per kernel: addressed from
// the array itself everywhere (a pointer passed to an out-of-line routine
// would be generic: flat loads).  Layout: 2^(j/64) [64] (pnjl::exp_tab), pairs
// (1/c_j, log c_j) [128] (log_p), then the rules, each as nodes t[n] and
// weights w[n] of sum_i s w_i f(x0 + s t_i).
constexpr int kPLog = 64;
constexpr int kPRules = kPLog + 256;
// power-clustered left / right (x0 = a, s = b - a), double exponential and
// Gauss-Legendre (x0 = centre, s = half length)
enum { R_L16 = kPRules, R_L32 = R_L16 + 32, R_R32 = R_L32 + 64, R_DE = R_R32 + 64, R_G16 = R_DE + 66, R_G32 = R_G16 + 32 };
constexpr int kTabLen = R_G32 + 64;
__shared__ double ptab[kTabLen];

struct Phys {
    double Lambda, Nc;
};

// Julia eps(x): spacing of doubles at |x|
__device__ __forceinline__ double jeps(double x)
{
    x = fabs(x);
    if (!(x >= 2.2250738585072014e-308)) return 4.9406564584124654e-324;
    return ldexp(1.0, ilogb(x) - 52);
}

__device__ __forceinline__ double jsign(double x) { return x > 0 ? 1.0 : (x < 0 ? -1.0 : x); }
__device__ __forceinline__ double clamp_e(double e) { return e < 1e-200 ? 1e-200 : (e > 1e200 ? 1e200 : e); }

// ---- arithmetic of the node loops ----------------------------------------------
// The quadratures are bound by the FP64 instructions of their nodes (a square
// root, an exponential, a logarithm and quotients each).  The helpers below
// round like the library's within a bit, without its scaling and special
// cases, which the callers' tests cover.

// sqrt(x), NaN for x < 0: v_rsq_f64 estimate, one Goldschmidt step and a
// residual correction (Markstein, IA-64 and Elementary Functions, 2000)
__device__ __forceinline__ double sqrt_p(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double e = fma(-g, h, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    g = fma(fma(-g, g, x), h, g);
    return x == 0.0 ? 0.0 : g;
}

// 1/d to about 2^-45 (v_rcp_f64 and one Newton step)
__device__ __forceinline__ double rcp1(double d)
{
    const double r = __builtin_amdgcn_rcp(d);
    return fma(r, fma(-d, r, 1.0), r);
}

// n/d from r ~ 1/d: the residual correction leaves about half an ulp
__device__ __forceinline__ double div_r(double n, double d, double r)
{
    const double q = n * r;
    return fma(fma(-d, q, n), r, q);
}
__device__ __forceinline__ double div_p(double n, double d) { return div_r(n, d, rcp1(d)); }

// exp(x) as pnjl::exp_tab (Tang's table method, x clamped to [-800, 700]) with
// the table entry added last: within about 0.6 ulp
__device__ __forceinline__ double exp_p(double x)
{
    x = fmin(fmax(x, -800.0), 700.0);
    const double nd = rint(x * 0x1.71547652b82fep+6);   // 64 / ln 2
    double r = fma(nd, -0x1.62e42fee00000p-7, x);       // ln 2 / 64, split
    r = fma(nd, -0x1.a39ef35793c76p-39, r);
    const int n = (int)nd;
    double p = pnjl::fma_k(r, 1.0 / 120.0, 1.0 / 24.0);
    p = pnjl::fma_k(r, p, 1.0 / 6.0);
    p = fma(r, p, 0.5);
    p = fma(r * r, p, r);   // e^r - 1
    const double t = ptab[pnjl::kExpTab + (n & 63)];
    return ldexp(fma(t, p, t), n >> 6);
}

// log(x), x > 0 normal (Tang, ACM TOMS 16(4), 1990, on 128 intervals of [1,
// 2)): the upper half counts as [1/2, 1) of the next binade and the intervals
// next to 1 have c_j = 1, so the result keeps its relative accuracy near x = 1.
__device__ __forceinline__ double log_p(double x)
{
    const double ln2_hi = 0x1.62e42fee00000p-1;
    const double ln2_lo = 0x1.a39ef35793c76p-33;
    int e;
    const double m = 2.0 * frexp(x, &e);   // [1, 2)
    const int j = (int)((uint32_t)(__double2hiint(m)) >> 13) & 127;
    const double inv = ptab[kPLog + 2 * j], lc = ptab[kPLog + 2 * j + 1];
    const double r = fma(m, inv, -1.0);
    double p = pnjl::fma_k(r, -1.0 / 8.0, 1.0 / 7.0);
    p = pnjl::fma_k(r, p, -1.0 / 6.0);
    p = pnjl::fma_k(r, p, 1.0 / 5.0);
    p = pnjl::fma_k(r, p, -0.25);
    p = pnjl::fma_k(r, p, 1.0 / 3.0);
    p = fma(r, p, -0.5);
    const double ed = (double)(e - 1 + (j >> 6));
    return fma(ed, ln2_hi, lc) + (r + fma(r * r, p, ed * ln2_lo));
}

// log(x) of any x >= 0 or NaN, subnormal x excepted
__device__ __forceinline__ double log_c(double x)
{
    const double v = log_p(x);
    return x > 0.0 && x <= 1.7976931348623157e308 ? v : (x == 0.0 ? -__builtin_inf() : x);
}

// PNJL distributions and their antiderivatives  QuarkDistribution.jl:14-99
// The medium of one evaluation.  joint: |mu|/T < 150, so one exponential
// serves quark and antiquark (exp(-(E + mu)/T) = exp(-(E - mu)/T) exp(-2
// mu/T)) without leaving the range; otherwise each has its own.
struct Medium {
    double mu, T, beta, K2, Phi, Phib;
    bool joint;
};

__device__ __forceinline__ Medium make_medium(double mu, double T, double Phi, double Phib)
{
    Medium M{mu, T, 1 / T, 0.0, Phi, Phib, false};
    M.joint = M.beta > 0.0 && M.beta < 1e300 && fabs(mu) * M.beta < 150.0;
    M.K2 = exp_p(-2.0 * mu * M.beta);
    return M;
}

// exp(-(E - mu)/T) and exp(-(E + mu)/T), clamped to [1e-200, 1e200]
__device__ __forceinline__ void boltzmann(const Medium& M, double E, double& ep, double& em)
{
    const double x = (M.mu - E) * M.beta;
    const double t = exp_p(x);
    ep = clamp_e(t);
    em = clamp_e(t * M.K2);
    if (!M.joint) {
        const double y = -(E + M.mu) * M.beta;
        em = y != y ? y : clamp_e(exp_p(y));   // a NaN exponent stays one
        ep = x != x ? x : ep;
    }
}

// the distributions of both B0 signs, f(E) and 1 - fbar(E) (f+(-E) = 1 - f-(E))
//   distribution_value_b0  OneLoopIntegrals.jl:68-83
__device__ __forceinline__ void dist2(const Medium& M, double E, double& dp, double& dm)
{
    double ep, em;
    boltzmann(M, E, ep, em);
    const double p2 = ep * ep, p3 = p2 * ep, m2 = em * em, m3 = m2 * em;
    const double np = M.Phi * ep + 2 * M.Phib * p2 + p3, nm = M.Phib * em + 2 * M.Phi * m2 + m3;
    const double Dp = 1 + 3 * M.Phi * ep + 3 * M.Phib * p2 + p3, Dm = 1 + 3 * M.Phib * em + 3 * M.Phi * m2 + m3;
    dp = div_p(np, Dp);
    dm = 1.0 - div_p(nm, Dm);
}

// antiderivatives of both distributions at E: -T ln(1 + 3 c1 e + 3 c2 e^2 + e^3) / 3
__device__ __forceinline__ void anti2(const Medium& M, double E, double& ap, double& am)
{
    double ep, em;
    boltzmann(M, E, ep, em);
    const double p2 = ep * ep, m2 = em * em;
    const double dp = 1 + 3 * M.Phi * ep + 3 * M.Phib * p2 + p2 * ep, dm = 1 + 3 * M.Phib * em + 3 * M.Phi * m2 + m2 * em;
    ap = -M.T * log_c(dp <= 1e-300 ? 1e-300 : dp) / 3;
    am = -M.T * log_c(dm <= 1e-300 ? 1e-300 : dm) / 3;
}

// energy_cutoff / internal_momentum  OneLoopIntegrals.jl:37-48
__device__ __forceinline__ double e_cut(const Phys& P, double m)
{
    double mp = m > 0 ? m : 0.0;
    return sqrt_p(mp * mp + P.Lambda * P.Lambda);
}

__device__ __forceinline__ double p_int(double E, double m)
{
    double mp = m > 0 ? m : 0.0;
    return sqrt_p(E * E - mp * mp);
}

// A segment of a piecewise rule: sum over the rule's nodes of s w_i f(x0 + s t_i);
// n = 0 where the segment is empty (integrate_hybrid_interval returns 0 for
// b <= a and for ends that are not finite).
struct Seg {
    double x0, s;
    int off, n;
};
__device__ __forceinline__ Seg seg_power(double a, double b, int off, int n)
{
    return Seg{a, b - a, off, (isfinite(a) && isfinite(b) && b > a) ? n : 0};
}
// by value: a choice between the objects themselves would keep them in memory
__device__ __forceinline__ double pick(bool c, double a, double b) { return c ? a : b; }
__device__ __forceinline__ Seg seg_pick(bool c, Seg a, Seg b)
{
    return Seg{pick(c, a.x0, b.x0), pick(c, a.s, b.s), c ? a.off : b.off, c ? a.n : b.n};
}
__device__ __forceinline__ Seg seg_mid(double a, double b, int off, int n)
{
    return Seg{(a + b) / 2, (b - a) / 2, off, (isfinite(a) && isfinite(b) && b > a) ? n : 0};
}

// ---- B~0 for both distribution signs ---------------------------------------------
// One evaluation at (lambda, k, m, m') gives B~0 with f(E) ("plus") and with
// 1 - fbar(E) ("minus"): the two integrals have the same poles, breakpoints
// and nodes and share everything but the distribution, and B0 of equal masses
// (or its average over +-k0) needs both at the same lambda.  The nodes of all
// of an evaluation's segments run through one loop, whichever rule and
// integrand a lane has, so the lanes of a wavefront do not wait for each
// other's branches.
//
// L > 1: the L consecutive lanes of a group evaluate the nodes i = q, q + L,
// ... of a segment (q the lane's number in the group) and leave the terms in
// the group's LDS row, then every lane adds them in the order of the nodes --
// the one-lane loop's sums, bit for bit.  Control flow is uniform in a group
// (same arguments on every lane), and a group's lanes are in one wavefront,
// whose LDS accesses complete in program order.
constexpr int kRowTerms = 33;   // terms of the longest rule

template <int L>
__device__ __forceinline__ double2* term_rows()
{
    __shared__ double2 rows[L > 1 ? 256 / L * kRowTerms : 1];
    return rows + (L > 1 ? threadIdx.x / L * kRowTerms : 0);
}

// acc += the n terms of the segment, in order, on every lane of the group
template <int L>
__device__ __forceinline__ void add_terms(int n, double& ap, double& am)
{
    const double2* row = term_rows<L>();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // n = 16, 32 or 33: the loads of four terms issue together
#pragma unroll 1
    for (int b = 0; b + 4 <= n; b += 4) {
        double2 t[4];
#pragma unroll
        for (int j = 0; j < 4; j++) t[j] = row[b + j];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            ap += t[j].x;
            am += t[j].y;
        }
    }
    if (n & 1) {
        ap += row[n - 1].x;
        am += row[n - 1].y;
    }
    // the row is written again only after every lane has read it
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
struct Pair {
    double rp, ip, rm, im;   // plus: real, imaginary; minus
};

// singularity_k_positive  OneLoopIntegrals.jl:239-330 -> number of intervals in iv (0..2)
__device__ int sing_kpos(double lam, double k, double m, double mp, double Emin, double Emax, double iv[2][2])
{
    int n = 0;
    const double a = lam * lam - k * k;
    const double d0 = k * k - lam * lam;
    const double denom = 2.0 * d0;
    if (fabs(a) < kEpsSeg) {
        if (lam > 0.0 && mp > m) {
            double m2d = mp * mp - m * m;
            double Ec = m2d / (4.0 * lam) + lam * m * m / m2d;
            if (Ec < Emax) {
                iv[0][0] = fmax(Ec, Emin);
                iv[0][1] = Emax;
                n = 1;
            }
        }
        return n;
    }
    const double A = lam * lam - k * k + m * m - mp * mp;
    const double disc = A * A + 4.0 * m * m * d0;
    if (disc < 0.0) return 0;
    const double sq = sqrt_p(disc);
    double E1 = (lam * A - k * sq) / denom, E2 = (lam * A + k * sq) / denom;
    if (E1 > E2) {
        double t = E1;
        E1 = E2;
        E2 = t;
    }
    if (E2 - E1 < kEpsSeg) return 0;
    if (a > 0.0) {
        if (E2 > Emin && E1 < Emax) {
            double c1 = fmax(E1, Emin), c2 = fmin(E2, Emax);
            if (c2 > c1) {
                iv[0][0] = c1;
                iv[0][1] = c2;
                n = 1;
            }
        }
        return n;
    }
    // the intervals of this branch are [Emin, c1] and [c2, Emax], stored as such
    const double c1 = E1 > Emin ? fmin(E1, Emax) : Emin, c2 = E2 < Emax ? fmax(E2, Emin) : Emax;
    const bool low = c1 > Emin, high = Emax > c2;
    iv[0][0] = low ? Emin : c2;
    iv[0][1] = low ? c1 : Emax;
    iv[1][0] = c2;
    iv[1][1] = Emax;
    return (low ? 1 : 0) + (high ? 1 : 0);
}

// lam_m: the minus term's own lambda, equal to lam or to its last bits (lambda
// = +-k0 + mu1 - mu2 rounds differently for the two signs of k0).  At rest and
// on a threshold, E0 = m, whether p(E0) exists hangs on those bits (a pole
// search started there ends or not), so each sign takes its own.
template <int L>
__device__ Pair tilde_B0(const Phys& P, const Medium& M, double lam, double lam_m, double k, double m_in, double mp_in,
                         int q)
{
    const double m = m_in > 0 ? m_in : 0.0, mp = mp_in > 0 ? mp_in : 0.0;
    const double Emin = m, Emax = e_cut(P, m);
    const bool at_rest = fabs(k) < kEpsK;
    // integrand: RATIO  f(E) ln|num / den| (k > 0); POLE  p f(E) / (lambda E + d);
    // REGULAR  (p f(E) - f0) / (E - E0), the principal value's regular part
    enum { RATIO, POLE, REGULAR };
    int form = RATIO;
    Seg sg[3] = {};
    Pair o{0.0, 0.0, 0.0, 0.0};          // what is not a node sum
    double scale = 1.0;                  // of the node sums
    double dterm = 0.0, E0 = 0.0, f0p = 0.0, f0m = 0.0, near = 0.0, wnear = 0.0;
    if (at_rest) {
        // OneLoopIntegrals.jl:117-224
        form = POLE;
        scale = 2.0;
        dterm = (lam * lam + m * m - mp * mp) / 2.0;
        E0 = -dterm / lam;
        bool has = false;
        if (isfinite(E0)) {   // singularity_k_zero  :144-157
            const double tol = 1e-8 * fmax(1.0, fabs(E0));
            has = (E0 > Emin - tol) && (E0 < Emax + tol);
        }
        if (!has) {
            sg[2] = seg_power(Emin, Emax, R_L16, 16);
            o.ip = o.im = 0.0 / lam;
        } else {
            double dp, dm;
            dist2(M, E0, dp, dm);
            const double p0 = p_int(E0, m), ps = isfinite(p0) ? p0 : 0.0;
            f0p = isfinite(ps * dp) ? ps * dp : 0.0;
            f0m = isfinite(ps * dm) ? ps * dm : 0.0;
            const double etol = 1e-10 * fmax(1.0, Emax - Emin);
            if (fabs(E0 - Emin) <= etol || fabs(Emax - E0) <= etol) {
                const double gap = fmax(kPvGapRel * (Emax - Emin), 64 * jeps(E0));
                const double left_end = fmax(Emin, E0 - gap), right_start = fmin(Emax, E0 + gap);
                if (left_end > Emin) sg[1] = seg_power(Emin, left_end, R_L16, 16);
                if (right_start < Emax) sg[2] = seg_power(right_start, Emax, R_L16, 16);
            } else {
                form = REGULAR;
                near = 64 * jeps(E0);
                sg[0] = seg_power(Emin, Emax, R_L32, 32);
                const double lt = log_c(fabs(Emax - E0)) - log_c(fabs(Emin - E0));
                scale = 2.0 / lam;
                o.rp = f0p * lt * scale;
                o.rm = f0m * lt * scale;
            }
            const double E0m = -((lam_m * lam_m + m * m - mp * mp) / 2.0) / lam_m;
            const double c = 2.0 * kPi / lam;
            o.ip = c * p0 * dp;
            o.im = c * p_int(E0m, m) * dm;
        }
    } else {
        // OneLoopIntegrals.jl:228-476: integrate_piecewise_hybrid's breakpoints :335-421
        double iv[2][2] = {};
        const int niv = sing_kpos(lam, k, m, mp, Emin, Emax, iv);
        scale = 1.0 / k;
        if (niv == 0) {
            sg[2] = seg_power(Emin, Emax, R_L16, 16);
        } else {
            double E1 = iv[0][0], E2 = iv[0][1];
            if (niv == 2) {
                const double tol = 1e-12 * fmax(1.0, Emax - Emin);
                E1 = iv[0][1];
                E2 = pick(fabs(iv[0][1] - Emax) <= tol, iv[0][0], iv[1][0]);
            }
            if (E1 > Emin) sg[0] = seg_power(Emin, E1, R_R32, 32);
            if (E2 > E1) sg[1] = seg_mid(E1, E2, R_DE, 33);
            if (Emax > E2) sg[2] = seg_power(E2, Emax, R_L16, 16);
            double sp = 0.0, sm = 0.0;
#pragma unroll 1
            for (int i = 0; i < niv; i++) {
                const double a = pick(i != 0, iv[1][0], iv[0][0]), b = pick(i != 0, iv[1][1], iv[0][1]);
                double apa, ama, apb, amb;
                anti2(M, a, apa, ama);
                anti2(M, b, apb, amb);
                sp += apb - apa;
                sm += (b - a) - (amb - ama);
            }
            const double c = kPi * jsign(lam);
            o.ip = sp * c / k;
            o.im = sm * c / k;
        }
    }
    double accp = 0.0, accm = 0.0;
#pragma unroll 1
    for (int g = 0; g < 3; g++) {
        const Seg S = seg_pick(g == 0, sg[0], seg_pick(g == 1, sg[1], sg[2]));
#pragma unroll 1
        for (int i = q; i < S.n; i += L) {
            const double E = S.x0 + S.s * ptab[S.off + i];
            const double w = S.s * ptab[S.off + S.n + i];
            const double p = p_int(E, m);
            double dp, dm, vp, vm;
            dist2(M, E, dp, dm);
            if (form == RATIO) {
                const double lpE = lam + E;
                const double common = lpE * lpE - mp * mp;
                const double pmk = p - k, ppk = p + k;
                const double num = common - pmk * pmk;
                double den = common - ppk * ppk;
                const bool tiny = fabs(den) < kEpsSeg;
                const bool ok = isfinite(num) && isfinite(den) && !(tiny && fabs(num) < kEpsSeg);
                if (tiny) den = (den == 0.0) ? kEpsSeg : jsign(den) * kEpsSeg;
                const double ratio = fabs(div_p(num, den));
                const double lt = (ok && isfinite(ratio)) ? log_p(fmax(ratio, 1e-300)) : 0.0;
                vp = dp * lt;
                vm = dm * lt;
            } else {
                vp = p * dp;
                vm = p * dm;
                double d = lam * E + dterm;
                if (form == REGULAR) {
                    d = E - E0;
                    vp = (isfinite(vp) ? vp : 0.0) - f0p;
                    vm = (isfinite(vm) ? vm : 0.0) - f0m;
                    if (fabs(d) < near) {   // takes the difference quotient, below
                        wnear += w;
                        vp = vm = 0.0;
                        d = 1.0;
                    }
                } else if (!isfinite(d) || fabs(d) < kEpsSeg) {
                    vp = vm = 0.0;
                    d = 1.0;
                }
                const double r = rcp1(d);
                vp = div_r(vp, d, r);
                vm = div_r(vm, d, r);
            }
            const double tp = isfinite(vp) ? w * vp : 0.0, tm = isfinite(vm) ? w * vm : 0.0;
            if constexpr (L > 1) {
                term_rows<L>()[i] = double2{tp, tm};
            } else {
                accp += tp;
                accm += tm;
            }
        }
        if constexpr (L > 1) add_terms<L>(S.n, accp, accm);
    }
    if (form == REGULAR) {
        // nodes next to E0: the difference quotient across it
        if constexpr (L > 1)
            for (int d = 1; d < L; d *= 2) wnear += __shfl_xor(wnear, d, L);
        if (wnear != 0.0) {
            const double del = fmax(1e-7 * (Emax - Emin), near);
            const double El = fmax(Emin, E0 - del), Er = fmin(Emax, E0 + del);
            double lp, lm, rp, rm;
            dist2(M, El, lp, lm);
            dist2(M, Er, rp, rm);
            const double pl = p_int(El, m), pr = p_int(Er, m), r = Er > El ? wnear / (Er - El) : 0.0;
            accp += r * (pr * rp - pl * lp);
            accm += r * (pr * rm - pl * lm);
        }
    }
    o.rp += accp * scale;
    o.rm += accm * scale;
    return o;
}

// ---- first-order anisotropy  OneLoopIntegralsAniso.jl ---------------------
// correction_cos_theta_coefficient (QuarkDistribution_Aniso.jl:14-86) of quark
// and antiquark at (p, E): xi p^2 / (2 E) df/dE
__device__ __forceinline__ void corr2(const Medium& M, double p, double E, double xi, double& cq, double& ca)
{
    double ep, em;
    boltzmann(M, E, ep, em);
    const double c = div_p(0.5 * xi * (p * p), E) * M.beta;
    auto slope = [&](double e, double c1, double c2) {
        const double e2 = e * e, e3 = e2 * e;
        const double num = c1 * e + 2 * c2 * e2 + e3;
        const double den = 1 + 3 * c1 * e + 3 * c2 * e2 + e3;
        const double dnum = -(c1 * e + 4 * c2 * e2 + 3 * e3);
        const double dden = -(3 * c1 * e + 6 * c2 * e2 + 3 * e3);
        const double t = dnum * den - num * dden, dd = den * den;
        return div_p(t, dd);
    };
    cq = c * slope(ep, M.Phi, M.Phib);
    ca = c * slope(em, M.Phib, M.Phi);
}

// find_roots_AB  :207-272 -> number of roots (ascending, unique)
__device__ int roots_AB(double lam, double k, double m, double mp, double Emin, double Emax, double r[2])
{
    const double C = lam * lam + m * m - mp * mp - k * k;
    const double a = k * k - lam * lam, b = -lam * C, c = -(k * k * m * m + C * C / 4);
    if (fabs(a) < 1e-14) {
        if (fabs(b) < 1e-14) return 0;
        double E = -c / b;
        if (E >= Emin && E <= Emax && E >= m) {
            double p = sqrt_p(fmax(0.0, E * E - m * m));
            double A = 2 * k * p, B = lam * lam + 2 * lam * E + m * m - mp * mp - k * k;
            if (fabs(A + B) < 1e-10 || fabs(A - B) < 1e-10) {
                r[0] = E;
                return 1;
            }
        }
        return 0;
    }
    const double D = b * b - 4 * a * c;
    if (D < 0) return 0;
    const double sD = sqrt_p(D);
    const double E12[2] = {(-b - sD) / (2 * a), (-b + sD) / (2 * a)};
    bool ok[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const double E = E12[i];
        const double p = sqrt_p(E * E - m * m);
        const double A = 2 * k * p, B = lam * lam + 2 * lam * E + m * m - mp * mp - k * k;
        ok[i] = E >= m && E >= Emin && E <= Emax && (fabs(A + B) < 1e-10 || fabs(A - B) < 1e-10);
    }
    if (ok[0] && ok[1]) {
        r[0] = fmin(E12[0], E12[1]);
        r[1] = fmax(E12[0], E12[1]);
        return r[0] == r[1] ? 1 : 2;
    }
    r[0] = pick(ok[0], E12[0], E12[1]);
    return (ok[0] || ok[1]) ? 1 : 0;
}

// tilde_B0_correction for the quark (plus) and antiquark (minus) coefficient:
// k = 0 :133-190, k > 0 :307-375
template <int L>
__device__ Pair tilde_Bc(const Phys& P, const Medium& M, double lam, double k, double m, double mp, double xi, int q)
{
    const double Emin = m, Emax = e_cut(P, m);
    const bool at_rest = !(k > kEpsK);
    Seg sg[5] = {};              // 3, 4: the imaginary part's
    Pair o{0.0, 0.0, 0.0, 0.0};
    double A0p = 0.0, A0m = 0.0;
    const double cE = 2.0 * lam, dc0 = lam * lam + m * m - mp * mp;
    // sqrt(p^2 + m^2): the node energy, but for a negative mass, whose momentum is clamped (p_int)
    auto energy = [&](double E, double p) { return m >= 0.0 ? E : sqrt_p(p * p + m * m); };
    if (at_rest) {
        const double E0 = -dc0 / cE;
        if (cE != 0.0 && isfinite(E0) && E0 >= Emin && E0 <= Emax) {
            const double p0 = p_int(E0, m);
            corr2(M, p0, energy(E0, p0), xi, A0p, A0m);
            A0p *= (4.0 / 3.0) * p0;
            A0m *= (4.0 / 3.0) * p0;
            const double lt = (log_c(fabs(cE * Emax + dc0)) - log_c(fabs(cE * Emin + dc0))) / cE;
            o.rp = A0p * lt;
            o.rm = A0m * lt;
            // imag_integrand_k_zero  :98-112
            const double c = kPi / cE;
            o.ip = c * A0p;
            o.im = c * A0m;
        }
        sg[0] = Seg{(Emax + Emin) / 2.0, (Emax - Emin) / 2.0, R_G32, 32};
    } else {
        double iv[2][2] = {}, r[2] = {};
        const int ni = sing_kpos(lam, k, m, mp, Emin, Emax, iv);
        const int nr = roots_AB(lam, k, m, mp, Emin, Emax, r);
        // build_intervals_from_roots  :275-292
        const double del = fmax(1e-10, 1e-8 * (Emax - Emin));
        const double b0 = nr >= 1 ? r[0] - del : Emax, a1 = r[0] + del, b1 = nr == 2 ? r[1] - del : Emax, a2 = r[1] + del;
        const bool v0 = b0 > Emin + 1e-16, v1 = nr >= 1 && b1 > a1 + 1e-16, v2 = nr == 2 && Emax > a2 + 1e-16;
        if (nr == 0) {
            if (v0) sg[2] = seg_power(Emin, Emax, R_L16, 16);
        } else {
            // the first of several intervals clusters to its right end, the last to its left, others to both
            const int nv = (v0 ? 1 : 0) + (v1 ? 1 : 0) + (v2 ? 1 : 0);
            if (v0) sg[0] = nv == 1 ? seg_mid(Emin, b0, R_DE, 33) : seg_power(Emin, b0, R_R32, 32);
            if (v1) sg[1] = (nv == 1 || (v0 && v2)) ? seg_mid(a1, b1, R_DE, 33)
                          : (v0 ? seg_power(a1, b1, R_L16, 16) : seg_power(a1, b1, R_R32, 32));
            if (v2) sg[2] = nv == 1 ? seg_mid(a2, Emax, R_DE, 33) : seg_power(a2, Emax, R_L16, 16);
        }
        if (ni > 0) sg[3] = Seg{(iv[0][0] + iv[0][1]) / 2, (iv[0][1] - iv[0][0]) / 2, R_G16, 16};
        if (ni > 1) sg[4] = Seg{(iv[1][0] + iv[1][1]) / 2, (iv[1][1] - iv[1][0]) / 2, R_G16, 16};
    }
    double sp = 0.0, sm = 0.0;
#pragma unroll 1
    for (int g = 0; g < 5; g++) {
        const Seg S = seg_pick(g == 0, sg[0], seg_pick(g == 1, sg[1], seg_pick(g == 2, sg[2], seg_pick(g == 3, sg[3], sg[4]))));
#pragma unroll 1
        for (int i = q; i < S.n; i += L) {
            const double E = S.x0 + S.s * ptab[S.off + i];
            const double w = S.s * ptab[S.off + S.n + i];
            const double p = p_int(E, m);
            double vp, vm, tp, tm;
            corr2(M, p, energy(E, p), xi, vp, vm);
            if (at_rest) {
                const double den = cE * E + dc0;
                vp = (4.0 / 3.0) * p * vp - A0p;
                vm = (4.0 / 3.0) * p * vm - A0m;
                // a zero denominator (lambda = 0, equal masses) stays infinite
                const double r = rcp1(den);
                const double up = den == 0.0 ? vp * __builtin_inf() : div_r(vp, den, r);
                const double um = den == 0.0 ? vm * __builtin_inf() : div_r(vm, den, r);
                tp = w * ((isfinite(den) && isfinite(vp)) ? up : 0.0);
                tm = w * ((isfinite(den) && isfinite(vm)) ? um : 0.0);
            } else {
                // compute_coefficients, real_integral_tool, imag_integral_tool  :26-61
                const double dc = lam * lam + 2 * lam * E + m * m - mp * mp - k * k;
                const double cx = 2 * p * k, ic = rcp1(cx), ic2 = ic * ic;
                const double t2 = div_r(dc * dc, cx * cx * cx, ic2 * ic);
                double tool = kPi * t2;
                if (g < 3) {
                    const double ratio = fabs(div_p(cx + dc, cx - dc));
                    const bool ok = ratio > 0.0 && isfinite(ratio);
                    tool = ok ? div_r(-2 * dc, cx * cx, ic2) + t2 * log_p(ok ? ratio : 1.0) : __builtin_nan("");
                }
                tool *= 2.0 * p;
                vp *= tool;
                vm *= tool;
                tp = isfinite(vp) ? w * vp : 0.0;
                tm = isfinite(vm) ? w * vm : 0.0;
            }
            if constexpr (L > 1) {
                term_rows<L>()[i] = double2{tp, tm};
            } else {
                sp += tp;
                sm += tm;
            }
        }
        if constexpr (L > 1) add_terms<L>(S.n, sp, sm);
        if (g == 2) {
            o.rp += sp;
            o.rm += sm;
            sp = sm = 0.0;
        }
    }
    const double s = jsign(lam);
    o.ip += sp * s;
    o.im += sm * s;
    return o;
}

// B0 (part 1), B0_correction (part 2) or both summed (part 3), symmetrised
// over +-k0 for num_s = 1:
//   B0  OneLoopIntegrals.jl:489-503: B~+(-l; m1, m2, mu1) - B~-(l; m1, m2, mu1)
//       + B~+(l; m2, m1, mu2) - B~-(-l; m2, m1, mu2)
//   B0_correction  OneLoopIntegralsAniso.jl:396-413: the same arguments with
//       the quark / antiquark coefficients, all four added
//   polarization_aniso  PolarizationAniso.jl:29-54: l = k0 + mu1 - mu2, averaged with l' = -k0 + mu1 - mu2
// With mu1 = mu2 the plus and minus terms pair up at equal (lambda, m): two
// evaluations for equal masses, four for the average, instead of four and
// eight.  A group of L x S lanes gives every evaluation L lanes and runs S of
// them at once; the evaluations are summed in their order in every lane.
template <int L = 1, int S = 1>
__device__ void b0_sum(const Phys& P, int part, double l0, double l1, double k, double m1, double m2, double mu1,
                       double mu2, double T, double Phi, double Phib, double xi, int nv, double& br, double& bi)
{
    const int gl = (int)(threadIdx.x & (L * S - 1)), q = gl & (L - 1);
    const bool eqmu = mu1 == mu2, two = eqmu && m1 == m2 && nv == 1;
    const bool four = !two && eqmu && nv == 2;
    const int ne = two ? 2 : (four ? 4 : 4 * nv);
    const double wgt = nv == 2 ? 0.5 : 1.0;
    double r = 0.0, i = 0.0;
#pragma unroll 1
    for (int e0 = 0; e0 < ne; e0 += S) {
        const int e = e0 + gl / L, t = e & 3;
        const bool swap = t >= 2, neg = t == 0 || t == 3;
        // the plus and the minus term's l; with four, l1 = -l0 to the last bits
        const double l = pick(e >= 4, l1, l0), lp = four && (t & 1) ? -l1 : l, lm = four && !(t & 1) ? -l1 : l;
        const bool both = two || four;
        const bool plus = both || !(t & 1), minus = both || (t & 1);
        double br0 = 0.0, bi0 = 0.0, br1 = 0.0, bi1 = 0.0;
        if (S == 1 || e < ne) {
            const Medium M = make_medium(swap ? mu2 : mu1, T, Phi, Phib);
            const double lam = neg ? -lp : lp, lam_m = neg ? -lm : lm, ma = swap ? m2 : m1, mb = swap ? m1 : m2;
            if (part & 1) {
                const Pair b = tilde_B0<L>(P, M, lam, both ? lam_m : lam, k, ma, mb, q);
                br0 = wgt * ((plus ? b.rp : 0.0) - (minus ? b.rm : 0.0));
                bi0 = wgt * ((plus ? b.ip : 0.0) - (minus ? b.im : 0.0));
            }
            if (part & 2) {
                const Pair b = tilde_Bc<L>(P, M, lam, k, ma, mb, xi, q);
                br1 = wgt * ((plus ? b.rp : 0.0) + (minus ? b.rm : 0.0));
                bi1 = wgt * ((plus ? b.ip : 0.0) + (minus ? b.im : 0.0));
            }
        }
#pragma unroll
        for (int j = 0; j < S; j++) {
            r += S > 1 ? __shfl(br0, j * L, L * S) : br0;
            i += S > 1 ? __shfl(bi0, j * L, L * S) : bi0;
            r += S > 1 ? __shfl(br1, j * L, L * S) : br1;
            i += S > 1 ? __shfl(bi1, j * L, L * S) : bi1;
        }
    }
    br = r;
    bi = i;
}

template <int L = 1, int S = 1>
__device__ void b0_total(const Phys& P, double k0, double k, double m1, double m2, double mu1, double mu2, double T,
                         double Phi, double Phib, double xi, int num_s, double& br, double& bi)
{
    b0_sum<L, S>(P, fabs(xi) > kEpsSeg ? 3 : 1, k0 + mu1 - mu2, -k0 + mu1 - mu2, k, m1, m2, mu1, mu2, T, Phi, Phib, xi, num_s == 1 ? 2 : 1, br,
                 bi);
}

// polarization_aniso / polarization_with_width  PolarizationAniso.jl:22-118
__device__ void pi_value(const Phys& P, int channel, int width, double k0, double gamma, double k, double m1,
                         double m2, double lam, double A12, double br, double bi, double& re, double& im)
{
    const double factor = -P.Nc / (8 * (kPi * kPi));
    double real = A12, imag = 0.0;
    double pref = k * k - lam * lam;
    pref += channel == PNJL_CHANNEL_P ? (m1 - m2) * (m1 - m2) : (m1 + m2) * (m1 + m2);
    if (width) {
        pref += (gamma * gamma) / 4.0;
        real += pref * br - gamma * lam * bi;
        imag += pref * bi + gamma * lam * br;
    } else {
        real += pref * br;
        imag += pref * bi;
    }
    re = factor * real;
    im = factor * imag;
}

// PNJL distributions  QuarkDistribution.jl:14-60
__device__ __forceinline__ double dist_ratio(double e, double c1, double c2)
{
    double e2 = e * e, e3 = e2 * e;
    return (c1 * e + 2 * c2 * e2 + e3) / (1 + 3 * c1 * e + 3 * c2 * e2 + e3);
}

__device__ __forceinline__ double quark_f(double E, double mu, double T, double Phi, double Phib)
{
    return dist_ratio(clamp_e(exp(-(E - mu) * (1 / T))), Phi, Phib);
}

__device__ __forceinline__ double antiquark_f(double E, double mu, double T, double Phi, double Phib)
{
    return dist_ratio(clamp_e(exp(-(E + mu) * (1 / T))), Phib, Phi);
}

// A / A_aniso  OneLoopIntegrals.jl:507-543, OneLoopIntegralsAniso.jl:446-467
__device__ double A_const(const Phys& P, double m)
{
    const double mp = m > 0 ? m : 0.0;
    const double L = P.Lambda;
    if (mp < 1e-14) return (L * L) / 2.0;
    const double s = sqrt(L * L + mp * mp);
    return (L * s - mp * mp * log((L + s) / mp)) / 2.0;
}

__device__ double A_value(const Phys& P, double m, double mu, double T, double Phi, double Phib, double xi, int np,
                          const double* xp, const double* wp, int nc, const double* xc, const double* wc)
{
    double integral = 0.0;
    if (nc <= 0) {
        integral = -A_const(P, m);
        for (int i = 0; i < np; i++) {
            double p = xp[i], E = sqrt(p * p + m * m);
            integral += wp[i] * (p * p) / E * (quark_f(E, mu, T, Phi, Phib) + antiquark_f(E, mu, T, Phi, Phib));
        }
        return 4.0 * integral;
    }
    for (int i = 0; i < np; i++) {
        double p = xp[i], aq = 0.0, aa = 0.0;
        double E = sqrt(p * p + m * m);
        for (int j = 0; j < nc; j++) {
            double pc = p * xc[j];
            double Ea = sqrt(p * p + m * m + xi * (pc * pc));
            aq += wc[j] * (p * p) / E * quark_f(Ea, mu, T, Phi, Phib);
            aa += wc[j] * (p * p) / E * antiquark_f(Ea, mu, T, Phi, Phib);
        }
        integral += wp[i] * (aq + aa);
    }
    return 2.0 * integral - 4.0 * A_const(P, m);
}

// ---- kernels -----------------------------------------------------------------
__device__ __forceinline__ void load_tabs(const double* tab)
{
    for (int i = threadIdx.x; i < kTabLen; i += blockDim.x) ptab[i] = tab[i];
    __syncthreads();
}

// query i = thread / (L S stride): L x S lanes per query (stride 1), or one
// query per wavefront on one lane (stride 64, for counting FLOPs)
template <int L, int S>
__global__ void __launch_bounds__(256, 3) query_kernel(Phys P, const double* tab, int64_t n, const pnjl_pol_query* qs,
                                                    double* re, double* im, int stride)
{
    load_tabs(tab);
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t % stride) return;
    const int64_t i = t / (L * S * stride);
    if (i >= n) return;
    const pnjl_pol_query a = qs[i];
    double r = __builtin_nan(""), m = __builtin_nan("");   // unsupported channel
    if (a.channel == PNJL_CHANNEL_P || a.channel == PNJL_CHANNEL_S) {
        double br, bi;
        b0_total<L, S>(P, a.k0, a.k, a.m1, a.m2, a.mu1, a.mu2, a.T, a.Phi, a.Phib, a.xi, a.num_s, br, bi);
        pi_value(P, a.channel, a.width, a.k0, a.gamma, a.k, a.m1, a.m2, a.k0 + a.mu1 - a.mu2, a.A1 + a.A2, br, bi, r,
                 m);
    }
    if (threadIdx.x % (L * S) == 0) {
        re[i] = r;
        im[i] = m;
    }
}

__global__ void __launch_bounds__(256, 3) b0_kernel(Phys P, const double* tab, int64_t n, const double* args, int corr,
                                                 double* re, double* im)
{
    load_tabs(tab);
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    // B0(lambda, k, m1, mu1, m2, mu2, T, Phi, Phib), B0_correction(lambda, k, m1, m2, mu1, mu2, T, Phi, Phib, xi)
    const double* a = args + i * (corr ? 10 : 9);
    b0_sum(P, corr ? 2 : 1, a[0], a[0], a[1], a[2], corr ? a[3] : a[4], corr ? a[4] : a[3], a[5], a[6], a[7], a[8],
           corr ? a[9] : 0.0, 1, re[i], im[i]);
}

__global__ void __launch_bounds__(256) a_kernel(Phys P, int64_t n, const double* args, int np, const double* xp,
                                                const double* wp, int nc, const double* xc, const double* wc,
                                                double* out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int w = nc > 0 ? 6 : 5;
    const double* a = args + i * w;
    out[i] = A_value(P, a[0], a[1], a[2], a[3], a[4], nc > 0 ? a[5] : 0.0, np, xp, wp, nc, xc, wc);
}

// grid: A_aniso(m_u), A_aniso(m_s) per point -> A[pt*2 + f]
__global__ void __launch_bounds__(256) grid_a_kernel(Phys P, int npts, const pnjl_pol_point* pts, int np,
                                                     const double* xp, const double* wp, int nc, const double* xc,
                                                     const double* wc, double* A)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * npts) return;
    const pnjl_pol_point s = pts[i >> 1];
    const double m = (i & 1) ? s.m_s : s.m_u;
    A[i] = A_value(P, m, s.mu, s.T, s.Phi, s.Phib, s.xi, np, xp, wp, nc, xc, wc);
}

// k extent of a wavefront's (k0, k) tile: 8 x 8 tiles keep the lanes of a
// wavefront closer in both momenta than a 1 x 64 row (measured on one 256 x
// 128 x 64 grid: 10.5 ms per call against 12.8 ms for 1 x 64 rows, 10.6 for
// 4 x 16, 10.8 for 16 x 4, 11.3 for 32 x 2).
#ifndef PNJL_GRID_TILE_K
#define PNJL_GRID_TILE_K 8
#endif
// grid: L x S lanes per (point, pair, k0, k); both channels written.
// The quadrature kernels are held to 3 waves per SIMD (168 VGPRs): latency
// hiding pays more than a few spills cost.
template <int L, int S>
__global__ void __launch_bounds__(256, 3) grid_pi_kernel(Phys P, const double* tab, int npts, const pnjl_pol_point* pts,
                                                      const double* A, int nk0, const double* k0s, int nk,
                                                      const double* ks, double* re, double* im)
{
    load_tabs(tab);
    const int64_t tid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / (L * S);
    const int64_t plane = (int64_t)nk0 * nk;
    if (tid >= (int64_t)npts * 3 * plane) return;
    int64_t j, i0;
    int pair, pt;
    constexpr int TK = PNJL_GRID_TILE_K, T0 = 64 / TK;
    if (L * S == 1 && TK < 64 && nk % TK == 0 && nk0 % T0 == 0) {
        // a wavefront takes a T0 (k0) x TK (k) tile of one (point, pair) plane
        const int64_t lane = tid & 63, tile = tid >> 6;
        const int64_t ntk = nk / TK, tiles = ntk * (nk0 / T0);
        const int64_t pp = tile / tiles, tl = tile - pp * tiles;
        j = (tl % ntk) * TK + lane % TK;
        i0 = (tl / ntk) * T0 + lane / TK;
        pair = (int)(pp % 3);
        pt = (int)(pp / 3);
    } else {
        j = tid % nk, i0 = (tid / nk) % nk0;
        pair = (int)((tid / plane) % 3);
        pt = (int)(tid / (3 * plane));
    }
    const pnjl_pol_point s = pts[pt];
    const double m1 = pair == 2 ? s.m_s : s.m_u, m2 = pair == 0 ? s.m_u : s.m_s;
    const double A12 = A[pt * 2 + (pair == 2 ? 1 : 0)] + A[pt * 2 + (pair == 0 ? 0 : 1)];
    const double k0 = k0s[i0], k = ks[j];
    double br, bi;
    b0_total<L, S>(P, k0, k, m1, m2, s.mu, s.mu, s.T, s.Phi, s.Phib, s.xi, pair, br, bi);
    if (threadIdx.x % (L * S)) return;
    const int64_t base = ((int64_t)pt * 3 + pair) * 2 * plane + i0 * nk + j;
    for (int c = 0; c < 2; c++) {
        double r, m;
        pi_value(P, c == 0 ? PNJL_CHANNEL_P : PNJL_CHANNEL_S, 0, k0, 0.0, k, m1, m2, k0, A12, br, bi, r, m);
        re[base + c * plane] = r;
        im[base + c * plane] = m;
    }
}

// ---- consumers of Pi ---------------------------------------------------------------
__device__ __forceinline__ void store_kc(double* o, const meson::KCoef& c)
{
    o[0] = c.K0p, o[1] = c.K0m, o[2] = c.K123p, o[3] = c.K123m, o[4] = c.K4567p, o[5] = c.K4567m;
    o[6] = c.K8p, o[7] = c.K8m, o[8] = c.K08p, o[9] = c.K08m, o[10] = c.detKp, o[11] = c.detKm;
}

__device__ __forceinline__ meson::KCoef load_kc(const double* o)
{
    return meson::KCoef{o[0], o[1], o[2], o[3], o[4], o[5], o[6], o[7], o[8], o[9], o[10], o[11]};
}

__device__ __forceinline__ void store_c(double* o, meson::C v) { o[0] = v.r, o[1] = v.i; }

// in[i*4] = (A_u, A_s, m_u, m_s), or in[i*2] = (G_u, G_s) -> G_f[i*2] (optional), kc[i*12]
__global__ void __launch_bounds__(256) couplings_kernel(int64_t n, const double* in, int from_gf, double G, double K,
                                                        int Nc, double* Gf, double* kc)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double Gu, Gs;
    if (from_gf) {
        Gu = in[i * 2], Gs = in[i * 2 + 1];
    } else {
        const double* a = in + i * 4;
        Gu = meson::G_from_A(a[0], a[2], Nc), Gs = meson::G_from_A(a[1], a[3], Nc);
    }
    if (Gf) Gf[i * 2] = Gu, Gf[i * 2 + 1] = Gs;
    store_kc(kc + i * 12, meson::couplings(G, K, Gu, Gs));
}

// kc[i*12], pi[i*12] (six slots) -> out[i*36] (layout of pnjl_meson_propagators_batch)
__global__ void __launch_bounds__(256) meson_kernel(int64_t n, const double* kc, const double* pi, double* out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    using meson::C;
    const meson::KCoef k = load_kc(kc + i * 12);
    C P[6];
    for (int s = 0; s < 6; s++) P[s] = C{pi[i * 12 + 2 * s], pi[i * 12 + 2 * s + 1]};
    double* o = out + i * 36;
    store_c(o + 0, meson::simple(k.K123p, P[0]));
    store_c(o + 2, meson::simple(k.K4567p, P[2]));
    store_c(o + 4, meson::simple(k.K123m, P[1]));
    store_c(o + 6, meson::simple(k.K4567m, P[3]));
    double J[2][2];   // currents a (u ubar) and b (s sbar)
    meson::current(0, 0, J[0][0], J[0][1]);
    meson::current(2, 2, J[1][0], J[1][1]);
    for (int ch = 0; ch < 2; ch++) {
        C M00, M08, M88;
        const double detK = ch == 0 ? k.detKp : k.detKm;
        if (ch == 0)
            meson::mixing(P[0], P[4], k.K0p, k.K8p, k.K08p, k.detKp, M00, M08, M88);
        else
            meson::mixing(P[1], P[5], k.K0m, k.K8m, k.K08m, k.detKm, M00, M08, M88);
        store_c(o + 8 + 6 * ch, M00);
        store_c(o + 10 + 6 * ch, M08);
        store_c(o + 12 + 6 * ch, M88);
        for (int c = 0; c < 4; c++) {
            const double* Ja = J[c >> 1];
            const double* Jb = J[c & 1];
            store_c(o + 20 + 8 * ch + 2 * c, meson::mixed(detK, M00, M08, M88, Ja[0], Ja[1], Jb[0], Jb[1]));
        }
    }
}

// the meson mask of a query, or MS_NONE for a process / channel / mask outside the table
__device__ __host__ __forceinline__ unsigned query_mesons(const pnjl_prop_query& q, const meson::ProcRow* tab)
{
    if (q.process < 0 || q.process >= PNJL_PROC_COUNT || q.channel < 0 || q.channel > 2) return meson::MS_NONE;
    if (q.mesons) return (q.mesons & ~0x3f) ? meson::MS_NONE : (unsigned)q.mesons;
    return tab[q.process].ch[q.channel];
}

// ---- work order of the propagator batch ----------------------------------------
// The (pair, query) items the queries' mesons need are bucketed by what sets
// the branch structure of B0 -- pair, m1, |lambda| = |k0 + mu1 - mu2| and k --
// and evaluated bucket by bucket, so that the lanes of a wavefront take the
// same singularity branches (a counting sort: count, scan, scatter).  Items
// of no need are not evaluated at all.  The order inside a bucket follows the
// atomics and varies from call to call; each item's arithmetic does not.
constexpr int kBM = 8, kBL = 16, kBK = 16;
constexpr int kPropBuckets = 3 * kBM * kBL * kBK;

__device__ __forceinline__ int bin_of(double x, double scale, int nb)
{
    const double v = x * scale;
    if (!(v > 0.0)) return 0;   // negative or NaN
    return v >= (double)(nb - 1) ? nb - 1 : (int)v;
}

__device__ __forceinline__ unsigned item_need(const pnjl_prop_query& a, int pair)
{
    const unsigned mes = query_mesons(a, meson::kProcs);
    return mes == meson::MS_NONE ? 0u : (meson::slots_for(mes) >> (2 * pair)) & 3u;
}

__device__ __forceinline__ int item_bucket(const pnjl_prop_query& a, int pair)
{
    const double m1 = pair == 2 ? a.m_s : a.m_u;
    const double mu1 = pair == 2 ? a.mu_s : a.mu_u, mu2 = pair == 0 ? a.mu_u : a.mu_s;
    const int bm = bin_of(m1, 4.0, kBM), bl = bin_of(fabs(a.k0 + mu1 - mu2), 4.0, kBL), bk = bin_of(a.k, 5.0, kBK);
    return ((pair * kBM + bm) * kBL + bl) * kBK + bk;
}

__global__ void __launch_bounds__(256) zero_u32(unsigned* p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// item t = pair * n + i: bucket counts; the Pi slots of items of no need are zeroed
__global__ void __launch_bounds__(256) prop_count_kernel(int64_t n, const pnjl_prop_query* qs, unsigned* counts,
                                                         double* pib)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 3 * n) return;
    const int pair = (int)(t / n);
    const int64_t i = t - pair * n;
    const pnjl_prop_query a = qs[i];
    if (item_need(a, pair)) {
        atomicAdd(&counts[item_bucket(a, pair)], 1u);
    } else {
        double* o = pib + i * 12 + 4 * pair;
        o[0] = o[1] = o[2] = o[3] = 0.0;
    }
}

// exclusive scan of the bucket counts (one block of 256); offs[kPropBuckets] = total
__global__ void __launch_bounds__(256) prop_scan_kernel(const unsigned* counts, unsigned* offs)
{
    constexpr int per = kPropBuckets / 256;
    static_assert(kPropBuckets % 256 == 0, "bucket count");
    __shared__ unsigned part[256];
    const int b0 = threadIdx.x * per;
    unsigned s = 0;
    for (int j = 0; j < per; j++) s += counts[b0 + j];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {   // Hillis-Steele inclusive scan
        const unsigned v = threadIdx.x >= d ? part[threadIdx.x - d] : 0u;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    unsigned run = part[threadIdx.x] - s;
    for (int j = 0; j < per; j++) {
        offs[b0 + j] = run;
        run += counts[b0 + j];
    }
    if (threadIdx.x == 255) offs[kPropBuckets] = part[255];
}

__global__ void __launch_bounds__(256) prop_scatter_kernel(int64_t n, const pnjl_prop_query* qs, const unsigned* offs,
                                                           unsigned* cursor, unsigned* items)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 3 * n) return;
    const int pair = (int)(t / n);
    const int64_t i = t - pair * n;
    const pnjl_prop_query a = qs[i];
    if (!item_need(a, pair)) return;
    const int b = item_bucket(a, pair);
    items[offs[b] + atomicAdd(&cursor[b], 1u)] = (unsigned)(i * 3 + pair);
}

// Pi of one worklist item (query i, pair): one B0 serves both channels of the
// pair.  pib[i*12 + 2*slot] as in pnjl_polarization_grid's order.  Threads
// past the worklist's length (offs[kPropBuckets]) exit; stride 64 puts one
// item per wavefront, for counting FLOPs.
template <int L, int S>
__global__ void __launch_bounds__(256, 3) prop_pi_kernel(Phys P, const double* tab, const pnjl_prop_query* qs,
                                                      const unsigned* items, const unsigned* offs, double* pib,
                                                      int stride)
{
    const int64_t per = (int64_t)L * S * stride;   // threads per item
    const int64_t total = (int64_t)offs[kPropBuckets];
    if ((int64_t)blockIdx.x * blockDim.x >= total * per) return;   // uniform per block
    load_tabs(tab);
    const int64_t ts = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (ts % stride) return;
    const int64_t t = ts / per;
    if (t >= total) return;
    const unsigned code = items[t];
    const int pair = (int)(code % 3u);
    const int64_t i = code / 3u;
    const pnjl_prop_query a = qs[i];
    const unsigned need = item_need(a, pair);
    double* o = pib + i * 12 + 4 * pair;
    const double m1 = pair == 2 ? a.m_s : a.m_u, m2 = pair == 0 ? a.m_u : a.m_s;
    const double mu1 = pair == 2 ? a.mu_s : a.mu_u, mu2 = pair == 0 ? a.mu_u : a.mu_s;
    const double A1 = pair == 2 ? a.A_s : a.A_u, A2 = pair == 0 ? a.A_u : a.A_s;
    double br, bi;
    b0_total<L, S>(P, a.k0, a.k, m1, m2, mu1, mu2, a.T, a.Phi, a.Phib, a.xi, pair, br, bi);
    if (threadIdx.x % (L * S)) return;
    for (int c = 0; c < 2; c++) {
        if (need & (1u << c))
            pi_value(P, c == 0 ? PNJL_CHANNEL_P : PNJL_CHANNEL_S, 0, a.k0, 0.0, a.k, m1, m2, a.k0 + mu1 - mu2, A1 + A2,
                     br, bi, o[2 * c], o[2 * c + 1]);
        else
            o[2 * c] = o[2 * c + 1] = 0.0;
    }
}

// (D_S, D_P) per query from its Pi slots; kc == nullptr: couplings from A
__global__ void __launch_bounds__(256) prop_compose_kernel(int64_t n, const pnjl_prop_query* qs, const double* kc,
                                                           double G, double K, int Nc, const double* pib,
                                                           double* out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    using meson::C;
    const pnjl_prop_query a = qs[i];
    const unsigned mes = query_mesons(a, meson::kProcs);
    double* o = out + i * 4;
    if (mes == meson::MS_NONE) {
        o[0] = o[1] = o[2] = o[3] = __builtin_nan("");
        return;
    }
    const meson::KCoef k = kc ? load_kc(kc + i * 12)
                              : meson::couplings(G, K, meson::G_from_A(a.A_u, a.m_u, Nc),
                                                 meson::G_from_A(a.A_s, a.m_s, Nc));
    C pi[6];
    for (int s = 0; s < 6; s++) pi[s] = C{pib[i * 12 + 2 * s], pib[i * 12 + 2 * s + 1]};
    C DS, DP;
    meson::by_channel(meson::kProcs[a.process], a.channel, mes, k, pi, DS, DP);
    store_c(o, DS);
    store_c(o + 2, DP);
}

// ---- meson pole masses (MesonMass.jl) -------------------------------------------------
constexpr double kFdStep = 6.055454452393343e-06;   // cbrt(eps): FiniteDiff's central relstep = absstep

// principal square root
__device__ __forceinline__ meson::C csqrt_p(meson::C z)
{
    if (z.r == 0.0 && z.i == 0.0) return meson::C{0.0, z.i};
    const double t = sqrt((fabs(z.r) + hypot(z.r, z.i)) * 0.5);
    if (z.r >= 0.0) return meson::C{t, z.i / (2.0 * t)};
    return meson::C{fabs(z.i) / (2.0 * t), copysign(t, z.i)};
}

// The residual at (k0, gamma) needs B0 of one quark pair (two for the mixed
// mesons) at k0 only: gamma enters polarization_with_width algebraically.
// B0 is therefore computed once per k0 and reused for the gamma column of
// the finite-difference Jacobian (the same values a recomputation gives).
struct MassB0 {
    double r[2], i[2];
};

__device__ __forceinline__ void mass_pair(const pnjl_mass_query& a, int pair, double& m1, double& m2, double& mu1,
                                          double& mu2, double& A12)
{
    m1 = pair == 2 ? a.m_s : a.m_u, m2 = pair == 0 ? a.m_u : a.m_s;
    mu1 = pair == 2 ? a.mu_s : a.mu_u, mu2 = pair == 0 ? a.mu_u : a.mu_s;
    A12 = (pair == 2 ? a.A_s : a.A_u) + (pair == 0 ? a.A_u : a.A_s);
}

// the pairs of a meson: pi, sigma_pi -> uu; K, sigma_K -> us; mixed -> uu, ss
__device__ __forceinline__ int mass_pairs(int m, int* pairs)
{
    if (m >= PNJL_MESON_ID_ETA) {
        pairs[0] = 0, pairs[1] = 2;
        return 2;
    }
    pairs[0] = (m == PNJL_MESON_ID_K || m == PNJL_MESON_ID_SIGMA_K) ? 1 : 0;
    return 1;
}

// B0 (symmetrised for u sbar, + correction) of the meson's pairs at k0
//   MesonMass.jl:34-60, :222-231 (MesonMass passes num_s 0 for s sbar, equivalent to 2)
template <int L>
__device__ __forceinline__ void mass_b0(const Phys& P, const pnjl_mass_query& a, double k0, MassB0& B)
{
    int pairs[2];
    const int np = mass_pairs(a.meson, pairs);
#pragma unroll 1
    for (int j = 0; j < np; j++) {
        double m1, m2, mu1, mu2, A12;
        mass_pair(a, pairs[j], m1, m2, mu1, mu2, A12);
        b0_total<L>(P, k0, a.k, m1, m2, mu1, mu2, a.T, a.Phi, a.Phib, a.xi, pairs[j] == 1 ? 1 : 0, B.r[j], B.i[j]);
    }
}

// meson_mass_equation  MesonMass.jl:211-233 from the B0 at k0: 1 - 4 K Pi, or
// for the mixed mesons the light / heavy eigenvalue of 2M,
// (M00 + M88) -/+ sqrt((M00 - M88)^2 + 4 M08^2)
__device__ void mass_residual(const Phys& P, const pnjl_mass_query& a, const meson::KCoef& k, const MassB0& B,
                              double k0, double gamma, double* f)
{
    using meson::C;
    const int m = a.meson;
    int pairs[2];
    const int np = mass_pairs(m, pairs);
    const bool pch = m == PNJL_MESON_ID_PI || m == PNJL_MESON_ID_K || m == PNJL_MESON_ID_ETA ||
                     m == PNJL_MESON_ID_ETA_PRIME;
    const int ch = pch ? PNJL_CHANNEL_P : PNJL_CHANNEL_S;
    C Pi[2];
    for (int j = 0; j < np; j++) {
        double m1, m2, mu1, mu2, A12;
        mass_pair(a, pairs[j], m1, m2, mu1, mu2, A12);
        pi_value(P, ch, 1, k0, gamma, a.k, m1, m2, k0 + mu1 - mu2, A12, B.r[j], B.i[j], Pi[j].r, Pi[j].i);
    }
    C res;
    if (m < PNJL_MESON_ID_ETA) {
        const double K = m == PNJL_MESON_ID_PI ? k.K123p
                       : m == PNJL_MESON_ID_K  ? k.K4567p
                       : m == PNJL_MESON_ID_SIGMA_PI ? k.K123m : k.K4567m;
        const double k4 = 4.0 * K;
        res = C{1.0 - k4 * Pi[0].r, -(k4 * Pi[0].i)};
    } else {
        C M00, M08, M88;
        if (pch)
            meson::mixing(Pi[0], Pi[1], k.K0p, k.K8p, k.K08p, k.detKp, M00, M08, M88);
        else
            meson::mixing(Pi[0], Pi[1], k.K0m, k.K8m, k.K08m, k.detKm, M00, M08, M88);
        const C dm = meson::csub(M00, M88);
        const C sq = csqrt_p(meson::cadd(meson::cmul(dm, dm), meson::rmul(4.0, meson::cmul(M08, M08))));
        const C tr = meson::cadd(M00, M88);
        res = (m == PNJL_MESON_ID_ETA || m == PNJL_MESON_ID_SIGMA) ? meson::csub(tr, sq) : meson::cadd(tr, sq);
    }
    f[0] = res.r;
    f[1] = res.i;
}

// step of the central finite differences (FiniteDiff) at x
__device__ __forceinline__ double fd_step(double x) { return fmax(kFdStep * fabs(x), kFdStep); }

__device__ __forceinline__ double wnorm2(const double* d, const double* v)
{
    return sqrt((d[0] * v[0]) * (d[0] * v[0]) + (d[1] * v[1]) * (d[1] * v[1]));
}

// NLsolve dogleg! for 2 x 2 (a singular Jacobian takes the scaled steepest-descent branch)
__device__ void dogleg2(double* p, const double* r, const double* d, const double J[2][2], double delta)
{
    const double det = J[0][0] * J[1][1] - J[0][1] * J[1][0];
    double pi_[2];
    if (det != 0.0 && isfinite(det)) {
        pi_[0] = -((J[1][1] * r[0] - J[0][1] * r[1]) / det);
        pi_[1] = -((-J[1][0] * r[0] + J[0][0] * r[1]) / det);
    } else {
        pi_[0] = pi_[1] = __builtin_inf();
    }
    if (wnorm2(d, pi_) <= delta) {
        p[0] = pi_[0], p[1] = pi_[1];
        return;
    }
    double g[2], Jg[2];
    for (int j = 0; j < 2; j++) g[j] = (J[0][j] * r[0] + J[1][j] * r[1]) / (d[j] * d[j]);
    for (int i = 0; i < 2; i++) Jg[i] = J[i][0] * g[0] + J[i][1] * g[1];
    const double wg = wnorm2(d, g);
    const double coef = -(wg * wg) / (Jg[0] * Jg[0] + Jg[1] * Jg[1]);
    const double pc[2] = {coef * g[0], coef * g[1]};
    if (wnorm2(d, pc) >= delta) {
        const double sc = -delta / wg;
        p[0] = g[0] * sc, p[1] = g[1] * sc;
        return;
    }
    const double pd[2] = {pi_[0] - pc[0], pi_[1] - pc[1]};
    const double b = 2.0 * ((d[0] * pc[0]) * (d[0] * pd[0]) + (d[1] * pc[1]) * (d[1] * pd[1]));
    const double wa = wnorm2(d, pd);
    const double aa = wa * wa;
    const double wpc = wnorm2(d, pc);
    const double tau = (-b + sqrt(b * b - 4.0 * aa * (wpc * wpc - delta * delta))) / (2.0 * aa);
    p[0] = pc[0] + tau * pd[0], p[1] = pc[1] + tau * pd[1];
}

// default_meson_mass_guess  MesonMass.jl:183-204 (d = u)
__device__ __forceinline__ double mass_guess(const pnjl_mass_query& a)
{
    switch (a.meson) {
        case PNJL_MESON_ID_PI: return a.m_u + a.m_u;
        case PNJL_MESON_ID_K:
        case PNJL_MESON_ID_SIGMA_K: return a.m_u + a.m_s;
        case PNJL_MESON_ID_ETA_PRIME:
        case PNJL_MESON_ID_SIGMA_PRIME: return 2.0 * a.m_s;
        default: return 2.0 * a.m_u;
    }
}

// Trust-region state of a pole search between the launches of
// pnjl_meson_mass_batch (every field it carries from one iteration to the next).
struct MassState {
    double x[2], r[2], J[2][2], d[2], delta;
    int it, conv, stopped, pad;
};

// solve_meson_mass  MesonMass.jl:241-276 with NLsolve's trust region (dogleg,
// autoscale, factor 1) and a central-difference Jacobian.
// out[i*6] = (mass, gamma, residual_norm (inf), converged, iterations, exception)
//
// The queries run in phases of growing iteration budgets (16, 16, 32, ...,
// then unlimited): phase 0 starts every query; a query that is not done when
// its phase's budget is spent saves its state and joins the list of the next
// phase.  The searches differ by orders of magnitude in length (most stop in
// a few dozen iterations, some run NLsolve's full 1000), so one launch would
// hold every wavefront for its longest query; the phases keep the long ones
// packed together.
//
// G lanes per query.  An iteration needs B0 at the trial k0 and at k0 +- h for
// the Jacobian's k0 column: with 16 or 64 lanes, four sub-groups evaluate the
// three at once (the fourth repeats the first), each splitting its nodes over
// G/4 lanes; one lane (for counting FLOPs, stride 64: one query per wavefront)
// takes them one after the other.  Every lane runs the same control logic on
// the same values, so a query's arithmetic does not depend on G.  The time is
// that of the longest searches (NLsolve's 1000 iterations), so the residual
// code is inlined into one trip loop: nothing of it goes through memory.
// 18 432 queries (48 x 48 points, 8 mesons): 65.6 -> 13.0 ms; 524 288: 168 ->
// 98 ms.  Giving sub-groups several evaluations at once instead of all their
// lanes to one (8 x 2, 4 x 4 of 16 lanes) took 14.7 and 24.3 ms.
// The residual f at x and the Jacobian J there by central finite differences
// (FiniteDiff): J[:, j] = (f(x + e_j h) - f(x - e_j h)) / 2h, from B0 at x[0]
// and x[0] +- h (the gamma column needs no new B0).  A group's sub-groups
// evaluate B0 at the three, then the lanes of each eight take one of the five
// residuals each (x, x[0] +- h, x[1] +- h; the rest repeat the first), and the
// group exchanges them.
template <int G>
__device__ __forceinline__ void mass_group(const Phys& P, const pnjl_mass_query& a, const meson::KCoef& k,
                                           const double* x, double* f, double J[2][2])
{
    constexpr int kSub = G == 1 ? 1 : G / 4;   // lanes per B0
    const double h0 = fd_step(x[0]), h1 = fd_step(x[1]);
    if constexpr (G == 1) {
        MassB0 Bx{}, Bp{}, Bm{};
        mass_b0<1>(P, a, x[0], Bx);
        mass_b0<1>(P, a, x[0] + h0, Bp);
        mass_b0<1>(P, a, x[0] - h0, Bm);
        double fp[2], fm[2], gp[2], gm[2];
        mass_residual(P, a, k, Bx, x[0], x[1], f);
        mass_residual(P, a, k, Bp, x[0] + h0, x[1], fp);
        mass_residual(P, a, k, Bm, x[0] - h0, x[1], fm);
        mass_residual(P, a, k, Bx, x[0], x[1] + h1, gp);
        mass_residual(P, a, k, Bx, x[0], x[1] - h1, gm);
        for (int i = 0; i < 2; i++) {
            J[i][0] = (fp[i] - fm[i]) / (2.0 * h0);
            J[i][1] = (gp[i] - gm[i]) / (2.0 * h1);
        }
    } else {
        const int gl = (int)(threadIdx.x % G), sub = gl / kSub, w = gl & 7;
        MassB0 B{};
        mass_b0<kSub>(P, a, sub == 1 ? x[0] + h0 : (sub == 2 ? x[0] - h0 : x[0]), B);
        const int from = w == 1 ? kSub : (w == 2 ? 2 * kSub : 0);
        for (int j = 0; j < 2; j++) {
            B.r[j] = __shfl(B.r[j], from, G);
            B.i[j] = __shfl(B.i[j], from, G);
        }
        double g[2];
        mass_residual(P, a, k, B, w == 1 ? x[0] + h0 : (w == 2 ? x[0] - h0 : x[0]),
                      w == 3 ? x[1] + h1 : (w == 4 ? x[1] - h1 : x[1]), g);
        for (int i = 0; i < 2; i++) {
            f[i] = __shfl(g[i], 0, G);
            J[i][0] = (__shfl(g[i], 1, G) - __shfl(g[i], 2, G)) / (2.0 * h0);
            J[i][1] = (__shfl(g[i], 3, G) - __shfl(g[i], 4, G)) / (2.0 * h1);
        }
    }
}

template <int G>
__global__ void __launch_bounds__(256, G == 1 ? 3 : 2) mass_kernel(Phys P, const double* tab, int64_t n,
                                                   const pnjl_mass_query* qs, const double* kc, double Gc, double K,
                                                   int Nc, double* out, int stride, MassState* states,
                                                   const int32_t* in_list, const unsigned* in_count,
                                                   int32_t* out_list, unsigned* out_count, int budget)
{
    const bool first = (in_list == nullptr);
    const int64_t count = first ? n : (int64_t)*in_count, per = (int64_t)G * stride;
    // blocks past the list leave before the table load (uniform per block)
    if ((int64_t)blockIdx.x * blockDim.x >= count * per) return;
    load_tabs(tab);
    const int64_t ts = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (ts % stride) return;
    const int64_t slot = ts / per;
    if (slot >= count) return;   // whole groups leave together
    const bool lead = G == 1 || threadIdx.x % G == 0;
    const int64_t i = first ? slot : (int64_t)in_list[slot];
    const pnjl_mass_query a = qs[i];
    double* o = out + i * 6;
    const meson::KCoef k = kc ? load_kc(kc + i * 12)
                              : meson::couplings(Gc, K, meson::G_from_A(a.A_u, a.m_u, Nc),
                                                 meson::G_from_A(a.A_s, a.m_s, Nc));
    double x[2], r[2], J[2][2], d[2], p[2], xold[2], delta;
    int it = 0;
    bool conv = false, stopped = false, fresh = first;
    if (first) {
        if (a.meson < 0 || a.meson >= PNJL_MESON_ID_COUNT || a.max_iter < 0) {
            if (lead)
                for (int j = 0; j < 6; j++) o[j] = __builtin_nan("");
            return;
        }
        x[0] = isnan(a.mass0) ? mass_guess(a) : a.mass0;
        x[1] = a.gamma0;
    } else {
        const MassState& S = states[i];
        x[0] = S.x[0], x[1] = S.x[1], r[0] = S.r[0], r[1] = S.r[1];
        J[0][0] = S.J[0][0], J[0][1] = S.J[0][1], J[1][0] = S.J[1][0], J[1][1] = S.J[1][1];
        d[0] = S.d[0], d[1] = S.d[1], delta = S.delta;
        it = S.it;
    }
    // one trip: the step to the trial point (none on a fresh search), the
    // residual and Jacobian there, and the trust region's decision
    for (int spent = 0;; spent++) {
        if (!fresh) {
            if (stopped || conv || it >= a.max_iter || (budget >= 0 && spent >= budget)) break;
            it++;
            dogleg2(p, r, d, J, delta);
            xold[0] = x[0], xold[1] = x[1];
            x[0] += p[0], x[1] += p[1];
        }
        double fn[2], Jn[2][2];
        mass_group<G>(P, a, k, x, fn, Jn);
        if (fresh) {
            fresh = false;
            spent--;
            r[0] = fn[0], r[1] = fn[1];
            if (!isfinite(r[0]) || !isfinite(r[1])) {   // NLsolve's IsFiniteException at the start
                if (lead) o[0] = x[0], o[1] = x[1], o[2] = __builtin_nan(""), o[3] = 0.0, o[4] = 0.0, o[5] = 1.0;
                return;
            }
            for (int q = 0; q < 2; q++) J[q][0] = Jn[q][0], J[q][1] = Jn[q][1];
            conv = fmax(fabs(r[0]), fabs(r[1])) < a.ftol;
            stopped = isnan(x[0]) || isnan(x[1]) || isnan(r[0]) || isnan(r[1]);
            d[0] = d[1] = delta = 0.0;
            if (!conv) {
                for (int j = 0; j < 2; j++) {
                    d[j] = sqrt(J[0][j] * J[0][j] + J[1][j] * J[1][j]);
                    if (d[j] == 0.0) d[j] = 1.0;
                }
                delta = 1.0 * wnorm2(d, x);
                if (delta == 0.0) delta = 1.0;
            }
            continue;
        }
        double rp[2];
        for (int q = 0; q < 2; q++) rp[q] = J[q][0] * p[0] + J[q][1] * p[1] + r[q];
        const double ssr = r[0] * r[0] + r[1] * r[1];
        const double rho = (ssr - (fn[0] * fn[0] + fn[1] * fn[1])) / (ssr - (rp[0] * rp[0] + rp[1] * rp[1]));
        if (rho > 1e-4) {
            r[0] = fn[0], r[1] = fn[1];
            for (int q = 0; q < 2; q++) J[q][0] = Jn[q][0], J[q][1] = Jn[q][1];
            for (int j = 0; j < 2; j++) d[j] = fmax(0.1 * d[j], sqrt(J[0][j] * J[0][j] + J[1][j] * J[1][j]));
            const bool xc = fmax(fabs(x[0] - xold[0]), fabs(x[1] - xold[1])) < a.xtol;
            conv = xc || fmax(fabs(r[0]), fabs(r[1])) < a.ftol;
        } else {
            x[0] -= p[0], x[1] -= p[1];
            conv = false;
        }
        if (rho < 0.1)
            delta = delta / 2.0;
        else if (rho >= 0.9)
            delta = 2.0 * wnorm2(d, p);
        else if (rho >= 0.5)
            delta = fmax(delta, 2.0 * wnorm2(d, p));
        stopped = isnan(x[0]) || isnan(x[1]) || isnan(fn[0]) || isnan(fn[1]);
    }
    if (!lead) return;
    if (!stopped && !conv && it < a.max_iter) {
        // budget spent: save the state for the next phase
        MassState& S = states[i];
        S.x[0] = x[0], S.x[1] = x[1], S.r[0] = r[0], S.r[1] = r[1];
        S.J[0][0] = J[0][0], S.J[0][1] = J[0][1], S.J[1][0] = J[1][0], S.J[1][1] = J[1][1];
        S.d[0] = d[0], S.d[1] = d[1], S.delta = delta;
        S.it = it, S.conv = 0, S.stopped = 0;
        out_list[atomicAdd(out_count, 1u)] = (int32_t)i;
        return;
    }
    o[0] = x[0], o[1] = x[1], o[2] = fmax(fabs(r[0]), fabs(r[1])), o[3] = conv ? 1.0 : 0.0, o[4] = (double)it;
    o[5] = 0.0;
}

}  // namespace polar

// =============================================================================
// host side
// =============================================================================
struct PolarGraph {
    int npts = 0, nk0 = 0, nk = 0, np = 0, nc = 0;
    hipStream_t cap = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    pnjl_pol_point* pts = nullptr;
    double *k0 = nullptr, *k = nullptr, *A = nullptr, *re = nullptr, *im = nullptr, *nodes = nullptr;
};

namespace pnjl_host {

void polar_release(pnjl_ctx* c)
{
    if (c->pgraph) {
        PolarGraph* g = c->pgraph;
        if (g->exec) (void)hipGraphExecDestroy(g->exec);
        if (g->graph) (void)hipGraphDestroy(g->graph);
        for (void* p : {(void*)g->pts, (void*)g->k0, (void*)g->k, (void*)g->A, (void*)g->re, (void*)g->im,
                        (void*)g->nodes})
            if (p) (void)hipFree(p);
        if (g->cap) (void)hipStreamDestroy(g->cap);
        delete g;
        c->pgraph = nullptr;
    }
    if (c->polar_tab) (void)hipFree(c->polar_tab);
    c->polar_tab = nullptr;
}

}  // namespace pnjl_host

namespace {

polar::Phys phys(const pnjl_ctx* c) { return polar::Phys{c->params.Lambda, (double)c->params.N_color}; }

// the quadrature kernels' tables (layout: polar::ptab)
//   rules: IntervalQuadratureStrategies.jl:56-85
int polar_tab(pnjl_ctx* ctx, double** out)
{
    if (!ctx->polar_tab) {
        std::vector<double> t(polar::kTabLen), x16, w16, x32, w32;
        for (int j = 0; j < 64; j++) t[pnjl::kExpTab + j] = (double)exp2l((long double)j / 64.0L);
        for (int j = 0; j < 128; j++) {
            // the first and last intervals take c = 1 and c = 2: log(1) = 0 there
            const long double c = j == 0 ? 1.0L : (j == 127 ? 2.0L : 1.0L + ((long double)j + 0.5L) / 128.0L);
            const double inv = (double)(1.0L / c);
            t[polar::kPLog + 2 * j] = inv;
            t[polar::kPLog + 2 * j + 1] = (double)(-logl((j >= 64 ? 2.0L : 1.0L) * (long double)inv));
        }
        gl_rule(16, x16, w16);
        gl_rule(32, x32, w32);
        const double ia = 1.0 / polar::kAlpha;
        auto put = [&](int off, int i, int n, double node, double weight) {
            t[off + i] = node;
            t[off + n + i] = weight;
        };
        for (int i = 0; i < 16; i++) {
            const double u = (x16[i] + 1) / 2;
            put(polar::R_L16, i, 16, pow(u, ia), w16[i] * (ia * pow(u, ia - 1) / 2));
            put(polar::R_G16, i, 16, x16[i], w16[i]);
        }
        for (int i = 0; i < 32; i++) {
            const double u = (x32[i] + 1) / 2;
            put(polar::R_L32, i, 32, pow(u, ia), w32[i] * (ia * pow(u, ia - 1) / 2));
            put(polar::R_R32, i, 32, 1 - pow(1 - u, ia), w32[i] * (ia * pow(1 - u, ia - 1) / 2));
            put(polar::R_G32, i, 32, x32[i], w32[i]);
        }
        for (int k = -16; k <= 16; k++) {
            double tk = k * polar::kDeH;
            double s = polar::kPi / 2 * sinh(tk);
            double sech = 1.0 / cosh(s);
            put(polar::R_DE, k + 16, 33, tanh(s), polar::kDeH * (polar::kPi / 2) * cosh(tk) * (sech * sech));
        }
        HIPCHK(ctx, hipMalloc(&ctx->polar_tab, t.size() * sizeof(double)));
        HIPCHK(ctx, hipMemcpy(ctx->polar_tab, t.data(), t.size() * sizeof(double), hipMemcpyHostToDevice));
    }
    *out = ctx->polar_tab;
    return PNJL_OK;
}

// Lanes per item of the quadrature kernels (an item is a Pi query, a grid cell
// or a propagator query's quark pair, about two per query): one lane walks
// the ~60 to 320 nodes of an item alone, which is the cheapest use of the
// chip but leaves it idle below its ~2 x 10^5 resident lanes, so smaller calls
// split each item over more lanes.  Measured, ms at 1 / 4 / 16 / 64 lanes: Pi
// queries 1000: 0.62 / 0.36 / 0.19 / 0.16, 10 000: 0.74 / 0.35 / 0.26 / 0.32,
// 60 000: 0.98 / 0.93 / 0.93, 200 000: 2.90 / 2.90 / 3.07; grid cells 81 000:
// 0.72 / 0.56 / 0.63 / 1.20, 307 200: 1.17 / 1.25 / 1.70; propagator queries
// 1000: 0.48 / 0.22 / 0.11 / 0.09, 5000: 0.48 / 0.22 / 0.13 / 0.18, 65 536:
// 0.55 / 0.43 / 0.70, 131 072: 0.71 / 0.71 / 1.30.
int item_lanes(int64_t items) { return items <= 4096 ? 64 : (items <= 32768 ? 16 : (items <= 196608 ? 4 : 1)); }

// f(L, S) with the kernels' compile-time split of `lanes`: L lanes per evaluation, S evaluations at once
template <class F>
void launch_lanes(int lanes, const F& f)
{
    using std::integral_constant;
    switch (lanes) {
    case 64: f(integral_constant<int, 16>(), integral_constant<int, 4>()); break;
    case 16: f(integral_constant<int, 4>(), integral_constant<int, 4>()); break;
    case 4: f(integral_constant<int, 4>(), integral_constant<int, 1>()); break;
    default: f(integral_constant<int, 1>(), integral_constant<int, 1>()); break;
    }
}

int blocks_for(int64_t n) { return (int)((n + 255) / 256); }

}  // namespace

extern "C" {

int pnjl_polarization_batch(pnjl_ctx* ctx, int64_t n, const pnjl_pol_query* q, double* re, double* im, int flags,
                            void* stream)
{
    if (!ctx) return PNJL_ERR_ARG;
    if (n < 0 || (n > 0 && (!q || !re || !im)))
        return set_err(ctx, PNJL_ERR_ARG, "pnjl_polarization_batch: bad argument");
    if (n == 0) return PNJL_OK;
    HIPCHK(ctx, hipSetDevice(ctx->device));
    hipStream_t st = (hipStream_t)stream;
    const bool dev = flags & PNJL_FLAG_DEVICE_PTRS;
    if (!dev)
        for (int64_t i = 0; i < n; i++)
            if (q[i].channel != PNJL_CHANNEL_P && q[i].channel != PNJL_CHANNEL_S)
                return set_err(ctx, PNJL_ERR_ARG, "pnjl_polarization_batch: unsupported channel (use P or S)");
    double* tab = nullptr;
    if (int rc = polar_tab(ctx, &tab)) return rc;
    const pnjl_pol_query* dq = q;
    double *dre = re, *dim = im;
    if (!dev) {
        void *a, *b, *c;
        if (int rc = stage_buf(ctx, 60, (size_t)n * sizeof(pnjl_pol_query), &a)) return rc;
        if (int rc = stage_buf(ctx, 61, (size_t)n * sizeof(double), &b)) return rc;
        if (int rc = stage_buf(ctx, 62, (size_t)n * sizeof(double), &c)) return rc;
        HIPCHK(ctx, hipMemcpyAsync(a, q, (size_t)n * sizeof(pnjl_pol_query), hipMemcpyHostToDevice, st));
        dq = (const pnjl_pol_query*)a;
        dre = (double*)b;
        dim = (double*)c;
    }
    HIPCHK(ctx, hipEventRecord(ctx->ev0, st));
    const int stride = (flags & PNJL_FLAG_ONE_PER_WAVE) ? 64 : 1;
    const int lanes = stride > 1 ? 1 : item_lanes(n);
    launch_lanes(lanes, [&](auto L, auto S) {
        hipLaunchKernelGGL((polar::query_kernel<L(), S()>), dim3(blocks_for(n * stride * lanes)), dim3(256), 0, st,
                           phys(ctx), tab, n, dq, dre, dim, stride);
    });
    HIPCHK(ctx, hipGetLastError());
    HIPCHK(ctx, hipEventRecord(ctx->ev1, st));
    if (!dev) {
        HIPCHK(ctx, hipMemcpyAsync(re, dre, (size_t)n * sizeof(double), hipMemcpyDeviceToHost, st));
        HIPCHK(ctx, hipMemcpyAsync(im, dim, (size_t)n * sizeof(double), hipMemcpyDeviceToHost, st));
    }
    if (!(flags & PNJL_FLAG_ASYNC) || !dev) {
        HIPCHK(ctx, hipStreamSynchronize(st));
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess) ctx->last_ms = ms;
    }
    return PNJL_OK;
}

static int b0_common(pnjl_ctx* ctx, int64_t n, const double* args, int corr, double* re, double* im)
{
    if (!ctx) return PNJL_ERR_ARG;
    if (n < 0 || (n > 0 && (!args || !re || !im))) return set_err(ctx, PNJL_ERR_ARG, "B0 batch: bad argument");
    if (n == 0) return PNJL_OK;
    HIPCHK(ctx, hipSetDevice(ctx->device));
    double* tab = nullptr;
    if (int rc = polar_tab(ctx, &tab)) return rc;
    const int w = corr ? 10 : 9;
    void *a, *b, *c;
    if (int rc = stage_buf(ctx, 60, (size_t)n * w * sizeof(double), &a)) return rc;
    if (int rc = stage_buf(ctx, 61, (size_t)n * sizeof(double), &b)) return rc;
    if (int rc = stage_buf(ctx, 62, (size_t)n * sizeof(double), &c)) return rc;
    HIPCHK(ctx, hipMemcpy(a, args, (size_t)n * w * sizeof(double), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(polar::b0_kernel, dim3(blocks_for(n)), dim3(256), 0, 0, phys(ctx), tab, n, (const double*)a,
                       corr, (double*)b, (double*)c);
    HIPCHK(ctx, hipGetLastError());
    HIPCHK(ctx, hipMemcpy(re, b, (size_t)n * sizeof(double), hipMemcpyDeviceToHost));
    HIPCHK(ctx, hipMemcpy(im, c, (size_t)n * sizeof(double), hipMemcpyDeviceToHost));
    return PNJL_OK;
}

int pnjl_B0_batch(pnjl_ctx* ctx, int64_t n, const double* args, double* re, double* im)
{
    return b0_common(ctx, n, args, 0, re, im);
}

int pnjl_B0_correction_batch(pnjl_ctx* ctx, int64_t n, const double* args, double* re, double* im)
{
    return b0_common(ctx, n, args, 1, re, im);
}

int pnjl_A_batch(pnjl_ctx* ctx, int64_t n, const double* args, int np, const double* nodes_p, const double* weights_p,
                 int nc, const double* nodes_cos, const double* weights_cos, double* out)
{
    if (!ctx) return PNJL_ERR_ARG;
    if (n < 0 || np <= 0 || np > 65536 || nc < 0 || nc > 4096 || (n > 0 && (!args || !out)) || !nodes_p ||
        !weights_p || (nc > 0 && (!nodes_cos || !weights_cos)))
        return set_err(ctx, PNJL_ERR_ARG, "pnjl_A_batch: bad argument");
    if (n == 0) return PNJL_OK;
    HIPCHK(ctx, hipSetDevice(ctx->device));
    const int w = nc > 0 ? 6 : 5;
    void *a, *nd, *o;
    if (int rc = stage_buf(ctx, 60, (size_t)n * w * sizeof(double), &a)) return rc;
    if (int rc = stage_buf(ctx, 61, (size_t)(2 * np + 2 * nc) * sizeof(double), &nd)) return rc;
    if (int rc = stage_buf(ctx, 62, (size_t)n * sizeof(double), &o)) return rc;
    double* d = (double*)nd;
    HIPCHK(ctx, hipMemcpy(a, args, (size_t)n * w * sizeof(double), hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d, nodes_p, np * sizeof(double), hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(d + np, weights_p, np * sizeof(double), hipMemcpyHostToDevice));
    if (nc > 0) {
        HIPCHK(ctx, hipMemcpy(d + 2 * np, nodes_cos, nc * sizeof(double), hipMemcpyHostToDevice));
        HIPCHK(ctx, hipMemcpy(d + 2 * np + nc, weights_cos, nc * sizeof(double), hipMemcpyHostToDevice));
    }
    hipLaunchKernelGGL(polar::a_kernel, dim3(blocks_for(n)), dim3(256), 0, 0, phys(ctx), n, (const double*)a, np, d,
                       d + np, nc, d + 2 * np, d + 2 * np + nc, (double*)o);
    HIPCHK(ctx, hipGetLastError());
    HIPCHK(ctx, hipMemcpy(out, o, (size_t)n * sizeof(double), hipMemcpyDeviceToHost));
    return PNJL_OK;
}

int pnjl_polarization_grid(pnjl_ctx* ctx, int npts, const pnjl_pol_point* pts, int nk0, const double* k0, int nk,
                           const double* k, int np, int nc, double* re, double* im, int flags, void* stream)
{
    if (!ctx) return PNJL_ERR_ARG;
    if (npts <= 0 || nk0 <= 0 || nk <= 0 || np <= 0 || np > 4096 || nc <= 0 || nc > 64 || !pts || !k0 || !k ||
        !re || !im)
        return set_err(ctx, PNJL_ERR_ARG, "pnjl_polarization_grid: bad argument");
    const int64_t nout = (int64_t)npts * 6 * nk0 * nk;
    if (nout > ((int64_t)1 << 31)) return set_err(ctx, PNJL_ERR_ARG, "pnjl_polarization_grid: grid too large");
    HIPCHK(ctx, hipSetDevice(ctx->device));
    double* tab = nullptr;
    if (int rc = polar_tab(ctx, &tab)) return rc;
    PolarGraph* g = ctx->pgraph;
    if (g && (g->npts != npts || g->nk0 != nk0 || g->nk != nk || g->np != np || g->nc != nc)) {
        polar_release(ctx);   // a new shape: rebuild the graph (tables are rebuilt too)
        if (int rc = polar_tab(ctx, &tab)) return rc;
        g = nullptr;
    }
    if (!g) {
        g = new PolarGraph();
        ctx->pgraph = g;
        g->npts = npts;
        g->nk0 = nk0;
        g->nk = nk;
        g->np = np;
        g->nc = nc;
        HIPCHK(ctx, hipStreamCreate(&g->cap));
        HIPCHK(ctx, hipMalloc(&g->pts, (size_t)npts * sizeof(pnjl_pol_point)));
        HIPCHK(ctx, hipMalloc(&g->k0, (size_t)nk0 * sizeof(double)));
        HIPCHK(ctx, hipMalloc(&g->k, (size_t)nk * sizeof(double)));
        HIPCHK(ctx, hipMalloc(&g->A, (size_t)npts * 2 * sizeof(double)));
        HIPCHK(ctx, hipMalloc(&g->re, (size_t)nout * sizeof(double)));
        HIPCHK(ctx, hipMalloc(&g->im, (size_t)nout * sizeof(double)));
        // momentum nodes GL on [0, 10] fm^-1, cos nodes GL on [-1, 1]
        std::vector<double> xp, wp, xc, wc;
        gl_rule(np, xp, wp);
        for (int i = 0; i < np; i++) {
            xp[i] = 5.0 * xp[i] + 5.0;
            wp[i] = 5.0 * wp[i];
        }
        gl_rule(nc, xc, wc);
        std::vector<double> nodes;
        nodes.insert(nodes.end(), xp.begin(), xp.end());
        nodes.insert(nodes.end(), wp.begin(), wp.end());
        nodes.insert(nodes.end(), xc.begin(), xc.end());
        nodes.insert(nodes.end(), wc.begin(), wc.end());
        HIPCHK(ctx, hipMalloc(&g->nodes, nodes.size() * sizeof(double)));
        HIPCHK(ctx, hipMemcpy(g->nodes, nodes.data(), nodes.size() * sizeof(double), hipMemcpyHostToDevice));
        // capture the A and Pi kernels once; later calls replay the graph
        HIPCHK(ctx, hipStreamBeginCapture(g->cap, hipStreamCaptureModeThreadLocal));
        hipLaunchKernelGGL(polar::grid_a_kernel, dim3(blocks_for(2 * (int64_t)npts)), dim3(256), 0, g->cap,
                           phys(ctx), npts, (const pnjl_pol_point*)g->pts, np, g->nodes, g->nodes + np, nc,
                           g->nodes + 2 * np, g->nodes + 2 * np + nc, g->A);
        const int lanes = item_lanes(nout / 2);
        launch_lanes(lanes, [&](auto L, auto S) {
            hipLaunchKernelGGL((polar::grid_pi_kernel<L(), S()>), dim3(blocks_for(nout / 2 * lanes)), dim3(256), 0,
                               g->cap, phys(ctx), tab, npts, (const pnjl_pol_point*)g->pts, (const double*)g->A, nk0,
                               (const double*)g->k0, nk, (const double*)g->k, g->re, g->im);
        });
        HIPCHK(ctx, hipStreamEndCapture(g->cap, &g->graph));
        HIPCHK(ctx, hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0));
    }
    hipStream_t st = stream ? (hipStream_t)stream : g->cap;
    const bool dev = flags & PNJL_FLAG_DEVICE_PTRS;
    const hipMemcpyKind in = dev ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    const hipMemcpyKind outk = dev ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost;
    HIPCHK(ctx, hipMemcpyAsync(g->pts, pts, (size_t)npts * sizeof(pnjl_pol_point), in, st));
    HIPCHK(ctx, hipMemcpyAsync(g->k0, k0, (size_t)nk0 * sizeof(double), in, st));
    HIPCHK(ctx, hipMemcpyAsync(g->k, k, (size_t)nk * sizeof(double), in, st));
    HIPCHK(ctx, hipEventRecord(ctx->ev0, st));
    HIPCHK(ctx, hipGraphLaunch(g->exec, st));
    HIPCHK(ctx, hipEventRecord(ctx->ev1, st));
    HIPCHK(ctx, hipMemcpyAsync(re, g->re, (size_t)nout * sizeof(double), outk, st));
    HIPCHK(ctx, hipMemcpyAsync(im, g->im, (size_t)nout * sizeof(double), outk, st));
    if (!(flags & PNJL_FLAG_ASYNC) || !dev) {
        HIPCHK(ctx, hipStreamSynchronize(st));
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess) ctx->last_ms = ms;
    }
    return PNJL_OK;
}

int pnjl_effective_couplings_batch(pnjl_ctx* ctx, int64_t n, const double* in, int from_gf, double G, double K,
                                   double* G_f, double* kc)
{
    if (!ctx) return PNJL_ERR_ARG;
    if (n < 0 || (n > 0 && (!in || !kc)))
        return set_err(ctx, PNJL_ERR_ARG, "pnjl_effective_couplings_batch: bad argument");
    if (n == 0) return PNJL_OK;
    HIPCHK(ctx, hipSetDevice(ctx->device));
    const int w = from_gf ? 2 : 4;
    void *a, *g, *o;
    if (int rc = stage_buf(ctx, 80, (size_t)n * w * sizeof(double), &a)) return rc;
    if (int rc = stage_buf(ctx, 81, (size_t)n * 2 * sizeof(double), &g)) return rc;
    if (int rc = stage_buf(ctx, 82, (size_t)n * PNJL_KCOEF_FIELDS * sizeof(double), &o)) return rc;
    HIPCHK(ctx, hipMemcpy(a, in, (size_t)n * w * sizeof(double), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(polar::couplings_kernel, dim3(blocks_for(n)), dim3(256), 0, 0, n, (const double*)a,
                       from_gf ? 1 : 0, G, K, ctx->params.N_color, (double*)g, (double*)o);
    HIPCHK(ctx, hipGetLastError());
    if (G_f) HIPCHK(ctx, hipMemcpy(G_f, g, (size_t)n * 2 * sizeof(double), hipMemcpyDeviceToHost));
    HIPCHK(ctx, hipMemcpy(kc, o, (size_t)n * PNJL_KCOEF_FIELDS * sizeof(double), hipMemcpyDeviceToHost));
    return PNJL_OK;
}

int pnjl_meson_propagators_batch(pnjl_ctx* ctx, int64_t n, const double* kc, const double* pi, double* out)
{
    if (!ctx) return PNJL_ERR_ARG;
    if (n < 0 || (n > 0 && (!kc || !pi || !out)))
        return set_err(ctx, PNJL_ERR_ARG, "pnjl_meson_propagators_batch: bad argument");
    if (n == 0) return PNJL_OK;
    HIPCHK(ctx, hipSetDevice(ctx->device));
    void *k, *p, *o;
    if (int rc = stage_buf(ctx, 80, (size_t)n * PNJL_KCOEF_FIELDS * sizeof(double), &k)) return rc;
    if (int rc = stage_buf(ctx, 81, (size_t)n * 12 * sizeof(double), &p)) return rc;
    if (int rc = stage_buf(ctx, 82, (size_t)n * PNJL_MESON_PROP_FIELDS * sizeof(double), &o)) return rc;
    HIPCHK(ctx, hipMemcpy(k, kc, (size_t)n * PNJL_KCOEF_FIELDS * sizeof(double), hipMemcpyHostToDevice));
    HIPCHK(ctx, hipMemcpy(p, pi, (size_t)n * 12 * sizeof(double), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(polar::meson_kernel, dim3(blocks_for(n)), dim3(256), 0, 0, n, (const double*)k,
                       (const double*)p, (double*)o);
    HIPCHK(ctx, hipGetLastError());
    HIPCHK(ctx, hipMemcpy(out, o, (size_t)n * PNJL_MESON_PROP_FIELDS * sizeof(double), hipMemcpyDeviceToHost));
    return PNJL_OK;
}

int pnjl_propagator_by_channel_batch(pnjl_ctx* ctx, int64_t n, const pnjl_prop_query* q, const double* kc,
                                     double* out, int flags, void* stream)
{
    if (!ctx) return PNJL_ERR_ARG;
    if (n < 0 || (n > 0 && (!q || !out)))
        return set_err(ctx, PNJL_ERR_ARG, "pnjl_propagator_by_channel_batch: bad argument");
    if (n == 0) return PNJL_OK;
    if (n > ((int64_t)1 << 29) || ((flags & PNJL_FLAG_ONE_PER_WAVE) && n > ((int64_t)1 << 23)))
        return set_err(ctx, PNJL_ERR_ARG, "pnjl_propagator_by_channel_batch: n too large");
    HIPCHK(ctx, hipSetDevice(ctx->device));
    hipStream_t st = (hipStream_t)stream;
    const bool dev = flags & PNJL_FLAG_DEVICE_PTRS;
    if (!dev)
        for (int64_t i = 0; i < n; i++)
            if (polar::query_mesons(q[i], meson::kProcsHost) == meson::MS_NONE)
                return set_err(ctx, PNJL_ERR_ARG,
                               "pnjl_propagator_by_channel_batch: process, channel or meson mask not in the table");
    double* tab = nullptr;
    if (int rc = polar_tab(ctx, &tab)) return rc;
    void *pib, *ints, *items;
    if (int rc = stage_buf(ctx, 83, (size_t)n * 12 * sizeof(double), &pib)) return rc;
    const int nb = polar::kPropBuckets;
    if (int rc = stage_buf(ctx, 84, (size_t)(3 * nb + 1) * sizeof(unsigned), &ints)) return rc;
    if (int rc = stage_buf(ctx, 85, (size_t)3 * n * sizeof(unsigned), &items)) return rc;
    unsigned* counts = (unsigned*)ints;   // counts[nb] | cursor[nb] | offs[nb + 1]
    unsigned* cursor = counts + nb;
    unsigned* offs = cursor + nb;
    const pnjl_prop_query* dq = q;
    const double* dkc = kc;
    double* dout = out;
    if (!dev) {
        void *a, *b, *c = nullptr;
        if (int rc = stage_buf(ctx, 80, (size_t)n * sizeof(pnjl_prop_query), &a)) return rc;
        if (int rc = stage_buf(ctx, 81, (size_t)n * 4 * sizeof(double), &b)) return rc;
        if (kc)
            if (int rc = stage_buf(ctx, 82, (size_t)n * PNJL_KCOEF_FIELDS * sizeof(double), &c)) return rc;
        HIPCHK(ctx, hipMemcpyAsync(a, q, (size_t)n * sizeof(pnjl_prop_query), hipMemcpyHostToDevice, st));
        if (kc)
            HIPCHK(ctx, hipMemcpyAsync(c, kc, (size_t)n * PNJL_KCOEF_FIELDS * sizeof(double), hipMemcpyHostToDevice,
                                       st));
        dq = (const pnjl_prop_query*)a;
        dkc = (const double*)c;
        dout = (double*)b;
    }
    HIPCHK(ctx, hipEventRecord(ctx->ev0, st));
    const int stride = (flags & PNJL_FLAG_ONE_PER_WAVE) ? 64 : 1;
    hipLaunchKernelGGL(polar::zero_u32, dim3(blocks_for(2 * nb)), dim3(256), 0, st, counts, 2 * nb);
    hipLaunchKernelGGL(polar::prop_count_kernel, dim3(blocks_for(3 * n)), dim3(256), 0, st, n, dq, counts,
                       (double*)pib);
    hipLaunchKernelGGL(polar::prop_scan_kernel, dim3(1), dim3(256), 0, st, (const unsigned*)counts, offs);
    hipLaunchKernelGGL(polar::prop_scatter_kernel, dim3(blocks_for(3 * n)), dim3(256), 0, st, n, dq,
                       (const unsigned*)offs, cursor, (unsigned*)items);
    const int lanes = stride > 1 ? 1 : item_lanes(2 * n);
    launch_lanes(lanes, [&](auto L, auto S) {
        hipLaunchKernelGGL((polar::prop_pi_kernel<L(), S()>), dim3(blocks_for(3 * n * stride * lanes)), dim3(256), 0,
                           st, phys(ctx), tab, dq, (const unsigned*)items, (const unsigned*)offs, (double*)pib,
                           stride);
    });
    HIPCHK(ctx, hipGetLastError());
    hipLaunchKernelGGL(polar::prop_compose_kernel, dim3(blocks_for(n)), dim3(256), 0, st, n, dq, dkc, ctx->params.G,
                       ctx->params.K, ctx->params.N_color, (const double*)pib, dout);
    HIPCHK(ctx, hipGetLastError());
    HIPCHK(ctx, hipEventRecord(ctx->ev1, st));
    if (!dev) HIPCHK(ctx, hipMemcpyAsync(out, dout, (size_t)n * 4 * sizeof(double), hipMemcpyDeviceToHost, st));
    if (!(flags & PNJL_FLAG_ASYNC) || !dev) {
        HIPCHK(ctx, hipStreamSynchronize(st));
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess) ctx->last_ms = ms;
    }
    return PNJL_OK;
}

int pnjl_meson_mass_batch(pnjl_ctx* ctx, int64_t n, const pnjl_mass_query* q, const double* kc, double* out,
                          int flags, void* stream)
{
    if (!ctx) return PNJL_ERR_ARG;
    if (n < 0 || (n > 0 && (!q || !out)) || n > ((int64_t)1 << 28) ||
        ((flags & PNJL_FLAG_ONE_PER_WAVE) && n > ((int64_t)1 << 22)))
        return set_err(ctx, PNJL_ERR_ARG, "pnjl_meson_mass_batch: bad argument");
    if (n == 0) return PNJL_OK;
    HIPCHK(ctx, hipSetDevice(ctx->device));
    hipStream_t st = (hipStream_t)stream;
    const bool dev = flags & PNJL_FLAG_DEVICE_PTRS;
    if (!dev)
        for (int64_t i = 0; i < n; i++)
            if (q[i].meson < 0 || q[i].meson >= PNJL_MESON_ID_COUNT || q[i].max_iter < 0)
                return set_err(ctx, PNJL_ERR_ARG, "pnjl_meson_mass_batch: unknown meson or negative max_iter");
    double* tab = nullptr;
    if (int rc = polar_tab(ctx, &tab)) return rc;
    const pnjl_mass_query* dq = q;
    const double* dkc = kc;
    double* dout = out;
    if (!dev) {
        void *a, *b, *c = nullptr;
        if (int rc = stage_buf(ctx, 86, (size_t)n * sizeof(pnjl_mass_query), &a)) return rc;
        if (int rc = stage_buf(ctx, 87, (size_t)n * 6 * sizeof(double), &b)) return rc;
        if (kc)
            if (int rc = stage_buf(ctx, 88, (size_t)n * PNJL_KCOEF_FIELDS * sizeof(double), &c)) return rc;
        HIPCHK(ctx, hipMemcpyAsync(a, q, (size_t)n * sizeof(pnjl_mass_query), hipMemcpyHostToDevice, st));
        if (kc)
            HIPCHK(ctx, hipMemcpyAsync(c, kc, (size_t)n * PNJL_KCOEF_FIELDS * sizeof(double), hipMemcpyHostToDevice,
                                       st));
        dq = (const pnjl_mass_query*)a;
        dkc = (const double*)c;
        dout = (double*)b;
    }
    // phases of growing iteration budgets; the last one runs every remaining
    // query to its end (max_iter)
    constexpr int kPhases = 8;
    const int budgets[kPhases] = {16, 16, 32, 64, 128, 256, 512, -1};
    void *vs = nullptr, *vl0 = nullptr, *vl1 = nullptr, *vc = nullptr;
    if (int rc = stage_buf(ctx, 89, (size_t)n * sizeof(polar::MassState), &vs)) return rc;
    if (int rc = stage_buf(ctx, 90, (size_t)n * sizeof(int32_t), &vl0)) return rc;
    if (int rc = stage_buf(ctx, 91, (size_t)n * sizeof(int32_t), &vl1)) return rc;
    if (int rc = stage_buf(ctx, 92, kPhases * sizeof(unsigned), &vc)) return rc;
    unsigned* cnt = (unsigned*)vc;
    int32_t* lists[2] = {(int32_t*)vl0, (int32_t*)vl1};
    HIPCHK(ctx, hipEventRecord(ctx->ev0, st));
    hipLaunchKernelGGL(polar::zero_u32, dim3(1), dim3(64), 0, st, cnt, kPhases);
    const int stride = (flags & PNJL_FLAG_ONE_PER_WAVE) ? 64 : 1;
    // from kTailPhase on: few queries, hundreds of iterations each.  16 lanes
    // for every other phase (524 288 queries: 111 ms, with one lane in the
    // first two phases 153), 64 in the tail while the longest searches set the
    // time (tail at 16 / 64 lanes: 18 432 queries 21.7 / 13.0 ms, 131 072
    // queries 50 / 43); one lane where 16 pass the launch limit of 2^32 - 1
    // threads (the last 16 batch sizes of all).
    constexpr int kTailPhase = 2;
    const bool one = stride > 1 || 256 * (int64_t)blocks_for(16 * n) > 0xffffffffLL;
    const int head = one ? 1 : 16, tail = (!one && n <= 131072) ? 64 : head;
    for (int ph = 0; ph < kPhases; ph++) {
        const int32_t* in_list = ph == 0 ? nullptr : lists[(ph - 1) & 1];
        const unsigned* in_count = ph == 0 ? nullptr : cnt + ph - 1;
        const int lanes = ph >= kTailPhase ? tail : head;
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(blocks_for(n * stride * lanes)), dim3(256), 0, st, phys(ctx), tab, n, dq,
                               dkc, ctx->params.G, ctx->params.K, ctx->params.N_color, dout, stride,
                               (polar::MassState*)vs, in_list, in_count, lists[ph & 1], cnt + ph, budgets[ph]);
        };
        if (lanes == 64) launch(polar::mass_kernel<64>);
        else if (lanes == 16) launch(polar::mass_kernel<16>);
        else launch(polar::mass_kernel<1>);
        HIPCHK(ctx, hipGetLastError());
    }
    HIPCHK(ctx, hipEventRecord(ctx->ev1, st));
    if (!dev) HIPCHK(ctx, hipMemcpyAsync(out, dout, (size_t)n * 6 * sizeof(double), hipMemcpyDeviceToHost, st));
    if (!(flags & PNJL_FLAG_ASYNC) || !dev) {
        HIPCHK(ctx, hipStreamSynchronize(st));
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1) == hipSuccess) ctx->last_ms = ms;
    }
    return PNJL_OK;
}

}  // extern "C"
