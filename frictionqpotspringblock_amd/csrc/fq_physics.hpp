// Per-particle force laws of the reference's policies, written as functions
// of register values so that every kernel (resident, service, no-passing)
// evaluates exactly the same expression tree as the reference.
#pragma once

#include "fq_common.hpp"

namespace fq {

constexpr double FQ_PI = 3.14159265358979323846;

// Cuspy::force detail.h:164-169: f = mu * (0.5 * (y_l + y_r) - u)
// SemiSmooth::force detail.h:261-276
// Smooth::force detail.h:402-408 (sin evaluated with fq_sin)
template <int POT>
FQ_HD double potential_force(const SysView& S, double u, double yl, double yr)
{
    if constexpr (POT == POT_CUSPY) {
        return (0.5 * (yl + yr) - u) * S.mu;
    }
    else if constexpr (POT == POT_SEMISMOOTH) {
        const double mu = S.mu, kappa = S.kappa;
        double xi = 0.5 * (yl + yr);
        double u_r = (mu * xi + kappa * yr) / (mu + kappa);
        double u_l = (mu * xi + kappa * yl) / (mu + kappa);
        if (u < u_l) {
            return kappa * (u - yl);
        }
        if (u <= u_r) {
            return mu * (0.5 * (yl + yr) - u);
        }
        return kappa * (u - yr);
    }
    else {
        double umin = 0.5 * (yl + yr);
        double dy = 0.5 * (yr - yl);
        return -S.mu * dy / FQ_PI * fq_sin(FQ_PI * (u - umin) / dy);
    }
}

// a / b, correctly rounded as the division is, from the correctly rounded
// reciprocal rb = 1 / b: two residual corrections, the last one from a
// quotient that is faithful (Markstein, IBM J. Res. Dev. 34, 1990), five
// operations instead of the division's eleven and no chain through the
// reciprocal. Exact for 2^-900 <= |a| < 2^900 and 2^-100 < b < 2^100 (no
// residual underflows); the callers divide outside.
FQ_HD double div_rcp(double a, double b, double rb)
{
    double q = a * rb;
    q = __builtin_fma(__builtin_fma(-b, q, a), rb, q);
    q = __builtin_fma(__builtin_fma(-b, q, a), rb, q);
    return q;
}

// The same forces with the constants of the current well computed once per
// well (when it changes) instead of every step: Cuspy its mid-point (c0);
// SemiSmooth the edges u_l (c0), u_r (c1) of the parabolic part (two
// divisions); Smooth the prefactor (-mu dy) / pi of the sine (c0) and 1 / dy
// (c1). Each constant is the subexpression of potential_force above (the
// quotient of the sine's argument is the division's, div_rcp), so the force
// is bit-identical. Selections instead of branches: the particles of a thread
// are then computed side by side.
template <int POT, class Sys>
FQ_HD void well_consts(const Sys& S, double yl, double yr, double& c0, double& c1)
{
    if constexpr (POT == POT_CUSPY) {
        c0 = 0.5 * (yl + yr);
        c1 = 0.0;
    }
    else if constexpr (POT == POT_SEMISMOOTH) {
        const double mu = S.mu, kappa = S.kappa;
        double xi = 0.5 * (yl + yr);
        c0 = (mu * xi + kappa * yl) / (mu + kappa);
        c1 = (mu * xi + kappa * yr) / (mu + kappa);
    }
    else {
        double dy = 0.5 * (yr - yl);
        c0 = -S.mu * dy / FQ_PI;
        c1 = dy > 0x1p-100 && dy < 0x1p100 ? 1.0 / dy : __builtin_nan("");
    }
}

template <int POT, class Sys>
FQ_HD double potential_force_wc(const Sys& S, double u, double yl, double yr, double c0, double c1)
{
    if constexpr (POT == POT_CUSPY) {
        return (c0 - u) * S.mu;
    }
    else if constexpr (POT == POT_SEMISMOOTH) {
        const bool in = u <= c1, left = u < c0;
        const double k = S.kappa * (u - (left ? yl : yr));
        const double m = S.mu * (0.5 * (yl + yr) - u);
        return in && !left ? m : k;
    }
    else {
        const double umin = 0.5 * (yl + yr);
        const double dy = 0.5 * (yr - yl);
        const double a = FQ_PI * (u - umin);
        double x = div_rcp(a, dy, c1);
        // outside 2^-900 <= |a| < 2^900 and for wells without a reciprocal:
        // the division
        const uint32_t e = (hiword(a) & 0x7fffffff) - 0x07b00000u;
        if (e >= 0x70800000u || x != x) {
            x = a / dy;
        }
        return c0 * fq_sin(x);
    }
}

// maxUniformDisplacement of one particle in its current well (yl <= u < yr):
//   Cuspy      detail.h:177-187  distance to the well's edge in `direction`
//   SemiSmooth detail.h:283-330  distance to the edge of the parabolic part;
//              `outside` is set (and +inf returned) when u is outside it
template <int POT>
FQ_HD double max_uniform_particle(const SysView& S, double up, double yl, double yr, int direction, int& outside)
{
    if constexpr (POT == POT_CUSPY) {
        return direction > 0 ? yr - up : up - yl;
    }
    else {
        const double mu = S.mu, kappa = S.kappa;
        double xi = 0.5 * (yl + yr);
        double u_r = (mu * xi + kappa * yr) / (mu + kappa);
        double u_l = (mu * xi + kappa * yl) / (mu + kappa);
        if (up < u_l || !(up <= u_r)) {
            outside = 1;
            return __builtin_inf();
        }
        return direction > 0 ? u_r - up : up - u_l;
    }
}

// Nearest-neighbour chain interactions of particle with slip u and
// neighbours um (p-1) and up (p+1), periodic.
//   Laplace1d         detail.h:480-486
//   Quartic1d         detail.h:784-803
//   QuarticGradient1d detail.h:642-651
// 2 u is exact, so um - 2 u rounds once either way: one fused operation.
template <int INT>
FQ_HD double chain_force(const SysView& S, double um, double u, double up)
{
    if constexpr (INT == INT_LAPLACE1D) {
        return (__builtin_fma(-2.0, u, um) + up) * S.k;
    }
    else if constexpr (INT == INT_QUARTIC1D) {
        double dup = up - u;
        double dun = um - u;
        return S.a1 * (__builtin_fma(-2.0, u, um) + up) + S.a2 * (dup * dup * dup + dun * dun * dun);
    }
    else if constexpr (INT == INT_QUARTICGRADIENT1D) {
        double du = up - um;
        return (__builtin_fma(-2.0, u, um) + up) * (S.k2 + S.k4_4 * du * du);
    }
    else {
        return 0.0;
    }
}

FQ_HD int64_t wrap(int64_t i, int64_t n)
{
    return i < 0 ? i + n : (i >= n ? i - n : i);
}

// Lattice interactions of site (i, j) read from a row-major slip field U;
// S supplies rows, cols (the periodic wrap) and k, k2, k4 (the system, or the
// extended rows of a tile).
//   Laplace2d         detail.h:545-583
//   QuarticGradient2d detail.h:682-750
template <int INT, class Sys, class Acc>
FQ_HD double lattice_force(const Sys& S, const Acc& U, int64_t i, int64_t j)
{
    const int64_t R = S.rows, C = S.cols;
    const int64_t im = wrap(i - 1, R), ip = wrap(i + 1, R), jm = wrap(j - 1, C), jp = wrap(j + 1, C);
    const double c0 = U(i * C + j);
    if constexpr (INT == INT_LAPLACE2D) {
        return (U(im * C + j) + U(ip * C + j) + U(i * C + jm) + U(i * C + jp) - 4 * c0) * S.k;
    }
    else {
        const double mk4_3 = S.k4 / 3.0;
        const double mk4_23 = 2.0 * mk4_3;
        const double uip = U(ip * C + j), uim = U(im * C + j), ujp = U(i * C + jp), ujm = U(i * C + jm);
        double l = uip + uim + ujp + ujm - 4 * c0;
        double dudx = 0.5 * (uip - uim);
        double dudy = 0.5 * (ujp - ujm);
        double d2udxdy = 0.25 * (U(ip * C + jp) - U(ip * C + jm) - U(im * C + jp) + U(im * C + jm));
        double d2udx2 = uip - 2 * c0 + uim;
        double d2udy2 = ujp - 2 * c0 + ujm;
        return l * (S.k2 + mk4_3) + mk4_23 * (dudx * dudx * d2udx2 + dudy * dudy * d2udy2 + 2.0 * dudx * dudy * d2udxdy);
    }
}

// The same of the site in row offset ric, column cjc (slip c0) with the rows
// above and below at offsets rim, rip and the columns beside it at cjm, cjp
// of the slip field U (the periodic wrap and the divisions done once per site
// instead of every step; 4 c0 is exact, so its subtraction rounds once either
// way).
template <int INT, class Sys>
FQ_HD double lattice_force_at(const Sys& S, const double* U, int rim, int ric, int rip, int cjm, int cjc, int cjp,
                              double c0)
{
    const double uim = U[rim + cjc], uip = U[rip + cjc], ujm = U[ric + cjm], ujp = U[ric + cjp];
    if constexpr (INT == INT_LAPLACE2D) {
        return __builtin_fma(-4.0, c0, uim + uip + ujm + ujp) * S.k;
    }
    else {
        const double mk4_3 = S.k4 / 3.0;
        const double mk4_23 = 2.0 * mk4_3;
        const double l = __builtin_fma(-4.0, c0, uip + uim + ujp + ujm);
        const double dudx = 0.5 * (uip - uim);
        const double dudy = 0.5 * (ujp - ujm);
        const double d2udxdy = 0.25 * (U[rip + cjp] - U[rip + cjm] - U[rim + cjp] + U[rim + cjm]);
        const double d2udx2 = __builtin_fma(-2.0, c0, uip) + uim;
        const double d2udy2 = __builtin_fma(-2.0, c0, ujp) + ujm;
        return l * (S.k2 + mk4_3) + mk4_23 * (dudx * dudx * d2udx2 + dudy * dudy * d2udy2 + 2.0 * dudx * dudy * d2udxdy);
    }
}

// LongRange1d::force detail.h:852-866 of a particle with slip `up`:
// sequential sum over i = 0..N-1. G[i] is the prefactor of the pair, from the
// table prefx of all differences i - p (G = prefx + N - 1 - p),
// so that a term is three operations without the fold of the distance; the
// particle's own entry is zero and adds +0 to a sum that is never -0.
// The sum is one chain of additions per particle: the operands of the next
// eight terms are loaded while the current eight are added (a step of a chain
// of 1000 over tiles: 16 us instead of 21 us with the compiler's unrolled
// loop; resident 56 us, LDS-bound, instead of 130 us with folded distances).
template <class Acc, class Pref>
FQ_HD double longrange_force(int n, const Acc& U, const Pref& G, double up)
{
    constexpr int C = 8;
    double fp = 0.0, x0[C], g0[C], x1[C], g1[C];
    auto load = [&](int i, double(&x)[C], double(&g)[C]) {
#pragma unroll
        for (int q = 0; q < C; ++q) {
            x[q] = U(i + q);
            g[q] = G(i + q);
        }
    };
    auto add = [&](const double(&x)[C], const double(&g)[C]) {
        double y[C]; // (independent of the chain)
#pragma unroll
        for (int q = 0; q < C; ++q) {
            y[q] = (x[q] - up) * g[q];
        }
#pragma unroll
        for (int q = 0; q < C; ++q) {
            fp += y[q];
        }
    };
    int i = 0;
    if (n >= C) {
        load(0, x0, g0);
        for (; i + 2 * C <= n; i += 2 * C) {
            load(i + C, x1, g1);
            add(x0, g0);
            if (i + 3 * C <= n) {
                load(i + 2 * C, x0, g0);
            }
            add(x1, g1);
        }
        if (i + C <= n) { // an odd number of blocks: the last one is loaded
            add(x0, g0);
            i += C;
        }
    }
    for (; i < n; ++i) {
        fp += (U(i) - up) * G(i);
    }
    return fp;
}

} // namespace fq
