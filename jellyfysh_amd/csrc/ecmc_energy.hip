// ecmc_energy.hip -- total pair energy of one configuration and its hand-written backward
// kernel: gradients with respect to the positions, to the potential's parameters and to
// the charges.
//
// U = 1/2 sum_i sum_{j != i, (i, j) in scope} U(s_ij), s_ij = minimum-image separation
// (hypercubic_setting.py:101-126).  The position gradient of a pair is the potential's own
// directional derivative -- the same device functions ECMC inverts
// (inverse_power_potential.py:71-94, lennard_jones_potential.py:63-81,
// displaced_even_power_potential.py:73-93, merged_image_coulomb_potential.c:205-274) -- so
// dU/dx_{i,d} = sum_j derivative(e_d, s_ij, c_i, c_j).
//
// One workgroup per row i: its 256 threads stride over j in a fixed order and reduce in a
// fixed tree, and a last kernel sums the rows in a fixed order, so results do not depend on
// scheduling.  All scratch lives in a caller-provided workspace; nothing is allocated here.
#include <hip/hip_runtime.h>
#include <math.h>
#include <string.h>
#include <algorithm>

#include "../../include/jellyfysh_amd.h"
#include "ecmc_common.h"
#include "ecmc_math.h"
#include "ecmc_potentials.h"

namespace ecmc {

constexpr int ET = 256;
constexpr int EROW = 9;   // a row's sums: energy, dU/dx_i (3), dU/dpar (4), dU/dc_i

// ---- merged-image Coulomb -------------------------------------------------------------------
// Pair function psi(s) = sum over the real-space images of the derivative's sphere of
// erfc(a |s + nL|) / |s + nL| + (1 / (pi L)) sum_{0 < |n| <= fc} exp(-pi^2 n^2 / alpha^2) / n^2
// cos(2 pi n.s / L) - pi / (alpha^2 L), a = alpha / L.  Its gradient is the reference's derivative;
// the last term (the neutralising background) makes psi independent of alpha up to truncation.
//
// A row's sum over j splits: the real-space images pair by pair, value and gradient from one
// exponential, root and reciprocal; the Fourier part through the structure factors
// S(k) = sum_j c_j exp(i k.x_j) (sum_j c_j cos(k.(x_j - x_i)) = Re(exp(-i k.x_i) S(k))), O(n) per
// wave vector instead of O(n^2), less the row's own term and the pairs out of scope.  Evaluated
// pair by pair (three calls of the derivative and one of psi, each with its own erfc and its own
// Fourier sum), 1000 units took 777 us forward and 1915 us backward.
//
// S(k) holds every charge of the system, so what a row takes off it again leaves rounding errors of
// that size.  A row takes this form only where the charge to take off (its own and its units' out of
// scope, by magnitude) is at most that of its partners, which bounds its error by twice the plain
// sum's; the other rows add their pairs' Fourier parts one by one.
struct CoulombWork {
    int32_t fc, n_img, direct;         // direct: the Fourier part pair by pair in every row (scope intra)
    double L, aol, aol2, two_aol_rpi, tpol, background;
    double2 *phase;                    // exp(2 pi i m x_d / L): [(d (fc + 1) + m) n + unit]
    double2 *S;                        // structure factors: wave vector of the half space (kvector)
    double *g;                         // Fourier weights of the octant [(i (fc + 1) + j) (fc + 1) + k]
    double *img;                       // image offsets, n_img x 3
    int32_t *pairwise;                 // per row: not 0 where it adds its pairs' Fourier parts one by one
};

struct EnergyArgs {
    int32_t pot, scope, use_charge, n;
    double par[4];
    double L, half;
    const double *pos;
    const double *charge;
    const int32_t *mol;
    CoulombWork cw;
    double *rows;        // n x EROW: energy, -, -, -, dU/dpar (4), -
    double *grad_pos, *grad_charge;
};

// Wave vector number v: (i, j, k) with 0 <= i <= fc, |j|, |k| <= fc; true in the half space (one of
// each pair k, -k) inside the sphere.
__device__ __forceinline__ bool kvector(int fc, int v, int &i, int &j, int &k) {
    const int w = 2 * fc + 1;
    i = v / (w * w);
    j = (v / w) % w - fc;
    k = v % w - fc;
    const bool half = i > 0 || j > 0 || (j == 0 && k > 0);
    return half && i * i + j * j + k * k <= fc * fc;
}
__device__ __forceinline__ int kvectors(int fc) { return (fc + 1) * (2 * fc + 1) * (2 * fc + 1); }

// exp(2 pi i (i x + j y + k z) / L) of one unit.
__device__ __forceinline__ double2 kphase(const CoulombWork &c, int n, int unit, int i, int j, int k) {
    const int nn = c.fc + 1;
    const double2 a = c.phase[(size_t)i * n + unit];
    double2 b = c.phase[(size_t)(nn + abs(j)) * n + unit], d = c.phase[(size_t)(2 * nn + abs(k)) * n + unit];
    b.y = j < 0 ? -b.y : b.y;
    d.y = k < 0 ? -d.y : d.y;
    const double2 e = make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
    return make_double2(fma(e.x, d.x, -(e.y * d.y)), fma(e.x, d.y, e.y * d.x));
}

// Phases of every unit and axis (x / L with its remainder, each multiple reduced to one period before
// its sine and cosine), the Fourier weights and the image offsets.
__global__ __launch_bounds__(ET) void coulomb_setup(EnergyArgs A, int position_cutoff, double alpha) {
    const CoulombWork &c = A.cw;
    const int nn = c.fc + 1, at = blockIdx.x * ET + threadIdx.x, n = A.n;
    if (at < 3 * n) {
        const int d = at / n, unit = at % n;
        const double x = A.pos[3 * (size_t)unit + d], h = x / c.L, rest = fma(-h, c.L, x) / c.L;
        for (int m = 0; m < nn; m++) {
            const double t = m * h, more = fma((double)m, h, -t) + m * rest;
            double s0, c0;
            sincospi(2.0 * (t - rint(t)), &s0, &c0);
            const double e = 2.0 * M_PI * more;
            c.phase[(size_t)(d * nn + m) * n + unit] = make_double2(fma(-s0, e, c0), fma(c0, e, s0));
        }
    }
    if (at < nn * nn * nn) {
        const int i = at / (nn * nn), j = (at / nn) % nn, k = at % nn, n2 = i * i + j * j + k * k;
        const double w = (i ? 2.0 : 1.0) * (j ? 2.0 : 1.0) * (k ? 2.0 : 1.0);
        c.g[at] = n2 == 0 || n2 > c.fc * c.fc ? 0.0 : w * exp(-M_PI * M_PI * n2 / (alpha * alpha)) / (M_PI * c.L * n2);
    }
    if (at == 0) {
        int m = 0;
        const int pc = position_cutoff;
        for (int k = -pc; k <= pc; k++)
            for (int j = -pc; j <= pc; j++)
                for (int i = -pc; i <= pc; i++)
                    if (i * i + j * j + k * k <= pc * pc) {
                        c.img[3 * m] = i * c.L;
                        c.img[3 * m + 1] = j * c.L;
                        c.img[3 * m + 2] = k * c.L;
                        m++;
                    }
    }
}

// Fixed-order sum over the lanes of a wavefront, in every lane.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Whether unit j is a partner of a row of molecule mi (j not the row's own unit).
__device__ __forceinline__ bool in_scope(const EnergyArgs &A, int mi, int j) {
    return A.scope == ECMC_SCOPE_ALL || (A.mol[j] == mi) == (A.scope == ECMC_SCOPE_INTRA);
}

// The form of row i's Fourier part, by one wavefront.
__device__ __forceinline__ void coulomb_row_form(const EnergyArgs &A, int i, int lane) {
    const int mi = A.scope != ECMC_SCOPE_ALL ? A.mol[i] : 0;
    double held = 0.0, excess = 0.0;   // the partners' charge, and the rest's
    for (int j = lane; j < A.n; j += 64) {
        const double q = A.use_charge ? fabs(A.charge[j]) : 1.0;
        if (j == i) excess += q;
        else if (in_scope(A, mi, j)) held += q;
        // (NaN where a unit is somewhere that is not finite: the structure factors then are NaN too)
        else excess += q + 0.0 * (A.pos[3 * (size_t)j] + A.pos[3 * (size_t)j + 1] + A.pos[3 * (size_t)j + 2]);
    }
    held = wave_sum(held);
    excess = wave_sum(excess);
    if (lane == 0) A.cw.pairwise[i] = !(excess <= held);
}

// One wavefront per row and per wave vector.  (1000 units: 9.6 us, 8.1 without the rows' forms; summed in
// each row's own workgroup they took 3.5 us a launch.)
__global__ __launch_bounds__(ET) void coulomb_structure(EnergyArgs A) {
    const CoulombWork &c = A.cw;
    const int row = blockIdx.x * (ET / 64) + (threadIdx.x >> 6), v = row - A.n, lane = threadIdx.x & 63;
    if (row < A.n) {
        coulomb_row_form(A, row, lane);
        return;
    }
    int i, j, k;
    if (v >= kvectors(c.fc) || !kvector(c.fc, v, i, j, k)) return;
    double re = 0.0, im = 0.0;
    for (int u = lane; u < A.n; u += 64) {
        const double2 e = kphase(c, A.n, u, i, j, k);
        const double q = A.use_charge ? A.charge[u] : 1.0;
        re = fma(q, e.x, re);
        im = fma(q, e.y, im);
    }
    re = wave_sum(re);
    im = wave_sum(im);
    if (lane == 0) c.S[v] = make_double2(re, im);
}

// Scaled complementary error function exp(x^2) erfc(x) for x >= 0: (1 + 2x) erfcx(x) as a polynomial
// in t = (x - 3.75) / (x + 3.75) (Shepherd and Laframboise, Math. Comp. 36, 249 (1981)), degree 24
// through the Chebyshev nodes of 80-digit values: 5.4e-18 off, 2.6e-16 with the roundings.  One
// reciprocal, no branch, where erfc takes one of four expansions and an exponential of its own.
__device__ __forceinline__ double erfcx_poly(double x) {
    static constexpr double C[25] = {0x1.3ccda0b5d5dc2p+0, -0x1.1f367683f89a5p-3, 0x1.d5f2948159e20p-9, 0x1.510169d096658p-4,
    -0x1.bda9309a28be0p-4, 0x1.7a14188a9ce86p-4, -0x1.e0d0fa6df428dp-5, 0x1.d0b0037d155f4p-6,
    -0x1.3f603c3682d81p-7, 0x1.cc3a0e7d99253p-10, 0x1.33fb27421f98cp-12, -0x1.303fa49e236d5p-12,
    0x1.b143d63ea931ep-15, 0x1.778b948121ce1p-16, -0x1.8002c11990e5bp-17, -0x1.0556aa18e657bp-20,
    0x1.d65081c59291dp-20, -0x1.eb7b41166a177p-25, -0x1.1636c8002e495p-22, 0x1.8fa2f9fdc0311p-26,
    0x1.4eb5efb28ed5dp-25, -0x1.01418b99efa2ep-28, -0x1.6b2228df54be4p-28, 0x1.55fb76b7dbdcfp-32,
    0x1.e7a100062f385p-32};
    const double lo = x + 3.75, hi = fma(2.0, x, 1.0), q = lo * hi;
    double r = __builtin_amdgcn_rcp(q);
    r = fma(r, fma(-q, r, 1.0), r);
    r = fma(r, fma(-q, r, 1.0), r);
    const double t = (x - 3.75) * hi * r;
    double p = C[24];
#pragma unroll
    for (int k = 23; k >= 0; k--) p = fma(p, t, C[k]);
    return p * (lo * r);
}

// Real-space part of psi(s) and, with BW, of its gradient (the derivative's sign).
template <bool BW>
__device__ __forceinline__ void coulomb_real(const CoulombWork &c, const double *s, double &psi, double *der) {
    psi = 0.0;
    if (BW) der[0] = der[1] = der[2] = 0.0;
    const double *__restrict__ img = c.img;
#pragma unroll 1
    for (int m = 0; m < c.n_img; m++) {
        const double vx = s[0] + img[3 * m], vy = s[1] + img[3 * m + 1], vz = s[2] + img[3 * m + 2];
        const double d2 = fma(vx, vx, fma(vy, vy, vz * vz));
        const bool touch = d2 == 0.0;   // two units at one place: an infinite value
        const double v2 = touch ? 1.0 : d2;
        // 1 / |v| to rounding: the hardware root (2^-26) and a third-order step
        double y = __builtin_amdgcn_rsq(v2);
        const double e = fma(-v2 * y, y, 1.0);
        y = fma(y * e, fma(e, 0.375, 0.5), y);
        double vn = v2 * y;
        vn = fma(0.5 * y, fma(-vn, vn, v2), vn);
        const double E = exp(-c.aol2 * v2);
        double f = E * erfcx_poly(c.aol * vn) * y;
        f = touch ? INFINITY : f;
        psi += f;
        if (BW) {
            const double h = fma(c.two_aol_rpi, E, f) * y * y;
            der[0] = fma(vx, h, der[0]);
            der[1] = fma(vy, h, der[1]);
            der[2] = fma(vz, h, der[2]);
        }
    }
}

// Fourier part of one pair from its units' phases: psi, and the gradient with the derivative's sign.
template <bool BW>
__device__ void coulomb_fourier_pair(const CoulombWork &c, int n, int a, int b, double &psi, double *der) {
    const int fc = c.fc, nn = fc + 1;
    auto axis = [&](int d, int m) {   // exp(2 pi i m (x_b - x_a) / L)
        const double2 p = c.phase[(size_t)(d * nn + m) * n + a], q = c.phase[(size_t)(d * nn + m) * n + b];
        return make_double2(fma(p.x, q.x, p.y * q.y), fma(p.x, q.y, -(p.y * q.x)));
    };
    psi = 0.0;
    double gx = 0.0, gy = 0.0, gz = 0.0;
    for (int i = 0; i <= fc; i++) {
        const double2 ex = axis(0, i);
        for (int j = 0; i * i + j * j <= fc * fc; j++) {
            const double2 ey = axis(1, j);
            for (int k = 0; i * i + j * j + k * k <= fc * fc; k++) {
                const double2 ez = axis(2, k);
                const double g = c.g[(i * nn + j) * nn + k], cc = g * ex.x * ey.x;
                psi = fma(cc, ez.x, psi);
                if (BW) {
                    gx = fma(g * (i * ex.y) * ey.x, ez.x, gx);
                    gy = fma(g * ex.x * (j * ey.y), ez.x, gy);
                    gz = fma(cc, k * ez.y, gz);
                }
            }
        }
    }
    if (BW) {
        der[0] = c.tpol * gx;
        der[1] = c.tpol * gy;
        der[2] = c.tpol * gz;
    }
}

// ---- the other potentials -------------------------------------------------------------------
// r2 ** (p / 2) correctly rounded (without a call for p = 6 and 12 in the usual range).
__device__ __forceinline__ double power_of(double r2, double p) {
    return p == 12.0 || p == 6.0 ? pow36(r2, p == 12.0) : cr_pow(r2, p / 2.0);
}

// What a pair needs of the parameters alone.
struct PairConstants {
    double k6, k12, s6, s12;      // Lennard-Jones: -k sigma^6, k sigma^12, sigma^6, sigma^12
    double rc2, rcp, lrc;         // truncated inverse power: cutoff^2, rc^-p, log rc
};
__device__ __forceinline__ PairConstants pair_constants(const EnergyArgs &A, int pot) {
    PairConstants c = {};
    if (pot == ECMC_POT_LENNARD_JONES) {
        const double x = A.par[1];   // cr_pow's double-double powers, the second the first's square
        if (x > 0x1p-30 && x < 0x1p30) {
            const dd x3 = dd_mul_d(two_prod(x, x), x), x6 = dd_mul(x3, x3);
            c.s6 = x6.h;
            c.s12 = dd_mul(x6, x6).h;
        } else {
            c.s6 = cr_pow(x, 6.0);
            c.s12 = cr_pow(x, 12.0);
        }
        c.k6 = -A.par[0] * c.s6;
        c.k12 = A.par[0] * c.s12;
    } else if (pot == ECMC_POT_INVERSE_POWER_TRUNC) {
        c.rc2 = A.par[2] * A.par[2];
        c.rcp = 1.0 / power_of(c.rc2, A.par[0]);
        c.lrc = cr_log(A.par[2]);
    }
    return c;
}

// Pair value u (charges included), the factor f of its gradient (dU/dx_i = f s), the parameter
// gradient and du/dc_i.  The powers of a pair are taken once: u's own serve the gradient
// (d/dr r^-p = -p r^-p / r), where each axis took two correctly rounded powers and a root.
template <int POT, bool BW>
__device__ __forceinline__ void pair_terms(const EnergyArgs &A, const PairConstants &c, double r2, double ci, double cj, double &u,
                                           double &f, double *dp, double &dc) {
    const double cp = ci * cj;
    u = f = dc = 0.0;
    dp[0] = dp[1] = dp[2] = 0.0;
    if (POT == ECMC_POT_INVERSE_POWER || POT == ECMC_POT_INVERSE_POWER_TRUNC) {
        const double p = A.par[0], k = A.par[1];
        const bool trunc = POT == ECMC_POT_INVERSE_POWER_TRUNC;
        if (trunc && !(r2 < c.rc2)) return;
        const double rp = 1.0 / power_of(r2, p);   // r^-p
        const double rcp = trunc ? c.rcp : 0.0;
        u = cp * k * (rp - rcp);
        if (BW) {
            f = p * (k * cp) * rp / r2;
            const double lr = 0.5 * cr_log(r2);
            dp[0] = -cp * k * (rp * lr - (trunc ? rcp * c.lrc : 0.0));
            dp[1] = cp * (rp - rcp);
            if (trunc) dp[2] = cp * k * p * rcp / A.par[2];
            dc = cj * k * (rp - rcp);
        }
    } else if (POT == ECMC_POT_LENNARD_JONES) {
        const double p3 = pow36(r2, false), p6 = pow36(r2, true);
        const double u6 = c.k6 / p3, u12 = c.k12 / p6;
        u = u6 + u12;
        if (BW) {
            f = (6.0 * u6 + 12.0 * u12) / r2;
            const double x6 = c.s6 / p3, x12 = c.s12 / p6;
            dp[0] = x12 - x6;
            dp[1] = A.par[0] * (12.0 * x12 - 6.0 * x6) / A.par[1];
        }
    } else if (POT == ECMC_POT_DISPLACED_EVEN_POWER) {
        const double r0 = A.par[0], p = A.par[1], k = A.par[2];
        const double r = sqrt(r2), dr = r - r0, dpw = cr_pow(dr, p);
        u = k * dpw;
        if (BW) {
            const double d1 = k * p * cr_pow(dr, p - 1.0);
            f = -d1 / r;
            dp[0] = -d1;
            dp[1] = dr != 0.0 ? k * dpw * cr_log(fabs(dr)) : 0.0;
            dp[2] = dpw;
        }
    }
}

// Minimum image of x in [0, L) (py_mod, whose one-period cases need no fmod).
__device__ __forceinline__ double wrapped(double x, double L) {
    if (x >= 0.0 && x < L) return x;
    if (x > -L && x < 0.0) return x + L;
    return py_mod(x, L);
}

// One workgroup per row i: its threads stride over j in a fixed order and reduce in a fixed tree.
// Bound by FP64 instructions; measured with the launches around it, see energy_launch.
template <int POT, bool BW>
__global__ __launch_bounds__(ET) void energy_rows(EnergyArgs A) {
    constexpr bool COULOMB = POT == ECMC_POT_MERGED_IMAGE_COULOMB;
    __shared__ double red[ET / 64][EROW];
    const int i = blockIdx.x, t = threadIdx.x, nt = blockDim.x;
    double acc[EROW];   // (Coulomb: [0] sum_j c_j psi, [1 .. 3] its gradient)
#pragma unroll
    for (int q = 0; q < EROW; q++) acc[q] = 0.0;
    const double ai[3] = {A.pos[3 * (size_t)i], A.pos[3 * (size_t)i + 1], A.pos[3 * (size_t)i + 2]};
    const double ci = A.use_charge ? A.charge[i] : 1.0;
    const int mi = A.scope != ECMC_SCOPE_ALL ? A.mol[i] : 0;
    const PairConstants pc = pair_constants(A, POT);
    const bool direct = COULOMB && (A.cw.direct || A.cw.pairwise[i]);
    for (int j = t; j < A.n; j += nt) {
        if (j == i) continue;
        const bool in = in_scope(A, mi, j);
        if (!in && !(COULOMB && !direct)) continue;
        const double cj = A.use_charge ? A.charge[j] : 1.0;
        if (COULOMB) {
            if (in) {
                double s[3], psi, der[3];
#pragma unroll
                for (int d = 0; d < 3; d++) s[d] = wrapped((A.pos[3 * (size_t)j + d] - ai[d]) + A.half, A.L) - A.half;
                coulomb_real<BW>(A.cw, s, psi, der);
                acc[0] = fma(cj, psi + A.cw.background, acc[0]);
                if (BW)
                    for (int d = 0; d < 3; d++) acc[1 + d] = fma(cj, der[d], acc[1 + d]);
            }
            if (in == direct) {   // the row's own pairs, or those that S(k) holds too much
                double psi, der[3];
                coulomb_fourier_pair<BW>(A.cw, A.n, i, j, psi, der);
                const double w = in ? cj : -cj;
                acc[0] = fma(w, psi, acc[0]);
                if (BW)
                    for (int d = 0; d < 3; d++) acc[1 + d] = fma(w, der[d], acc[1 + d]);
            }
        } else {
            double s[3], u, f, dp[3], dc;
#pragma unroll
            for (int d = 0; d < 3; d++) s[d] = wrapped((A.pos[3 * (size_t)j + d] - ai[d]) + A.half, A.L) - A.half;
            pair_terms<POT, BW>(A, pc, norm_sq<3>(s), ci, cj, u, f, dp, dc);
            acc[0] += u;
            if (BW) {
#pragma unroll
                for (int q = 0; q < 3; q++) acc[1 + q] = fma(f, s[q], acc[1 + q]);
#pragma unroll
                for (int q = 0; q < 3; q++) acc[4 + q] += dp[q];
                acc[8] += dc;
            }
        }
    }
    if (COULOMB && !direct) {
        // Re and Im of exp(-i k.x_i) S(k) over the half space, less the row's own term
        const int nv = kvectors(A.cw.fc), nn = A.cw.fc + 1;
        for (int v = t; v < nv; v += nt) {
            int a, b, d;
            if (!kvector(A.cw.fc, v, a, b, d)) continue;
            const double2 e = kphase(A.cw, A.n, i, a, b, d), S = A.cw.S[v];
            // twice the weight of one vector: the octant's weight counts every sign of each axis
            const double g = A.cw.g[(a * nn + abs(b)) * nn + abs(d)] * 2.0 / ((a ? 2.0 : 1.0) * (b ? 2.0 : 1.0) * (d ? 2.0 : 1.0));
            acc[0] = fma(g, fma(e.x, S.x, e.y * S.y) - ci, acc[0]);
            if (BW) {
                const double im = g * A.cw.tpol * fma(e.x, S.y, -(e.y * S.x));
                acc[1] = fma((double)a, im, acc[1]);
                acc[2] = fma((double)b, im, acc[2]);
                acc[3] = fma((double)d, im, acc[3]);
            }
        }
    }
    constexpr int USED = COULOMB ? (BW ? 4 : 1) : (BW ? EROW : 1);
#pragma unroll
    for (int q = 0; q < USED; q++) {
        const double v = wave_sum(acc[q]);
        if ((t & 63) == 0) red[t >> 6][q] = v;
    }
    __syncthreads();
    if (t < EROW) {
        auto total = [&](int q) {
            double s = red[0][q];
            for (int w = 1; w < nt / 64; w++) s += red[w][q];
            return s;
        };
        double out;
        if (COULOMB) {
            const double pre = A.par[3];
            const double sum = total(t >= 1 && t <= 3 && BW ? t : 0);
            out = t == 0 ? pre * ci * sum : (!BW ? 0.0 : (t <= 3 ? pre * ci * sum : (t == 7 ? ci * sum : (t == 8 ? pre * sum : 0.0))));
        } else {
            out = t < USED ? total(t) : 0.0;
        }
        if (t == 0 || (BW && t >= 4 && t <= 7)) A.rows[(size_t)i * EROW + t] = out;
        if (BW && t >= 1 && t <= 3) A.grad_pos[3 * (size_t)i + t - 1] = out;
        if (BW && t == 8 && A.grad_charge) A.grad_charge[i] = out;
    }
}

// Fixed-order sums over the rows: energy, or parameter gradient = half the row sums.
__global__ __launch_bounds__(ET) void energy_finish(const double *rows, int n, int backward, double *energy, double *grad_par) {
    __shared__ double red[ET / 64][4];
    const int t = threadIdx.x, first = backward ? 4 : 0, cols = backward ? 4 : 1;
    double acc[4] = {0, 0, 0, 0};
    for (int i = t; i < n; i += ET)
        for (int q = 0; q < cols; q++) acc[q] += rows[(size_t)i * EROW + first + q];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const double v = q < cols ? wave_sum(acc[q]) : 0.0;
        if ((t & 63) == 0) red[t >> 6][q] = v;
    }
    __syncthreads();
    if (t < cols) {
        double v = red[0][t];
        for (int w = 1; w < ET / 64; w++) v += red[w][t];
        (backward ? grad_par : energy)[t] = 0.5 * v;
    }
}

}  // namespace ecmc

using namespace ecmc;

// Doubles behind the rows: phases, structure factors, Fourier weights, image offsets, the rows' forms.
struct CoulombSizes {
    int64_t phase, S, g, img, form;
    int32_t n_img;
};
static CoulombSizes coulomb_sizes(const ecmc_energy_term *t, int64_t n) {
    CoulombSizes z = {};
    if (t->potential != ECMC_POT_MERGED_IMAGE_COULOMB) return z;
    // (cutoffs out of range are refused by the launch; no workspace is sized for them)
    const int64_t fc = std::min(32, std::max(0, (int)t->par[1])), pc = std::min(8, std::max(0, (int)t->par[2])), nn = fc + 1;
    for (int i = -pc; i <= pc; i++)
        for (int j = -pc; j <= pc; j++)
            for (int k = -pc; k <= pc; k++) z.n_img += i * i + j * j + k * k <= pc * pc;
    z.phase = 2 * 3 * nn * n;
    z.S = 2 * nn * (2 * fc + 1) * (2 * fc + 1);
    z.g = nn * nn * nn;
    z.img = 3 * (int64_t)z.n_img;
    z.form = (n + 1) / 2;
    return z;
}

extern "C" int ecmc_energy_workspace_bytes(const ecmc_energy_term *term, int32_t n, int64_t *bytes) {
    if (!term || !bytes || n < 0) return ecmc_fail(ECMC_ERR_ARGUMENT, "null argument or negative size");
    const CoulombSizes z = coulomb_sizes(term, n);
    *bytes = ((int64_t)n * EROW + (z.n_img ? 1 : 0) + z.phase + z.S + z.g + z.img + z.form) * 8;
    return ECMC_OK;
}

template <int POT>
static void launch_rows(const EnergyArgs &A, bool backward, int threads, hipStream_t st) {
    if (backward) hipLaunchKernelGGL((energy_rows<POT, true>), dim3(A.n), dim3(threads), 0, st, A);
    else hipLaunchKernelGGL((energy_rows<POT, false>), dim3(A.n), dim3(threads), 0, st, A);
}

static int energy_launch(const ecmc_energy_term *term, int32_t n, const double *d_pos, const double *d_charge,
                         const int32_t *d_mol, double L, bool backward, double *d_energy, double *d_grad_pos,
                         double *d_grad_par, double *d_grad_charge, void *d_work, void *stream) {
    if (!term || !d_pos || !d_work) return ecmc_fail(ECMC_ERR_ARGUMENT, "null argument");
    if (n < 2) return ecmc_fail(ECMC_ERR_ARGUMENT, "at least two units");
    if (!(L > 0.0)) return ecmc_fail(ECMC_ERR_ARGUMENT, "system length must be positive");
    if (term->scope < ECMC_SCOPE_ALL || term->scope > ECMC_SCOPE_INTRA)
        return ecmc_fail(ECMC_ERR_ARGUMENT, "unknown pair scope");
    if (term->scope != ECMC_SCOPE_ALL && !d_mol) return ecmc_fail(ECMC_ERR_ARGUMENT, "scope needs molecule indices");
    if (term->use_charge && !d_charge) return ecmc_fail(ECMC_ERR_ARGUMENT, "charged term needs charges");
    if (backward && (!d_grad_pos || !d_grad_par)) return ecmc_fail(ECMC_ERR_ARGUMENT, "null gradient output");
    if (d_grad_charge && !term->use_charge)
        return ecmc_fail(ECMC_ERR_ARGUMENT, "charge gradient of an uncharged term");
    EnergyArgs A;
    memset(&A, 0, sizeof(A));
    A.pot = term->potential;
    A.scope = term->scope;
    A.use_charge = term->use_charge;
    A.n = n;
    for (int q = 0; q < 4; q++) A.par[q] = term->par[q];
    A.L = L;
    A.half = 0.5 * L;
    A.pos = d_pos;
    A.charge = term->use_charge ? d_charge : nullptr;
    A.mol = d_mol;
    A.rows = (double *)d_work;
    A.grad_pos = d_grad_pos;
    A.grad_charge = d_grad_charge;
    hipStream_t st = (hipStream_t)stream;
    switch (A.pot) {
    case ECMC_POT_INVERSE_POWER:
        if (!(A.par[0] > 0.0)) return ecmc_fail(ECMC_ERR_CONFIGURATION, "power must be positive");
        break;
    case ECMC_POT_INVERSE_POWER_TRUNC:
        if (!(A.par[0] > 0.0)) return ecmc_fail(ECMC_ERR_CONFIGURATION, "power must be positive");
        if (!(A.par[2] > 0.0) || A.par[2] > 0.5 * L)
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "cutoff must lie in (0, L/2] (minimum image)");
        break;
    case ECMC_POT_LENNARD_JONES:
        break;
    case ECMC_POT_DISPLACED_EVEN_POWER: {
        double p = A.par[1];
        if (!(p > 0.0) || p != (double)(int)p || ((int)p) % 2)
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "the power must be a positive even integer");
        break;
    }
    case ECMC_POT_MERGED_IMAGE_COULOMB: {
        const int fc = (int)A.par[1], pc = (int)A.par[2];
        const double alpha = A.par[0];
        if (fc < 1 || fc > 32 || pc < 0 || pc > 8 || !(alpha > 0.0))
            return ecmc_fail(ECMC_ERR_CONFIGURATION, "Ewald cutoffs out of range");
        const CoulombSizes z = coulomb_sizes(term, n);
        CoulombWork &c = A.cw;
        double *w = A.rows + (size_t)n * EROW;
        if ((uintptr_t)w & 8) w++;   // 16-byte pairs (the workspace has a double to spare)
        c.phase = (double2 *)w;
        c.S = (double2 *)(w + z.phase);
        c.g = w + z.phase + z.S;
        c.img = c.g + z.g;
        c.pairwise = (int32_t *)(c.img + z.img);
        c.n_img = z.n_img;
        c.fc = fc;
        c.direct = A.scope == ECMC_SCOPE_INTRA;
        c.L = L;
        c.aol = alpha / L;
        c.aol2 = c.aol * c.aol;
        c.two_aol_rpi = 2.0 * c.aol / sqrt(M_PI);
        c.tpol = 2.0 * M_PI / L;
        c.background = -M_PI / (alpha * alpha * L);
        const int nn = fc + 1, tasks = std::max(3 * n, nn * nn * nn);
        hipLaunchKernelGGL(coulomb_setup, dim3((tasks + ET - 1) / ET), dim3(ET), 0, st, A, pc, alpha);
        if (!c.direct) {
            const int nv = nn * (2 * fc + 1) * (2 * fc + 1);
            hipLaunchKernelGGL(coulomb_structure, dim3((n + nv + 3) / 4), dim3(ET), 0, st, A);
        }
        break;
    }
    default:
        return ecmc_fail(ECMC_ERR_CONFIGURATION, "no energy for this potential");
    }
    const int threads = 64 * std::min(ET / 64, (n + 63) / 64);   // a row of few units needs no more wavefronts
    switch (A.pot) {
    case ECMC_POT_INVERSE_POWER: launch_rows<ECMC_POT_INVERSE_POWER>(A, backward, threads, st); break;
    case ECMC_POT_INVERSE_POWER_TRUNC: launch_rows<ECMC_POT_INVERSE_POWER_TRUNC>(A, backward, threads, st); break;
    case ECMC_POT_LENNARD_JONES: launch_rows<ECMC_POT_LENNARD_JONES>(A, backward, threads, st); break;
    case ECMC_POT_DISPLACED_EVEN_POWER: launch_rows<ECMC_POT_DISPLACED_EVEN_POWER>(A, backward, threads, st); break;
    default: launch_rows<ECMC_POT_MERGED_IMAGE_COULOMB>(A, backward, threads, st); break;
    }
    hipLaunchKernelGGL(energy_finish, dim3(1), dim3(ET), 0, st, (const double *)A.rows, n, backward ? 1 : 0, d_energy,
                       d_grad_par);
    if (hipGetLastError() != hipSuccess) return ecmc_fail(ECMC_ERR_HIP, "energy kernel launch failed");
    return ECMC_OK;
}

extern "C" int ecmc_energy_forward(const ecmc_energy_term *term, int32_t n, const double *d_pos,
                                   const double *d_charge, const int32_t *d_molecule, double system_length,
                                   double *d_energy, void *d_work, void *stream) {
    if (!d_energy) return ecmc_fail(ECMC_ERR_ARGUMENT, "null energy output");
    return energy_launch(term, n, d_pos, d_charge, d_molecule, system_length, false, d_energy, nullptr, nullptr,
                         nullptr, d_work, stream);
}

extern "C" int ecmc_energy_backward(const ecmc_energy_term *term, int32_t n, const double *d_pos,
                                    const double *d_charge, const int32_t *d_molecule, double system_length,
                                    double *d_grad_pos, double *d_grad_par, double *d_grad_charge, void *d_work,
                                    void *stream) {
    return energy_launch(term, n, d_pos, d_charge, d_molecule, system_length, true, nullptr, d_grad_pos, d_grad_par,
                         d_grad_charge, d_work, stream);
}
