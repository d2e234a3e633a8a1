// FP64 device math for the round-trip-matrix kernels (gfx950).
//
// log n!, modified Bessel functions of half-integer order and the Mie
// coefficients, evaluated per lane.  Each function follows the CaPS v0.5
// algorithm it cites, so that the GPU values agree with the reference to a
// few ulp of the log-domain results.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace capsd {

constexpr double LOG2 = 0.69314718055994530942;
constexpr double LOGPI = 1.14472988584940017414;
constexpr double HALF_LOG_2PI = 0.91893853320467274178;
constexpr int LFAC_TABLE = 1024;

// log n! : table of log Γ(n+1) below 1024 (filled by the host from lgamma),
// Stirling's series cut after 1/(12n) above.  Reference: src/logfac.c:66615-66628.
__device__ __forceinline__ double lfac(const double* __restrict__ tab, int n)
{
    if (n < LFAC_TABLE) return tab[n];
    const double dn = (double)n;
    return (dn + 0.5) * log(dn) - dn + HALF_LOG_2PI + (1. / 12) / dn;
}

// Debye polynomials u_k(p)/p^k in t = p², k = 1..5 (DLMF 10.41.10).
__device__ __forceinline__ void debye_u(double t, double& u1, double& u2, double& u3, double& u4, double& u5)
{
    u1 = (3 - 5 * t) / 24.;
    u2 = (81 + t * (-462 + 385 * t)) / 1152.;
    u3 = (30375 + t * (-369603 + t * (765765 - 425425 * t))) / 414720.;
    u4 = (4465125 + t * (-94121676 + t * (349922430 + t * (-446185740 + 185910725 * t)))) / 39813120.;
    u5 = (1519035525. + t * (-49286948607. + t * (284499769554. + t * (-614135872350.
          + t * (566098157625. - 188699385875. * t))))) / 6688604160.;
}

// log I_ν(x), log K_ν(x) by the uniform large-order expansion (DLMF 10.41.3-4).
// Reference: src/bessel.c:673-726.
__device__ inline double logInu_asymp(double nu, double x)
{
    const double z = x / nu, a = sqrt(1 + z * z), t = 1 / (1 + z * z);
    double u1, u2, u3, u4, u5;
    debye_u(t, u1, u2, u3, u4, u5);
    const double y = 1 / (nu * a);
    const double s = log1p(y * (u1 + y * (u2 + y * (u3 + y * (u4 + y * u5)))));
    return nu * (a + log(z / (1 + a))) - 0.5 * log(2 * M_PI * nu * a) + s;
}

__device__ inline double logKnu_asymp(double nu, double x)
{
    const double z = x / nu, a = sqrt(1 + z * z), t = 1 / (1 + z * z);
    double u1, u2, u3, u4, u5;
    debye_u(t, u1, u2, u3, u4, u5);
    const double y = -1 / (nu * a);
    const double s = log1p(y * (u1 + y * (u2 + y * (u3 + y * (u4 + y * u5)))));
    return -nu * (a + log(z / (1 + a))) - 0.5 * log(a) + 0.5 * log(0.5 * M_PI / nu) + s;
}

// I_ν(x)/I_{ν+1}(x) from the continued fraction DLMF 10.33.1 iterated to an
// exact fixed point.  Reference: src/bessel.c:635-660.  The iteration count
// is bounded (the reference's is not): NAN after 2^24 steps.
__device__ inline double ratioI(double nu, double x)
{
    const double invx2 = 2 / x;
    const double a1 = (nu + 1) * invx2, a2 = (nu + 2) * invx2;
    double num = a2 + 1 / a1, den = a2;
    double ratio = a1 * num / den, last = 0;
    for (int l = 3; l < (1 << 24); l++) {
        const double an = invx2 * (nu + l);
        num = an + 1 / num;
        den = an + 1 / den;
        ratio *= num / den;
        if (ratio == last) return ratio;
        last = ratio;
    }
    return NAN;
}

// log I_{n+1/2}(x), log K_{n+1/2}(x).  Reference: src/bessel.c:781-833.
__device__ inline void logInKn_half(int n, double x, double& logI, double& logK)
{
    const double logx = log(x), invx = 1 / x;
    double Kn = 1, Knp = 1 + invx;
    double pref = -x + 0.5 * (log(M_PI / 2) - logx);
    double lKn, lKnp;
    if (n == 0) {
        lKn = pref;
        lKnp = pref + log(Knp);
    } else if (n >= 100) {
        lKnp = logKnu_asymp(n + 1.5, x);
        lKn = logKnu_asymp(n + 0.5, x);
    } else {
        for (int l = 2; l <= n + 1; l++) {
            const double k = (2 * l - 1) * Knp * invx + Kn;
            Kn = Knp;
            Knp = k;
            if (Kn > 1e100) {
                Kn *= 1e-100;
                Knp *= 1e-100;
                pref += log(1e100);
            }
        }
        lKnp = pref + log(Knp);
        lKn = pref + log(Kn);
    }
    logK = lKn;
    if (n >= 100)
        logI = logInu_asymp(n + 0.5, x);
    else
        logI = -logx - lKnp - log1p(exp(lKn - lKnp - log(ratioI(n + 0.5, x))));
}

// Even and odd parts (in the order ν) of the uniform expansions U = Σ u_k/ν^k
// of I_ν, K_ν and V = Σ v_k/ν^k of their derivatives (DLMF 10.41.3-6, 10.41.10-11,
// five terms; remainder below 0.6/w^6), w = √(ν² + x²).
struct Uniform {
    double w, ue, uo, ve, vo;
};

__device__ inline Uniform uniform(double nu, double x)
{
    Uniform f;
    f.w = sqrt(nu * nu + x * x);
    const double y = 1 / f.w, q = nu * y, t = q * q;
    double u1, u2, u3, u4, u5;
    debye_u(t, u1, u2, u3, u4, u5);
    const double v1 = (-9 + 7 * t) / 24.;
    const double v2 = (-135 + t * (594 - 455 * t)) / 1152.;
    const double v3 = (-42525 + t * (451737 + t * (-883575 + 475475 * t))) / 414720.;
    const double v4 = (-5740875 + t * (111234708 + t * (-396578754 + t * (493152660 - 202076875 * t)))) / 39813120.;
    const double v5 = (-1856598975. + t * (56869556085. + t * (-317970330678. + t * (672625003050.
                     + t * (-611386010235. + 201713136625. * t))))) / 6688604160.;
    const double y2 = y * y;
    f.ue = 1 + y2 * (u2 + y2 * u4);
    f.uo = y * (u1 + y2 * (u3 + y2 * u5));
    f.ve = 1 + y2 * (v2 + y2 * v4);
    f.vo = y * (v1 + y2 * (v3 + y2 * v5));
    return f;
}

// I_{l-1/2}(x)/I_{l+1/2}(x) = I'/I + ν/x (ν = l + ½) from the uniform expansion
// where w >= 430 (remainder below 1e-16), else by the backward recurrence
// r_j = (2j+1)/x + 1/r_{j+1} from an l0 far enough for the expansion's error
// there (0.6/w^6, w >= 40) times the product of the r_j^-2, at least
// e^{-(l0² - l²)/x}, to be below 1e-16: at most 54 steps, where the continued
// fraction took up to √(40 x) steps of three divisions (x = nχ of a metal is some 10^4:
// 252 us for the coefficients of one ξ at R/L = 200; all of k_wave_start,
// whose runs of degrees go beside them, takes 14 us).
__device__ inline double ratio_half(int l, double x)
{
    int l0 = l;
    const double w2 = (double)l * l + x * x;
    if (w2 < 430. * 430.) {
        const double a = x < 40 ? 1600 - x * x : 0.0, c = w2 < 1e4 ? 15.0 : 9.0;
        l0 = (int)ceil(sqrt(fmax(a, (double)l * l) + c * x)) + 3;
    }
    const double nu = l0 + 0.5, ix = 1 / x;
    const Uniform f = uniform(nu, x);
    double r = (f.w * (f.ve + f.vo) / (f.ue + f.uo) + nu) * ix;
    for (int j = l0 - 1; j >= l; j--) {
        double q = __builtin_amdgcn_rcp(r);
        q = fma(fma(-r, q, 1.0), q, q);
        q = fma(fma(-r, q, 1.0), q, q);
        r = fma((double)(2 * j + 1), ix, q);
    }
    return r;
}

// K_{l-1/2}(x)/K_{l+1/2}(x) and log(I_{l+1/2}(x)/K_{l+1/2}(x)); r1 =
// I_{l+1/2}(x)/I_{l+3/2}(x).  l < 100: the upward recurrence of K and the
// Wronskian; above: the uniform expansions, the ratio of K taken eight orders
// lower (-K'/K - ν/x cancels for x < ν) and brought up by κ_{j+1} = 1/((2j+1)/x + κ_j).
__device__ inline void half_IK(int l, double x, double r1, double& kappa, double& lIK)
{
    const double ix = 1 / x;
    if (l < 100) {
        double Kn = 1, Knp = 1 + ix, pref = -x + 0.5 * (log(M_PI / 2) - log(x));
        double Km = 1;   // K_{l-1/2} in Kn's scale
        for (int j = 2; j <= l + 1; j++) {
            const double k = fma((2 * j - 1) * ix, Knp, Kn);
            Km = Kn;
            Kn = Knp;
            Knp = k;
            if (Knp > 1e100) {
                Km *= 1e-100;
                Kn *= 1e-100;
                Knp *= 1e-100;
                pref += 230.25850929940456840;
            }
        }
        kappa = Km / Kn;
        lIK = -log(x) - 2 * pref - log(Knp) - log(Kn) - log1p(Kn / Knp / r1);
        return;
    }
    const double nl = l - 7.5;
    Uniform f = uniform(nl, x);
    double k = (f.w * (f.ve - f.vo) / (f.ue - f.uo) - nl) * ix;
#pragma unroll
    for (int j = 0; j < 8; j++) k = 1 / fma((double)(2 * (l - 8 + j) + 1), ix, k);
    kappa = k;
    const double nu = l + 0.5;
    f = uniform(nu, x);
    lIK = 2 * (f.w + nu * log(x / (nu + f.w))) - LOGPI + log((f.ue + f.uo) / (f.ue - f.uo));
}

// log|a_l|, log|b_l| at χ = xi_/(1+L/R); epsm1 = ε(iξ)-1 of the sphere
// (+inf: perfect reflector).  Reference: src/libcaps.c:485-520, 557-602.
// With κ = K_{l-1/2}/K_{l+1/2}(χ), r = I_{l+1/2}/I_{l+3/2} at χ, q, q' the same and
// I_{l-1/2}/I_{l+1/2} at nχ, everything but I/K divided by I_{l+1/2}(nχ) and
// K_{l+1/2}(χ), and the 2l+1 of I_{l-1/2} = (2l+1)/x I_{l+1/2} + I_{l+3/2} taken out:
//   a: (ε-1)(l+1) + n²χ/r - nχ/q over (ε-1)(χκ + l) + χ(κ + n q'),
//   b: χ(n/q - 1/r) over χ(κ + n q').
__device__ inline void mie(double xi_, double LbyR, double epsm1, int l, double& lna, double& lnb)
{
    const double chi = xi_ / (1 + LbyR);
    const double r = ratio_half(l + 1, chi);
    double kappa, lIK;
    half_IK(l, chi, r, kappa, lIK);
    lIK += LOGPI - LOG2;
    if (isinf(epsm1)) {
        lnb = lIK;
        lna = lIK + log((l + 1 + chi / r) / (l + chi * kappa));
        return;
    }
    const double n = sqrt(1 + epsm1), q = ratio_half(l + 1, n * chi);
    const double q1 = (2 * l + 1) / (n * chi) + 1 / q;
    const double gd = chi * (kappa + n * q1);
    const double sc = 1 / fmax(1.0, epsm1), e = epsm1 * sc;   // (large ε: nothing overflows)
    lna = lIK + log(e * (l + 1) + (1 + epsm1) * sc * (chi / r) - n * sc * (chi / q))
        - log(e * (chi * kappa + l) + gd * sc);
    lnb = lIK + log(chi * (n / q - 1 / r)) - log(gd);
}

// Fresnel coefficients at k_ = xi_ sqrt(x²-1) (x = cosh of the integration
// variable).  Reference: src/libcaps.c:616-645.
__device__ __forceinline__ void fresnel(double epsm1, double xi_, double k_, double& rTE, double& rTM)
{
    if (isinf(epsm1)) {
        rTM = 1.0;
        rTE = -1.0;
        return;
    }
    const double x = xi_ * xi_ / (xi_ * xi_ + k_ * k_) * epsm1;
    const double bm1 = x / (sqrt(1 + x) + 1);
    rTE = -bm1 / (2 + bm1);
    rTM = (epsm1 - bm1) / (epsm1 + 2 + bm1);
}

}  // namespace capsd
