// thomas.cpp -- host FP64 set-up of the LOD solver's Thomas tables.
//
// Follows the first-call block of diffusion_decay_solver__constant_coefficients_LOD_3D
// (BioFVM_parallel.cpp:714-918), whose FP64 denominator recursion both storage paths
// keep: its values must be exact for the FP64 path to match the reference bit for bit,
// and the FP32 path only rounds the finished tables.  Built with -ffp-contract=off; the
// one fused operation of the reference (axpy, BioFVM_vector.cpp:336-352, contracted by
// g++ -O3) is written as std::fma.
#include <cmath>
#include <cstdint>
#include <limits>

#include "bfvmb_internal.hpp"

namespace bfvmb {

namespace {

typedef unsigned __int128 u128;

// inverse of a modulo the odd m (extended Euclid)
uint64_t inverse_mod(uint64_t a, uint64_t m)
{
    __int128 t = 0, nt = 1, r = m, nr = a % m;
    while (nr != 0) {
        const __int128 q = r / nr;
        __int128 x = t - q * nt;
        t = nt;
        nt = x;
        x = r - q * nr;
        r = nr;
        nr = x;
    }
    return (uint64_t)(t < 0 ? t + m : t);
}

// whether fma(A, hi, A*lo) is A/d rounded for each of the numerators 2^52 <= A < 2^53 with
// A * 2^k = +-J mod D, J odd up to jmax, k = 53 and 54
bool pair_holds(double d, uint64_t D, const uint64_t inv[2], double hi, double lo, int jmax)
{
    for (int k = 0; k < 2; ++k)
        for (int J = 1; J <= jmax; J += 2)
            for (int sign = 0; sign < 2; ++sign) {
                uint64_t A0 = (uint64_t)((u128)inv[k] * (unsigned)J % D);
                if (sign)
                    A0 = D - A0;
                for (const uint64_t A : {A0, A0 + D})
                    if (A >= (1ull << 52) && A < (1ull << 53)) {
                        const double a = (double)A;
                        if (std::fma(a, hi, a * lo) != a / d)
                            return false;
                    }
            }
    return true;
}

}  // namespace

// Division by a divisor known in advance in one product and one fused multiply-add (Brisebarre,
// Muller, Raina, IEEE Trans. Computers 53, 2004): with hi = RN(1/d) and lo = RN(1/d - hi),
// RN(a*hi + RN(a*lo)) is RN(a/d) for every a unless a/d lies so close to the midpoint of two
// neighbouring numbers that the pair's error (below 2^-106 for 1/2 < a/d < 2, significands A and
// D as integers) reaches it.  With A/D - M = J/(D 2^k), M the midpoint, k = 54 below 1 and 53
// above, only odd |J| up to 1 can be that close, and each J names one A modulo D.  So the pair is
// checked against the true division on those few numerators; an even D has none.  Where it
// fails (1.3% of divisors) lo is moved by a few units in the last place and checked again (each
// unit widens the range of J by 2; the ranges below hold a margin).  hi is always RN(1/d).
// Returns false, with lo = NaN, where no pair holds (0.1%) or d is not of ordinary size: such
// divisors take the corrected product (div_corr, two corrections after a*hi).
bool reciprocal_pair(double d, double *hi, double *lo)
{
    *hi = 1.0 / d;
    *lo = std::numeric_limits<double>::quiet_NaN();
    if (!(d > 0x1p-40 && d < 0x1p40))
        return false;
    const double near = std::fma(-*hi, d, 1.0) / d;  // the residual 1 - hi d is exact
    int e;
    const uint64_t D = (uint64_t)std::ldexp(std::frexp(d, &e), 53);
    if (!(D & 1)) {
        *lo = near;
        return true;
    }
    const uint64_t inv[2] = {inverse_mod((uint64_t)(((u128)1 << 53) % D), D),
                             inverse_mod((uint64_t)(((u128)1 << 54) % D), D)};
    const double inf = std::numeric_limits<double>::infinity();
    for (int j = 0; j <= 4; ++j)
        for (int up = 0; up < (j ? 2 : 1); ++up) {
            double zl = near;
            for (int q = 0; q < j; ++q)
                zl = std::nextafter(zl, up ? inf : -inf);
            if (pair_holds(d, D, inv, *hi, zl, 2 * j + 5)) {
                *lo = zl;
                return true;
            }
        }
    return false;
}

// c1 = ((D*dt)/dx)/dx, c2 = (decay*dt)/3, c3 = ((1+c1)+c1)+c2, c3a = (1+c1)+c2
// (BioFVM_parallel.cpp:780-801).
void lod_constants(int nsub, const double *D, const double *decay, double dt, double dx,
                   double *c1, double *c2, double *c3, double *c3a)
{
    for (int d = 0; d < nsub; ++d) {
        double a = D[d] * dt;
        a = a / dx;
        a = a / dx;
        double b = decay[d] * dt;
        b = b / 3.0;
        c1[d] = a;
        c2[d] = b;
        c3[d] = ((1.0 + a) + a) + b;
        c3a[d] = (1.0 + a) + b;
    }
}

// One axis, tables [nsub][n] (BioFVM_parallel.cpp:882-896; x at world size 1 :810-851):
// c = -c1, den = c3 with c3a at both ends (1+c2 when n == 1); c[0] /= den[0];
// den[i] = fma(c1, c[i-1], den[i]); c[i] /= den[i].
void thomas_axis(int n, int nsub, const double *c1, const double *c2, const double *c3,
                 const double *c3a, double *den, double *cc)
{
    for (int d = 0; d < nsub; ++d) {
        double *dd = den + (size_t)d * n;
        double *c = cc + (size_t)d * n;
        for (int i = 0; i < n; ++i) {
            c[i] = c1[d] * -1.0;
            dd[i] = c3[d];
        }
        dd[0] = c3a[d];
        dd[n - 1] = c3a[d];
        if (n == 1)
            dd[0] = 1.0 + c2[d];
        c[0] = c[0] / dd[0];
        for (int i = 1; i < n; ++i) {
            dd[i] = std::fma(c1[d], c[i - 1], dd[i]);
            c[i] = c[i] / dd[i];
        }
    }
}

}  // namespace bfvmb
