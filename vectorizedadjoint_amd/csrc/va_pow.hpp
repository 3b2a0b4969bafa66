// va_pow.hpp -- pow(x, y) with the rounding of the host C library's pow, for the
// step controller.  Compiles as HIP device code and as plain host C++.
//
// Boost.odeint's default_step_adjuster (called by the reference's controlled
// loop, lib/include/detail/runge_kutta.hpp:104-107) scales the step by
// std::pow(err, -1/q).  On Linux that is glibc's pow (2.28 and later), whose
// result is not always the correctly rounded power: on the controller's
// arguments about 8 in 10^4 calls differ from it by one ulp.  One ulp in a step
// size changes the rest of an instance's accept/reject history, so a device
// pow that rounded differently would change the reference's step sequence on
// several percent of the instances.  This file restates the published
// algorithm that glibc's pow uses (Szabolcs Nagy's log/exp pair, also in ARM's
// optimized-routines) in the operation order of its x86-64 FMA build, where
// the compiler contracts every a*b+c into one fused multiply-add:
//
//   log:  x = 2^k z with z in [0x1.69555p-1, 0x1.69555p0);
//         log x = k ln2 + log c + log1p(r),  r = z (1/c) - 1  (exact: 1/c has
//         few bits), c from a 128-entry table indexed by z's leading mantissa
//         bits; log1p(r) - r + r^2/2 by a polynomial in r; the sum carried as a
//         head hi and a tail lo.
//   mul:  y log x as ehi + elo, elo holding the rounding error of y*hi.
//   exp:  exp(ehi + elo) = 2^(j/128) exp(r'), j = round(128 ehi / ln2),
//         r' the reduced argument; 2^(j/128) = H (1 + T) from a 128-entry
//         table; exp(r') - 1 by a degree-5 polynomial; result scale + scale*tmp.
//
// Tables: va_pow_tables.hpp (generated from their definitions by
// gen_va_pow_tables.py).  The polynomial coefficients and ln2 splits are the
// published ones.  tests/test_pow_controller.py checks this code, built on
// the host, against the host's libm pow bit for bit.
//
// Domain: x > 0 normal or +inf (pow(+inf, y < 0) = +0), y negative with
// |y log x| < 512 -- the controller's error ratios in [5^-8, 1e300] and
// exponents -1/q.  The C library's special-case paths (zero, subnormal,
// negative or NaN x, huge or tiny exponents) are not restated.
#pragma once

#include <math.h>
#include <stdint.h>

#include "va_pow_tables.hpp"

#if defined(__HIPCC__)
#define VA_POW_HD __host__ __device__ __forceinline__
#else
#define VA_POW_HD inline
#endif

namespace va {
namespace powref {

VA_POW_HD double as_double(uint64_t u) { return __builtin_bit_cast(double, u); }
VA_POW_HD uint64_t as_bits(double d) { return __builtin_bit_cast(uint64_t, d); }

// a double from its halves (two moves on the device, no 64-bit arithmetic)
struct Halves {
    uint32_t lo, hi;
};
VA_POW_HD double from_halves(uint32_t hi, uint32_t lo)
{
    return __builtin_bit_cast(double, Halves{lo, hi});
}

// The algorithm's constants, as literals: each use forms the 64-bit value in a
// scalar register pair.  A caller may pass an object with the same members
// instead (PowRegs in va_device.hpp keeps them in vector registers).
struct PowLiterals {
    // log1p polynomial, scaled by the evaluation (p0 = -1/2)
    static constexpr double P0 = -0x1p-1;
    static constexpr double P1 = 0x1.555555555556p-2 * -2;
    static constexpr double P2 = -0x1.0000000000006p-2 * -2;
    static constexpr double P3 = 0x1.999999959554ep-3 * 4;
    static constexpr double P4 = -0x1.555555529a47ap-3 * 4;
    static constexpr double P5 = 0x1.2495b9b4845e9p-3 * -8;
    static constexpr double P6 = -0x1.0002b8b263fc3p-3 * -8;
    static constexpr double LN2_HI = 0x1.62e42fefa3800p-1;
    static constexpr double LN2_LO = 0x1.ef35793c76730p-45;
    // exp: 128/ln2, -ln2/128 split, rounding shift, polynomial
    static constexpr double INV_LN2_128 = 0x1.71547652b82fep0 * 128;
    static constexpr double NEG_LN2_HI_128 = -0x1.62e42fefa0000p-8;
    static constexpr double NEG_LN2_LO_128 = -0x1.cf79abc9e3b3ap-47;
    static constexpr double SHIFT = 0x1.8p52;
    static constexpr double E2 = 0x1.ffffffffffdbdp-2;
    static constexpr double E3 = 0x1.555555555543cp-3;
    static constexpr double E4 = 0x1.55555cf172b91p-5;
    static constexpr double E5 = 0x1.1111167a4d017p-7;
};
// bits of 0x1.69555p-1, below which the scaled argument z does not lie; their low
// half is zero, so the argument reduction works on the high 32 bits
constexpr uint32_t OFF_HI = 0x3fe69555u;

// Table access.  GlobalTables reads the constant tables; a caller may supply
// another accessor with the same two functions (the kernels read LDS copies).
struct GlobalTables {
    VA_POW_HD static void log_entry(int i, double &invc, double &logc, double &logctail)
    {
        invc = powtab::LOG[i][0];
        logc = powtab::LOG[i][1];
        logctail = powtab::LOG[i][2];
    }
    VA_POW_HD static void exp_entry(int i, uint64_t &tail_bits, uint64_t &scale_bits)
    {
        tail_bits = powtab::EXP[2 * i];
        scale_bits = powtab::EXP[2 * i + 1];
    }
};

// log(x) as hi + *lo for x > 0 normal (x given by its bits)
template <class T = GlobalTables, class C = PowLiterals>
VA_POW_HD double log_hilo(uint64_t ix, double *lo, const C &c = C())
{
    const uint32_t hx = (uint32_t)(ix >> 32), tmp = hx - OFF_HI;
    const int i = (int)((tmp >> 13) & 127);
    const int k = (int)tmp >> 20;
    const double z = from_halves(hx - (tmp & 0xfff00000u), (uint32_t)ix);
    const double kd = (double)k;
    double invc, logc, logctail;
    T::log_entry(i, invc, logc, logctail);
    const double r = fma(z, invc, -1.0);
    const double t1 = fma(kd, c.LN2_HI, logc);
    const double t2 = t1 + r;
    const double lo1 = fma(kd, c.LN2_LO, logctail);
    const double lo2 = t1 - t2 + r;
    const double ar = c.P0 * r;
    const double ar2 = r * ar;
    const double ar3 = r * ar2;
    const double hi = t2 + ar2;
    const double lo3 = fma(ar, r, -ar2);
    const double lo4 = t2 - hi + ar2;
    const double q =
        fma(ar2, fma(ar2, fma(r, c.P6, c.P5), fma(r, c.P4, c.P3)), fma(r, c.P2, c.P1));
    const double l = fma(ar3, q, lo1 + lo2 + lo3 + lo4);
    const double y = hi + l;
    *lo = hi - y + l;
    return y;
}

// exp(x + xtail) for |x| in [2^-54, 512)
template <class T = GlobalTables, class C = PowLiterals>
VA_POW_HD double exp_hilo(double x, double xtail, const C &c = C())
{
    double kd = fma(c.INV_LN2_128, x, c.SHIFT);
    const uint32_t ki = (uint32_t)as_bits(kd);
    kd = kd - c.SHIFT;
    double r = fma(kd, c.NEG_LN2_LO_128, fma(kd, c.NEG_LN2_HI_128, x));
    r = r + xtail;
    uint64_t tail_bits, scale_bits;
    T::exp_entry((int)(ki & 127), tail_bits, scale_bits);
    const double tail = as_double(tail_bits);
    // scale = 2^(ki / 128): the table's entry with ki / 128 added to its exponent
    // (ki << 45 in the 64-bit value: the high half alone)
    const double r2 = r * r;
    const double tmp = fma(r2 * r2, fma(r, c.E5, c.E4), fma(r2, fma(r, c.E3, c.E2), tail + r));
    const double scale =
        from_halves((uint32_t)(scale_bits >> 32) + (ki << 13), (uint32_t)scale_bits);
    return fma(scale, tmp, scale);
}

// pow(x, y) on the domain stated above, x finite
template <class T = GlobalTables, class C = PowLiterals>
VA_POW_HD double pow_finite(double x, double y, const C &c = C())
{
    double lo;
    const double hi = log_hilo<T>(as_bits(x), &lo, c);
    const double ehi = y * hi;
    const double elo = fma(y, lo, fma(y, hi, -ehi));
    return exp_hilo<T>(ehi, elo, c);
}

template <class T = GlobalTables>
VA_POW_HD double pow_ctrl(double x, double y)
{
    if (x == __builtin_huge_val()) return 0.0;
    return pow_finite<T>(x, y);
}

}  // namespace powref
}  // namespace va
