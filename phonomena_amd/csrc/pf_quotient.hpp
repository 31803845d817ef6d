// Host check of the FP64 quotients from reciprocals (quotient(),
// pf_formulas.hpp).  Plain C++.
#pragma once
#include <cmath>
#include <cstdint>

namespace pf {

// Whether quotient()'s three operations, with the reciprocal y, give RN(a / b)
// for every dividend a, b an integer of 53 bits (as a double).  With A the
// dividend's 53 bits, a quotient near a rounding boundary M (an odd integer of
// 54 bits, half an ulp its unit) has A 2^w = B M + t, w = 53 or 54, with |t| /
// 2B its distance in ulp.  The operations' error before the last rounding is
// below 2^-51 ulp for y = RN(1 / b) (1.5 ulp of the first quotient times the
// relative errors of 1 / b and of the remainder), so only |t| <= 8 matters;
// the dividends of |t| <= 16 are found from M = -t / B mod 2^w and tried.
inline bool quotients_exact(double b, double y) {
    const uint64_t B = (uint64_t)b;
    const int z = __builtin_ctzll(B);
    if (z > 4) return true;  // then |t| is 0 or above 16
    uint64_t inv = B >> z;   // (B / 2^z)^-1 mod 2^64, by Newton's steps
    for (int k = 0; k < 6; k++) inv *= 2 - (B >> z) * inv;
    for (int w = 53; w <= 54; w++)
        for (int t = -16; t <= 16; t++) {
            if (t == 0 || t % (1 << z)) continue;
            const uint64_t mod = 1ull << (w - z), lo = 1ull << 53;
            uint64_t M = ((uint64_t)(int64_t)(-t / (1 << z)) * inv) & (mod - 1);
            if (M < lo) M += (lo - M + mod - 1) / mod * mod;
            for (; M < 2 * lo; M += mod) {
                const uint64_t A = (uint64_t)(((unsigned __int128)B * M + (__int128)t) >> w);
                if (A < lo / 2 || A >= lo) continue;
                const double a = (double)A, q = a * y;
                if (std::fma(std::fma(-b, q, a), y, q) != a / b) return false;
            }
        }
    return true;
}

// The same for a spacing h > 0: only its significand matters.
inline bool quotient_exact(double h) {
    int e = 0;
    const double b = std::ldexp(std::frexp(h, &e), 53);
    return quotients_exact(b, 1.0 / b);
}

}  // namespace pf
