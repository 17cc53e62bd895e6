// The short FP64 division (div_mid) against the full one over the whole range
// that its comment states: random operands, and quotients next to a tie of
// the rounding (the midpoint of two doubles, subnormal ones among them).
#include "../../nyles_amd/csrc/nyl_internal.h"
#include "emu.h"
using namespace nyl;

int main() {
    std::mt19937_64 rng(1);
    std::uniform_real_distribution<double> u(1.0, 2.0);
    const double least = NYL_DIV_LEAST;
    const int le = std::ilogb(least);
    int bad = 0;
    auto one = [&](double a, double b) {
        if (std::fabs(a) < least) return;
        const double q = div_mid(a, b), w = a / b;
        if (memcmp(&q, &w, sizeof(q)) != 0 && bad++ < 5) printf("%a / %a = %a, want %a\n", a, b, q, w);
    };
    one(0.0, 3.0);
    for (int ea : {le, le + 1, le + 60, -700, -400, -149, -60, 0, 126, 200, 319})
        for (int eb : {-54, -53, 0, 1, 62, 120, 126, 184, 189})
            for (int k = 0; k < 20000; k++) {
                const double b = std::ldexp(u(rng), eb);
                one(std::ldexp(u(rng), ea) * (k & 1 ? -1 : 1), b);
                // a next to (q + half a unit) * b
                const double q = std::ldexp(u(rng), ea - eb);
                const double ulp = std::nextafter(q, 2 * q) - q;
                double a = std::fma(q, b, 0.5 * ulp * b);
                one(a, b);
                one(std::nextafter(a, 0.0), b);
                one(std::nextafter(a, 2 * a), b);
                // ... with few bits in the quotient
                const double m = (double)(2 * (rng() % 1000) + 1);
                a = std::ldexp(m * b, ea - eb - 10);
                one(a, b);
                one(std::nextafter(a, 0.0), b);
                one(std::nextafter(a, 2 * a), b);
            }
    // next to (m + half) of the least double, where the range has such quotients
    for (int eb : {-54, 0, 62, 126, 150, 184, 189})
        for (int em = 0; em < 52; em++)
            for (int k = 0; k < 2000; k++) {
                const double b = std::ldexp(u(rng), eb), m = std::floor(std::ldexp(u(rng), em));
                const double a = std::ldexp((2 * m + 1) * b, -1075);
                one(a, b);
                one(std::nextafter(a, 0.0), b);
                one(std::nextafter(a, 2 * a), b);
            }
    printf("division: %d mismatches\n", bad);
    printf(bad ? "FAIL\n" : "ALL OK\n");
    return bad != 0;
}
