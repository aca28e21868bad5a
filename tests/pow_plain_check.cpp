// Compares the branch-free powers of a point between two GLL points
// (se_pow::pow_plain_at, compiled here as host code) with the C library's
// pow(x, k) bit for bit, over the range pow_plain admits.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "glibc_pow.h"

static uint64_t state = 0x9E3779B97F4A7C15ULL;
static uint64_t next() {  // SplitMix64
    uint64_t z = (state += 0x9E3779B97F4A7C15ULL);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

static long bad = 0, total = 0;
static void check(double x) {
    if (!se_pow::pow_plain(x)) return;
    double lo, hi = se_pow::log_hi_lo(se_pow::bits(x) & 0x7fffffffffffffffULL, &lo);
    for (int k = 0; k <= 11; k++) {
        const double a = pow(x, (double)k), b = se_pow::pow_plain_at(x, hi, lo, k);
        total++;
        if (std::memcmp(&a, &b, 8) != 0) {
            if (bad < 5) std::printf("x=%a k=%d libm=%a here=%a\n", x, k, a, b);
            bad++;
        }
    }
}

int main(int argc, char** argv) {
    const long n = argc > 1 ? std::atol(argv[1]) : 100000;
    for (long t = 0; t < n; t++) {
        double x = (double)(next() >> 11) * 0x1p-53 * 2.0 - 1.0;  // uniform [-1, 1)
        if (t % 4 == 1) x = std::ldexp(x, -(int)(next() % 61));
        check(x);
    }
    // the ends of the range and around powers of two
    for (int e = 0; e <= 61; e++)
        for (long j = -3; j <= 3; j++) {
            double c = std::ldexp(1.0, -e), x;
            uint64_t u;
            std::memcpy(&u, &c, 8);
            u += j;
            std::memcpy(&x, &u, 8);
            check(x), check(-x);
        }
    const double out[] = {0.0, -0.0, 0x1.fp-61, -0x1p-1074, 1.0000000000000002, -1.0000000000000002, INFINITY, NAN};
    for (double x : out)
        if (se_pow::pow_plain(x)) bad++;
    std::printf("mismatches %ld of %ld\n", bad, total);
    return bad != 0;
}
