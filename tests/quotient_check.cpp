// quotient(a, r, 1 / r) of md_common.h against a / r on the host: argv[1] rounds
// of random operands, of significands next to 1 and 2 and to each other, of
// quotients next to midpoints, and of exponents up to the ends of the stated range.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "md_common.h"

static uint64_t g_state = 88172645463325252ull;
static uint64_t rnd() {
    g_state ^= g_state << 13;
    g_state ^= g_state >> 7;
    g_state ^= g_state << 17;
    return g_state;
}
static double number(uint64_t frac, int e) {
    const uint64_t u = ((uint64_t)(e + 1023) << 52) | (frac & ((1ull << 52) - 1));
    double d;
    memcpy(&d, &u, sizeof d);
    return d;
}
static uint64_t frac() {  // any, or within a few units of 1 or 2
    const uint64_t x = rnd();
    switch (x >> 62) {
        case 0: return x & 15u;
        case 1: return ~(x & 15u);
        default: return x;
    }
}

static long g_bad = 0, g_n = 0;
static void check(double a, double r) {
    const double want = a / r, got = md::quotient(a, r, 1.0 / r);
    if (!(fabs(want) >= 0x1p-1022 && fabs(want) < 0x1p1023)) return;
    ++g_n;
    if (memcmp(&want, &got, sizeof got) != 0 && g_bad++ < 5) printf("%a / %a: %a, not %a\n", a, r, got, want);
}

int main(int argc, char** argv) {
    const long rounds = argc > 1 ? atol(argv[1]) : 1000000;
    for (long k = 0; k < rounds; ++k) {
        const double s = rnd() & 1 ? -1.0 : 1.0;
        // ordinary separations
        check(s * number(frac(), (int)(rnd() % 40) - 30), number(frac(), (int)(rnd() % 8) - 5));
        // the whole range
        check(s * number(frac(), (int)(rnd() % 1980) - 960), number(frac(), (int)(rnd() % 2000) - 1000));
        // a next to (q + half a unit) r, both ways
        const double r = number(frac(), (int)(rnd() % 8) - 5), q = number(frac(), (int)(rnd() % 20) - 10);
        const double h = ldexp(1.0, ilogb(q) - 53), a = fma(q, r, h * r);
        check(s * a, r);
        check(s * nextafter(a, 0.0), r);
        check(s * nextafter(a, INFINITY), r);
        // equal and neighbouring significands
        const uint64_t f = frac();
        check(number(f, (int)(rnd() % 5)), number(f + (rnd() % 5) - 2, (int)(rnd() % 5)));
    }
    const double zero = md::quotient(0.0, 0.7, 1.0 / 0.7), minus = md::quotient(-0.0, 0.7, 1.0 / 0.7);
    if (zero != 0.0 || signbit(zero) || minus != 0.0 || signbit(minus)) ++g_bad;
    printf("%ld quotients, %ld differ\n", g_n, g_bad);
    return g_bad ? 1 : 0;
}
