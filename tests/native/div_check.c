/* div_check COUNT: fvc_div_near against the division on COUNT random
 * dividends for each of a set of divisors and on dividends next to multiples
 * of the divisor; prints the number compared and the number that differ. */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "fvc_div.h"

static uint64_t s = 88172645463325252ull;
static uint64_t rnd(void) {
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    return s;
}
static double unit(void) { return (double)(rnd() >> 11) * 0x1p-53; }

int main(int argc, char **argv) {
    const long count = argc > 1 ? atol(argv[1]) : 100000;
    /* grid spacings, frame lengths, the RK4 divisor, all-ones and one-bit mantissas, the ends of the range */
    double b[96];
    int nb = 0;
    const double fixed[] = {6.0,  0.02, 0.5,    0.01,     0.1,           2.0 / 255, 1.0 / 127, 2.5 / 79, 1.0 / 3,
                            1e-3, 3.0,  1e-99, 9.9e99, 0x1.fffffffffffffp0, 0x1.0000000000001p0, 0x1.fffffffffffffp-7};
    for (unsigned i = 0; i < sizeof fixed / sizeof *fixed; i++) b[nb++] = fixed[i];
    while (nb < 96) b[nb++] = ldexp(1.0 + unit(), (int)(rnd() % 60) - 40) * ((nb & 1) ? -1.0 : 1.0);
    long n = 0, bad = 0;
    for (int k = 0; k < nb; k++) {
        const double d = b[k], y = fvc_near_inverse(d);
        if (y == 0.0) return 2;
        for (long i = 0; i < count; i++) {
            double a;
            switch (i & 3) {
            case 0: a = d * (double)(rnd() % 4096) * (1.0 + ((int)(rnd() % 5) - 2) * 0x1p-52); break;
            case 1: a = ldexp(unit() - 0.5, (int)(rnd() % 200) - 100); break;
            case 2: { /* close to a tie between two quotients */
                const double q = (1.0 + unit()) * (double)(1 + rnd() % 64);
                a = q * d + 0.5 * (nextafter(q, 1e9) - q) * d;
                break;
            }
            default: a = (unit() - 0.25) * 4096.0 * d;
            }
            const double want = a / d, got = fvc_div_near(a, d, y);
            n++;
            if (memcmp(&want, &got, 8) && !(want == 0.0 && got == 0.0)) {
                if (bad++ < 10) printf("%a / %a = %a, not %a\n", a, d, want, got);
            }
        }
    }
    const int ranged = fvc_near_inverse(0.0) == 0.0 && fvc_near_inverse(1e-320) == 0.0 && fvc_near_inverse(1e200) == 0.0 &&
                       fvc_near_inverse(-1e200) == 0.0 && fvc_near_inverse(INFINITY) == 0.0 &&
                       fvc_near_inverse(NAN) == 0.0;
    printf("%ld %ld %d\n", n, bad, ranged);
    return 0;
}
