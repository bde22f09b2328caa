/* The pair pressure's two forms on the CPU: the reference's m (p_i + p_j) / (2 rho_j) and the tile passes' (m / 2)
 * quot(p_i + p_j, rho_j, 1 / rho_j), for pressures 0 or within [2^-40, 2^40] in magnitude, densities within [2^-40, 2^40]
 * and |m| = significand * 2^e, e uniform in [LO, HI].
 *
 *   half_mass N SEED LO HI      prints the number of pairs and of mismatches (the sign of a zero aside) */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static uint64_t state;
static uint64_t next(void) {
    uint64_t z = (state += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
/* significand in [1, 2) times 2^e, e in [lo, hi]; below 2^-126 rounded to a subnormal */
static float rnd(int lo, int hi) {
    const uint64_t r = next();
    const int e = lo + (int)(r % (uint64_t)(hi - lo + 1));
    return (float)ldexp(1.0 + (double)((uint32_t)(r >> 20) & 0x7fffffu) / 8388608.0, e) * (r >> 63 ? -1.0f : 1.0f);
}

int main(int argc, char** argv) {
    if (argc != 5) return 2;
    const long long n = atoll(argv[1]);
    state = strtoull(argv[2], 0, 0);
    const int lo = atoi(argv[3]), hi = atoi(argv[4]);
    long long bad = 0;
    for (long long i = 0; i < n; ++i) {
        const float m = rnd(lo, hi), rho = fabsf(rnd(-40, 40));
        const float a = (next() & 7) == 0 ? 0.0f : rnd(-40, 40), b = (next() & 7) == 0 ? 0.0f : rnd(-40, 40);
        const float sum = a + b, want_pressure = sum / (2.0f * rho);
        const float want = want_pressure > 0.0f ? m * want_pressure : 0.0f;
        const float y = 1.0f / rho, q0 = sum * y, twice = fmaf(fmaf(-rho, q0, sum), y, q0);
        const float got = twice > 0.0f ? (0.5f * m) * twice : 0.0f;
        bad += memcmp(&got, &want, 4) != 0 && !(got == 0.0f && want == 0.0f);
    }
    printf("%lld %lld\n", n, bad);
    return 0;
}
