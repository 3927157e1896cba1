"""quotient() of csrc/attention.h against the IEEE quotient, on every pair that could be rounded the other way.

With y = 1 / b rounded, q = a y rounded lies within 1.5 units in the last place (ulp) of a / b: y is off by half a ulp of its
own, which is at most one of the product, and the product's rounding adds half a one.  The residual a - q b is a multiple of
ulp(q) ulp(b) below 1.5 x 2^24 of them, so its rounding moves it by at most one.  What the last operation rounds is therefore
a / b + E with |E| <= (1.5 + 1.5) 2^-24 ulp: the half ulp of y on the correction, and that one multiple.  With the significands
A and B as integers in [2^23, 2^24), a / b lies |j| / (2 B) ulp from the next rounding boundary, where
2^24 A (A >= B) or 2^25 A (A < B) = j modulo B.  Only pairs with |j| <= 6 come close enough.  The program solves that
congruence for every B and |j| <= 8 and compares all of them; powers of two in a and b change nothing while the residual
stays above 2^-126 (e >= 2^-60 and sum < 1024: above 2^-118)."""
import subprocess

SOURCE = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static float quotient(float e, float sum, float inv) {
    const float q = e * inv;
    return fmaf(fmaf(-q, sum, e), inv, q);
}

int main(int argc, char** argv) {
    const int plain = argc > 1;                  /* without the correction: the search has to find what that gets wrong */
    uint64_t pairs = 0, wrong = 0;
#pragma omp parallel for reduction(+ : pairs, wrong) schedule(dynamic, 4096)
    for (uint32_t B = 1u << 23; B < 1u << 24; ++B) {
        const int twos = __builtin_ctz(B);
        const float b = ldexpf((float)B, -23 + (int)(B % 10)), inv = 1.0f / b;
        for (int k = 24; k <= 25; ++k) {
            const int t = twos < k ? twos : k;
            const uint64_t n = B >> t;           /* 2^(k - t) A = j / 2^t modulo n, n odd */
            uint64_t x = 1;                      /* the inverse of 2^(k - t) */
            for (int i = 0; i < k - t; ++i) x = x & 1 ? (x + n) / 2 : x / 2;
            for (int j = -8; j <= 8; ++j) {
                if (j % (1 << t) != 0) continue;
                const int64_t m = j / (1 << t), r = ((m % (int64_t)n) + (int64_t)n) % (int64_t)n;
                uint64_t A = (x % n) * (uint64_t)r % n;
                const uint64_t lo = k == 24 ? B : 1u << 23, hi = k == 24 ? 1u << 24 : B;
                if (A < lo) A += (lo - A + n - 1) / n * n;
                for (; A < hi; A += n) {
                    const float a = ldexpf((float)A, -24);
                    const float got = plain ? a * inv : quotient(a, b, inv), want = a / b;
                    ++pairs;
                    wrong += memcmp(&got, &want, 4) != 0;
                }
            }
        }
    }
    printf("%llu %llu\n", (unsigned long long)pairs, (unsigned long long)wrong);
    return 0;
}
"""


def test_quotient_is_the_ieee_quotient(tmp_path):
    source, program = tmp_path / "quotient.c", tmp_path / "quotient"
    source.write_text(SOURCE)
    subprocess.run(["gcc", "-O2", "-march=native", "-ffp-contract=off", "-fopenmp", str(source), "-o", str(program), "-lm"], check=True)
    pairs, wrong = map(int, subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.split())
    assert pairs > 10 ** 8 and wrong == 0
    _, plain = map(int, subprocess.run([str(program), "plain"], check=True, capture_output=True, text=True).stdout.split())
    assert plain > 10 ** 7
