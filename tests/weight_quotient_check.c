/* CPU check of the weight quantisers' quotient for qmax 7 (W4) and 127 (W8)
 * (csrc/q38m_layout.hip, quant_weights).  For a bf16 group maximum a with s =
 * RN(a/qmax) in [2^-120, FLT_MAX], r = RN(1/s), and a bf16 x with |x| <= a, the
 * device forms q0 = RN(x r), q = RN(q0 + RN(x - q0 s) r), clamps it to +-qmax and
 * rounds it by adding 1.5 * 2^23, whose low bits are then the integer.  Counts
 * the pairs where that integer differs from clamp(rint(RN(x/s))).
 *
 * Walked are all maxima of six binades, each with every such x: the one in
 * which s crosses 2^-120 (other scales divide) and the one above it, where
 * the residual x - q0 s comes nearest to the subnormals, three in the
 * middle, and the largest.  The binades between them are not walked: a and x
 * times a power of two give the same quotients as long as neither the
 * residual nor r leaves the normal range.
 *
 * Prints, per qmax, "binade <first a> qmax <q> checked <n> differ <m>" for each
 * and "pairs <n> mismatches <m>" for their sum.
 */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static float from_bits(uint32_t u) {
    float f;
    memcpy(&f, &u, sizeof f);
    return f;
}

static uint32_t to_bits(float f) {
    uint32_t u;
    memcpy(&u, &f, sizeof u);
    return u;
}

int main(void) {
    const int tops[2][6] = {{0x0480, 0x0500, 0x3780, 0x3f80, 0x7d00, 0x7f00},
                            {0x0680, 0x0700, 0x3780, 0x3f80, 0x7d00, 0x7f00}};
    const float qmaxes[2] = {7.0f, 127.0f};
    for (int k = 0; k < 2; ++k) {
        const float qmax = qmaxes[k];
        long long pairs = 0, mismatches = 0;
        for (int b = 0; b < 6; ++b) {
            long long checked = 0, differ = 0;
            for (int ah = tops[k][b]; ah < tops[k][b] + 128; ++ah) {
                const float a = from_bits((uint32_t)ah << 16);
                const float s = a / qmax;
                if (!(s >= 0x1p-120f && s <= 0x1.fffffep+127f)) continue;
                const float r = 1.0f / s;
                for (int xh = 0; xh <= ah; ++xh)
                    for (int sign = 0; sign < 2; ++sign) {
                        const float x = sign ? -from_bits((uint32_t)xh << 16) : from_bits((uint32_t)xh << 16);
                        const float want = fminf(fmaxf(rintf(x / s), -qmax), qmax);
                        const float q0 = x * r;
                        const float q = fmaf(fmaf(-q0, s, x), r, q0);
                        const uint32_t bits = to_bits(fminf(fmaxf(q, -qmax), qmax) + 12582912.0f);
                        ++checked;
                        if ((int8_t)(bits & 0xffu) != (int)want) ++differ;
                    }
            }
            printf("binade 0x%04x qmax %d checked %lld differ %lld\n", (unsigned)tops[k][b], (int)qmax,
                   checked, differ);
            pairs += checked;
            mismatches += differ;
        }
        printf("pairs %lld mismatches %lld\n", pairs, mismatches);
    }
    return 0;
}
