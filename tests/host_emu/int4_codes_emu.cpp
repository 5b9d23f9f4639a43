// The append's int4 codes (append_row.h int4_nibble, by Newton steps) against the division that
// defines them (int4_code): for every fp16 scale that the codec can give, values around each
// half-integer multiple, where rounding decides, and extremes.  Exits 0 when all agree.
#include <stdint.h>
#include <stdio.h>

#include <random>

#include "append_row.h"

using namespace vkv;

static long bad = 0;
static void check(float x, float sc, float inv) {
    const uint32_t got = int4_nibble(x, sc, inv), want = (uint32_t)int4_code(x, sc) & 0xfu;
    if (got != want && bad++ < 10) fprintf(stderr, "x %a sc %a: %u, not %u\n", x, sc, got, want);
}

int main() {
    std::mt19937 rng(1);
    for (uint32_t bits = 0x0011; bits <= 0x7bff; ++bits) {
        const float sc = half_bits_to_float(bits), inv = 1.0f / sc;
        for (int k = -10; k <= 9; ++k) {
            float x = (float)(((double)k + 0.5) * sc);
            for (int u = 0; u < 6; ++u) x = nextafterf(x, -INFINITY);
            for (int u = 0; u < 12; ++u, x = nextafterf(x, INFINITY)) check(x, sc, inv);
        }
        for (int i = 0; i < 20; ++i) check(__builtin_bit_cast(float, (uint32_t)rng()), sc, inv);
        for (float x : {0.f, -0.f, INFINITY, -INFINITY, NAN, 3.4e38f, -3.4e38f, 1e-45f, -1e-40f, 1.2e-38f}) check(x, sc, inv);
    }
    // the largest two magnitudes, NaN ignored, and the sums of a group's codes
    for (int i = 0; i < 20000; ++i) {
        float x[32];
        std::normal_distribution<float> n;
        for (float& v : x) v = n(rng) * (rng() % 40 == 0 ? 1e5f : 1.f);
        if (i % 3 == 0) x[rng() % 32] = NAN;
        if (i % 5 == 0) x[rng() % 32] = -INFINITY;
        const Int4Group q = int4_encode_group(x);
        float a1 = 0.f, a2 = 0.f;
        for (float v : x) {
            const float a = fabsf(v);
            if (a > a1) { a2 = a1; a1 = a; } else if (a > a2) a2 = a;
        }
        int s1 = 0, s2 = 0, sm = 0, c1, c2, cm;
        bool ok = q.s16 == int4_scale_bits(a2);
        for (int e = 0; e < 32; ++e) {
            const int code = int4_code(x[e], q.sc);
            ok = ok && ((q.w[e / 8] >> (4 * (e % 8))) & 0xfu) == ((uint32_t)code & 0xfu);
            s1 += code; s2 += code * code;
            sm = sm > (code < 0 ? -code : code) ? sm : (code < 0 ? -code : code);
        }
        int4_code_sums(q, c1, c2, cm);
        if (!(ok && c1 == s1 && c2 == s2 && cm == sm) && bad++ < 10) fprintf(stderr, "group %d: %d %d %d, not %d %d %d\n", i, c1, c2, cm, s1, s2, sm);
    }
    return bad ? 1 : 0;
}
